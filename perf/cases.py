"""
The work this package is used for, as cases with sizes, inputs, one pass
through the public entry points and, in 64 bits, what the pass returns.

Kinds of case (``case['kind']``):

* ``sweep``: P instances of one network integrated over a window of steps
  (``configs.SweepConfig.simulation`` / ``hip.Simulation``), with the monitor,
  BOLD and FC where the study wants them; the history in 32, 16 or 8 bits.
* ``subjects``: subjects with connectomes of different sizes in one launch
  (``hip.Batch``).
* ``gradient``: one evaluation of the FC-fit inversion, forward and backward
  (``autograd.integrate`` + ``autograd.fc_loss_device``).
* ``logp``: the Euler-Maruyama log-likelihood of a trajectory with its
  parameter gradients (``Simulation.logp``).
* ``fcfit``: the FC-fit loss of given samples, forward and backward.
* ``fc``: correlation matrices of given samples on the device.
* ``rmap``: surface vertices to regions and back (``hip.RegionMap``).

Connectomes follow the package's generator: symmetric Bernoulli pattern,
lognormal weights scaled to a maximum of 1, tract lengths uniform in 10 to
200 mm or distances in a ball.  Launch shapes are those that
``autotune.best_launch`` gives a configuration of these sizes.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), 'tvb-hpc_amd'))

# ---------------------------------------------------------------- the cases


def listed():
    return [
        # a whole small study on the smallest network: 64 couplings of a
        # 76-region Kuramoto model; latency of a step is all there is
        dict(name='kuramoto_n76_p64', kind='sweep', model='kuramoto',
             n_node=76, density=0.30, n_inst=64, n_speed=1, steps=200,
             ring='f32', tavg=0, bold=False, fc=False),
        # coupling x speed grid with BOLD and every instance's FC matrix
        dict(name='g2do_n84_p1024_bold_fc', kind='sweep', model='g2do',
             n_node=84, density=0.40, n_inst=1024, n_speed=16, steps=600,
             ring='f32', tavg=20, bold=True, fc=True),
        # 100 subjects on one sparsity pattern, own weights and delays
        dict(name='g2do_n84_100x64_pattern', kind='sweep', model='g2do_lin',
             n_node=84, density=0.15, n_inst=6400, n_speed=100, steps=500,
             ring='f32', tavg=0, bold=False, fc=False),
        # high resolution, exact delays, float32 history: the plain method
        dict(name='jansenrit_n998_p1024_f32', kind='sweep', model='jr',
             n_node=998, density=0.10, n_inst=1024, n_speed=1, steps=140,
             ring='f32', tavg=0, bold=False, fc=False),
        # the same network with 32 delay bins and a bfloat16 history: a
        # window of 50 monitor samples and its FC-SC error
        dict(name='jansenrit_n998_p1024_bf16_fc', kind='sweep', model='jr',
             n_node=998, density=0.10, n_inst=1024, n_speed=1, steps=1000,
             ring='bf16', tavg=20, bold=False, fc=True),
        # middle size, ragged in nodes and instances, 8-bit history
        dict(name='jansenrit_n379_p300_u8', kind='sweep', model='jr',
             n_node=379, density=0.15, n_inst=300, n_speed=1, steps=300,
             ring='u8', tavg=0, bold=False, fc=False),
        # 32 subjects of 68 to 400 regions, 64 instances each
        dict(name='rww_32_subjects', kind='subjects', n_subject=32,
             per_subject=64, density=0.30, steps=500),
        # one gradient of the FC-fit loss for 1024 instances
        dict(name='mpr_n84_p1024_gradient', kind='gradient', n_node=84,
             density=0.30, n_inst=1024, steps=1000, window=250, tavg=10),
        # log-likelihood of observed trajectories and its gradients
        dict(name='mpr_n84_p512_logp', kind='logp', n_node=84, density=0.30,
             n_inst=512, steps=300),
        # the loss alone, on samples that a program already holds
        dict(name='fcfit_m500_n84_p1024', kind='fcfit', n_sample=500,
             n_node=84, n_inst=1024),
        # FC of recorded samples, an odd atlas and an odd number of instances
        dict(name='fc_m200_n116_p700', kind='fc', n_sample=200, n_node=116,
             n_inst=700),
        # one cortical surface (two variables, one instance) and its regions
        dict(name='rmap_v20484_r148', kind='rmap', n_vertex=20484,
             n_region=148, n_var=2, n_inst=1),
    ]


def _log(rng, lo, hi):
    "an integer in [lo, hi], spread over its logarithm"
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return int(min(max(v, lo), hi))


def draw(rng):
    kind = rng.choice(['sweep', 'sweep', 'sweep', 'subjects', 'gradient',
                       'logp', 'fcfit', 'fc', 'rmap'])
    if kind == 'sweep':
        model = rng.choice(['kuramoto', 'g2do', 'g2do_lin', 'jr', 'jr'])
        n_node = _log(rng, 30, 998 if model == 'jr' else 400)
        density = rng.uniform(0.10, 0.30)
        n_speed, ring, tavg, bold, fc = 1, 'f32', 0, False, False
        if model.startswith('g2do'):
            n_speed = _log(rng, 1, 32)
        n_inst = 64 * n_speed if n_speed > 1 else _log(rng, 16, 1024)
        if model == 'jr':
            ring = rng.choice(['f32', 'bf16', 'f16', 'u8'])
        if model in ('g2do', 'jr') and rng.random() < 0.5:
            tavg, bold, fc = 20, model == 'g2do', True
        # about as many edge updates as the smallest and largest listed ones
        edges = density * n_node * n_node * n_inst
        steps = int(min(1000, max(40, rng.uniform(0.5, 2.0) * 4e9 / edges)))
        if tavg:
            steps = max(4, min(steps // tavg, 50)) * tavg
        return dict(kind=kind, model=model, n_node=n_node,
                    density=round(density, 3), n_inst=n_inst,
                    n_speed=n_speed, steps=steps, ring=ring, tavg=tavg,
                    bold=bold, fc=fc)
    if kind == 'subjects':
        return dict(kind=kind, n_subject=_log(rng, 2, 32),
                    per_subject=rng.choice([64, 64, 128, 37]),
                    density=round(rng.uniform(0.10, 0.30), 3),
                    steps=_log(rng, 40, 300))
    if kind == 'gradient':
        window = rng.choice([50, 100, 250])
        return dict(kind=kind, n_node=_log(rng, 30, 120),
                    density=round(rng.uniform(0.15, 0.35), 3),
                    n_inst=_log(rng, 32, 1024), tavg=10, window=window,
                    steps=window * rng.randint(2, 4))
    if kind == 'logp':
        return dict(kind=kind, n_node=_log(rng, 30, 120),
                    density=round(rng.uniform(0.15, 0.35), 3),
                    n_inst=_log(rng, 32, 1024), steps=_log(rng, 50, 400))
    if kind == 'fcfit':
        return dict(kind=kind, n_sample=_log(rng, 40, 1000),
                    n_node=_log(rng, 20, 120), n_inst=_log(rng, 1, 1024))
    if kind == 'fc':
        n_node = _log(rng, 20, 200)
        # the call's scratch holds the triangle and a copy of the samples
        n_sample = _log(rng, 20, 400)
        most = 100e6 / (4.0 * n_node * n_node + 4.0 * n_sample * n_node) - 64
        return dict(kind=kind, n_sample=n_sample, n_node=n_node,
                    n_inst=_log(rng, 1, max(1, min(1024, int(most)))))
    n_inst = _log(rng, 1, 64)
    n_var = rng.choice([1, 2, 6])
    return dict(kind=kind, n_vertex=_log(rng, 4000, 515056),
                n_region=_log(rng, 30, 400),
                n_var=2 if n_inst > 16 else n_var, n_inst=n_inst)


# ---------------------------------------------------------------- inputs

_PI2 = 2 * math.pi
# model: time step, conduction speed (m/s), noise, box of initial states
_MODELS = {
    'kuramoto': (0.1, 3.0, 0.01, [(0.0, _PI2)]),
    'g2do': (0.1, None, 0.005, [(-5, 5), (-5, 5)]),
    'g2do_lin': (0.1, 2.0, None, [(-5, 5), (-5, 5)]),
    'jr': (0.05, 5.0, None, [(-1, 1), (-500, 500), (-50, 50), (-6, 6),
                             (-20, 20), (-500, 500)]),
    # (the inversion starts from the resting branch, as after a burn-in)
    'mpr': (0.1, 3.0, 0.01, [(0.07, 0.09), (-2.2, -1.8)]),
}
_SIZES = (68, 84, 148, 246, 400)


def _pattern(rng, N, density, ball=False):
    "(rows, columns, weights, lengths) of a symmetric random connectome"
    iu = np.triu_indices(N, 1)
    mask = rng.random(iu[0].size) < density
    w = rng.lognormal(0.0, 1.0, iu[0].size)
    if ball:
        v = rng.normal(size=(N, 3))
        v /= np.linalg.norm(v, axis=1, keepdims=True)
        v *= 150.0 * rng.random(N)[:, None] ** (1.0 / 3.0)
        length = np.linalg.norm(v[iu[0]] - v[iu[1]], axis=1)
    else:
        length = rng.uniform(10.0, 200.0, iu[0].size)
    i, j, w, length = iu[0][mask], iu[1][mask], w[mask], length[mask]
    w = w / w.max() if w.size else w
    rows, cols = np.concatenate([i, j]), np.concatenate([j, i])
    order = np.lexsort((cols, rows))
    return (rows[order], cols[order], np.tile(w, 2)[order],
            np.tile(length, 2)[order])


def _delays(length, speed, dt):
    return np.maximum(1, np.rint(length / (speed * dt))).astype(np.int64)


def _bins(d, n):
    "delays at the centres of n equal bins"
    lo, hi = int(d.min()), int(d.max())
    if hi - lo + 1 <= n:
        return d
    edges = np.linspace(lo, hi + 1, n + 1)
    idx = np.clip(np.searchsorted(edges, d, side='right') - 1, 0, n - 1)
    mid = np.clip(np.rint((edges[:-1] + edges[1:] - 1) / 2), lo, hi)
    return mid[idx].astype(np.int64)


def _f32(a):
    return np.asarray(a, np.float64).astype(np.float32)


def _network(case, seed, model):
    "row index, column, weight (G or 1, nnz), delay (G, nnz) of a case"
    rng = np.random.default_rng([seed, 1])
    dt, speed = _MODELS[model][:2]
    N, G = case['n_node'], case.get('n_speed', 1)
    rows, cols, w, length = _pattern(rng, N, case['density'], model == 'jr')
    if model == 'g2do':
        d = np.stack([_delays(length, v, dt)
                      for v in np.linspace(2.0, 10.0, G)])
        w = w[None]
    elif model == 'g2do_lin':
        d = np.stack([_delays(length * rng.uniform(0.9, 1.1, length.size),
                              speed, dt) for _ in range(G)])
        w = w * rng.uniform(0.7, 1.3, (G, w.size))
    else:
        d, w = _delays(length, speed, dt)[None], w[None]
        if case.get('ring', 'f32') != 'f32' and d.size:
            d = _bins(d, 32)
            order = np.lexsort((cols, d[0], rows))
            rows, cols, w, d = rows[order], cols[order], w[:, order], d[:, order]
    return rows, cols, _f32(w), d


def _sweep_inputs(case, seed, model):
    "initial state and parameters"
    rng = np.random.default_rng([seed, 2])
    N, P, G = case['n_node'], case['n_inst'], case.get('n_speed', 1)
    x0 = np.stack([rng.uniform(lo, hi, (N, P))
                   for lo, hi in _MODELS[model][3]])
    top = {'kuramoto': 2.0, 'g2do': 1.0, 'g2do_lin': 0.5, 'jr': 1.0,
           'mpr': 1.0}[model]
    if G > 1:
        a = np.tile(np.linspace(0.0, top, P // G), G)
    else:
        a = np.sort(rng.uniform(0.0, top, P))
    par = {'c:a': _f32(a)}
    if model == 'kuramoto':
        par['m:omega'] = _f32(rng.normal(_PI2 * 10 / 1e3, 1e-3, N))
    if model == 'jr':
        par['m:mu'] = _f32(rng.uniform(0.1, 0.3, P))
    if model == 'mpr':
        par['m:eta'] = _f32(-5.0 + rng.uniform(-0.2, 0.2, (N, P)))
    return _f32(x0), par


def _subject_inputs(case, seed):
    "networks, initial states and per-instance parameters of the subjects"
    rng = np.random.default_rng([seed, 3])
    subs = []
    for k in range(case['n_subject']):
        N = _SIZES[k % len(_SIZES)]
        rows, cols, w, length = _pattern(rng, N, case['density'])
        d = _delays(length, float(rng.uniform(1.0, 10.0)), 0.1)
        x0 = _f32(rng.uniform(0.0, 1.0, (1, N, case['per_subject'])))
        subs.append((N, rows, cols, _f32(w)[None], d[None], x0))
    P = case['n_subject'] * case['per_subject']
    par = {'c:a': _f32(rng.uniform(0.0, 0.5, P)),
           'm:J': _f32(rng.uniform(0.1, 0.3, P)),
           'sigma': _f32(rng.uniform(1e-3, 1e-2, P))}
    return subs, par


def _signals(seed, n, N, P, device):
    "(n, N, P) correlated signals: 5 shared sources, mixed, plus noise"
    g = torch.Generator(device=device).manual_seed(1000003 + seed)
    src = torch.randn(n, 5, P, generator=g, device=device)
    mix = torch.randn(N, 5, generator=g, device=device)
    out = torch.randn(n, N, P, generator=g, device=device)
    return (out + 0.7 * torch.einsum('mkp,nk->mnp', src, mix)
            + 3.0).contiguous()


def _target_fc(seed, N):
    "a symmetric target matrix with unit diagonal"
    rng = np.random.default_rng([seed, 4])
    z = rng.normal(size=(3 * N, N)) + rng.normal(size=(3 * N, 1))
    return _f32(np.corrcoef(z.T)).reshape(N, N)


def _trajectory(case, seed, device):
    "(steps + 1, 2, N, P) frames near the model's resting branch"
    g = torch.Generator(device=device).manual_seed(2000003 + seed)
    n, N, P = case['steps'], case['n_node'], case['n_inst']
    box = torch.tensor(_MODELS['mpr'][3], device=device)
    x = torch.rand(1, 2, N, P, generator=g, device=device)
    x = box[:, 0, None, None] + x * (box[:, 1] - box[:, 0])[:, None, None]
    step = 0.004 * torch.randn(n, 2, N, P, generator=g, device=device)
    return torch.cat([x, x + step.cumsum(0)]).contiguous()


def _rmap(case, seed):
    rng = np.random.default_rng([seed, 5])
    # regions of uneven size, in patches as on a surface
    cut = np.sort(rng.choice(case['n_vertex'] - 1, case['n_region'] - 1,
                             replace=False)) + 1
    part = np.searchsorted(cut, np.arange(case['n_vertex']), side='right')
    return rng.permutation(case['n_region'])[part].astype(np.int32)


def _model_objects(model):
    from tvb_hpc import coupling as CF, model as M, scheme as SC
    dt, _, sigma = _MODELS[model][:3]
    osc = {'kuramoto': M.Kuramoto, 'g2do': M.Generic2dOscillator,
           'g2do_lin': M.Generic2dOscillator, 'jr': M.JansenRit,
           'mpr': M.MontbrioPazoRoxin}[model]()
    cf = {'kuramoto': CF.Kuramoto, 'g2do': CF.Sigmoidal,
          'g2do_lin': CF.Linear, 'jr': CF.Sigmoidal,
          'mpr': CF.Linear}[model](osc)
    if model == 'g2do':
        cf.param.update({'cmax': 1.0, 'midpoint': 0.0, 'r': 1.0})
    sc = SC.EulerStep(dt) if sigma is None else \
        SC.EulerMaryuyamaStep(dt, sigma=sigma)
    return osc, cf, sc


def _csr(N, rows, cols, w, d):
    from tvb_hpc.network import CSR
    row = np.searchsorted(rows, np.arange(N + 1))
    return CSR(N, row, cols, w if w.shape[0] > 1 else w[0], d)


def _config(case, seed, model):
    from tvb_hpc import configs
    osc, cf, sc = _model_objects(model)
    N, P, G = case['n_node'], case['n_inst'], case.get('n_speed', 1)
    ring = case.get('ring', 'f32')
    x0, par = _sweep_inputs(case, seed, model)
    kinds = {'c:a': 'inst', 'm:omega': 'node', 'm:mu': 'inst', 'm:eta': 'ni'}
    cfg = configs.SweepConfig(
        case.get('name') or case['kind'], osc, cf, sc,
        _csr(N, *_network(case, seed, model)), P, case['steps'], params=par,
        kinds={k: kinds[k] for k in par},
        group_size=P // G if G > 1 else None, tavg_period=case.get('tavg', 0),
        bold=case.get('bold', False), fc=case.get('fc', False),
        ring_dtype=ring,
        ring_scale=1.0 if ring == 'f32' else 1.0 / cf.param['cmax'])
    return cfg, x0, par


def prepare(case, seed):
    from tvb_hpc import autotune
    kind = case['kind']
    dev = torch.device('cuda')
    s = {'case': case, 'seed': seed}
    if kind == 'sweep':
        cfg, x0, _ = _config(case, seed, case['model'])
        sim = cfg.simulation(**autotune.best_launch(cfg))
        sim.set_state(x0)
        sim.init_history('zeros')
        if _MODELS[case['model']][2] is not None:
            sim.set_noise(seed=seed)
        s.update(sim=sim, x0=x0)
        if case['fc']:
            w = np.random.default_rng([seed, 6]).random((case['n_node'],) * 2)
            s['sc'] = _f32(np.triu(w, 1) + np.triu(w, 1).T)
    elif kind == 'subjects':
        from tvb_hpc import configs, coupling as CF, model as M, scheme as SC
        subs, par = _subject_inputs(case, seed)
        osc = M.ReducedWongWang()
        cfg = configs.BatchConfig(
            'subjects', osc, CF.Linear(osc), SC.EulerMaryuyamaStep(0.1),
            [(_csr(N, r, c, w, d), case['per_subject'])
             for N, r, c, w, d, _ in subs], case['steps'], params=par,
            kinds={k: 'inst' for k in par})
        b = cfg.batch(**autotune.best_batch_launch(cfg))
        for k, sub in enumerate(subs):
            b.set_state(k, sub[5])
        b.init_history('zeros')
        b.set_noise(seed=seed)
        b.set_exec(graph=True, window=100)
        s['batch'] = b
    elif kind in ('gradient', 'logp'):
        cfg, x0, par = _config(case, seed, 'mpr')
        launch = dict(autotune.best_launch(cfg))
        extra = dict(adjoint=True)
        if kind == 'gradient':
            extra['sample_slots'] = max(1, case['steps'] // case['tavg'])
        sim = cfg.simulation(**launch, **extra)
        s.update(sim=sim, x0=x0)
        if kind == 'gradient':
            s['a'] = torch.tensor(par['c:a'], device=dev, requires_grad=True)
            s['eta'] = torch.tensor(par['m:eta'], device=dev,
                                    requires_grad=True)
            s['target'] = torch.tensor(_target_fc(seed, case['n_node']),
                                       device=dev)
        else:
            s['traj'] = _trajectory(case, seed, dev)
            s['x0'] = s['traj'][0].cpu().numpy()
    elif kind == 'fcfit':
        s['x'] = _signals(seed, case['n_sample'], case['n_node'],
                          case['n_inst'], dev).requires_grad_()
        s['target'] = torch.tensor(_target_fc(seed, case['n_node']),
                                   device=dev)
    elif kind == 'fc':
        from tvb_hpc import hip
        s['x'] = _signals(seed, case['n_sample'], case['n_node'],
                          case['n_inst'], dev)
        s['out'] = torch.empty(case['n_inst'], case['n_node'],
                               case['n_node'], device=dev)
        s['ctx'] = hip.Context.default()
    else:
        from tvb_hpc import hip
        s['map'] = hip.RegionMap(_rmap(case, seed), case['n_region'])
        g = torch.Generator(device=dev).manual_seed(3000017 + seed)
        shape = (case['n_var'], case['n_inst'])
        s['node'] = torch.randn(case['n_vertex'], *shape, generator=g,
                                device=dev)
        s['roi'] = torch.randn(case['n_region'], *shape, generator=g,
                               device=dev)
    return s


def run(s):
    case, kind = s['case'], s['case']['kind']
    if kind == 'sweep':
        sim = s['sim']
        sim.run(case['steps'])
        x = torch.empty(s['x0'].shape, device='cuda')
        out = {'state': x}
        if case['tavg']:
            y = torch.empty(case['steps'] // case['tavg'], sim.N, sim.P,
                            device='cuda')
            sim.samples_into(y.data_ptr())
            out['samples'] = y
        if case['fc']:
            # every matrix of a small atlas; the window's FC-SC error of a
            # large one, whose matrices stay on the device
            if case['n_node'] <= 120:
                out['fc'] = sim.fc()
            else:
                out['error'] = sim.fc_sc_error(s['sc'])
            sim.fc_reset()
        sim.state_into(x.data_ptr())
        return out
    if kind == 'subjects':
        b = s['batch']
        b.run(case['steps'])
        b.sync()
        return [b.get_state(k) for k in range(len(b.subjects))]
    if kind == 'gradient':
        from tvb_hpc import autograd as AG
        s['a'].grad = s['eta'].grad = None
        y = AG.integrate(s['sim'], {'c:a': s['a'], 'm:eta': s['eta']},
                         s['x0'], case['steps'], case['window'],
                         seed=s['seed'])
        loss = AG.fc_loss_device(y, s['target'])
        loss.sum().backward()
        return {'loss': loss.detach(), 'a': s['a'].grad,
                'eta': s['eta'].grad}
    if kind == 'logp':
        sim = s['sim']
        sim.step = 0
        sim.set_state(s['x0'])
        sim.init_history('zeros')
        lp, g = sim.logp(s['traj'], grad=True)
        return {'logp': lp, 'a': g['c:a'], 'eta': g['m:eta']}
    if kind == 'fcfit':
        from tvb_hpc import autograd as AG
        s['x'].grad = None
        loss = AG.fc_loss_device(s['x'], s['target'])
        loss.sum().backward()
        return {'loss': loss.detach(), 'grad': s['x'].grad}
    if kind == 'fc':
        n, N, P = s['x'].shape
        s['ctx'].corr_noalloc(s['x'].data_ptr(), n, N, P,
                              s['out'].data_ptr())
        return s['out']
    return s['map'].to_avg(s['node']), s['map'].from_avg(s['roi'])


# ---------------------------------------------------------------- work

def _step_work(rows, cols, d, N, P, b, S, edge_flops, node_flops):
    """bytes and flops of a step: each history value that some node reads
    (distinct source and delay) and each new value once, the state in
    registers; the edges' and the nodes' arithmetic"""
    G = d.shape[0]
    distinct = sum(np.unique(cols * 65536 + d[g]).size for g in range(G)) / G
    return (b * (distinct + N) * P,
            (edge_flops * cols.size + node_flops * N) * P)


def work(case):
    kind = case['kind']
    if kind in ('sweep', 'gradient', 'logp'):
        model = case.get('model', 'mpr')
        rows, cols, w, d = _network(case, 0, model)
        N, P, n = case['n_node'], case['n_inst'], case['steps']
        b = {'f32': 4, 'bf16': 2, 'f16': 2, 'u8': 1}[case.get('ring', 'f32')]
        S = len(_MODELS[model][3])
        node = {'kuramoto': 20, 'g2do': 60, 'g2do_lin': 30, 'jr': 120,
                'mpr': 50}[model]
        by, fl = _step_work(rows, cols, d, N, P, b, S,
                            16 if model == 'kuramoto' else 2, node)
        if kind == 'sweep':
            m = n // case['tavg'] if case['tavg'] else 0
            fc = m * N * (N + 1) * P if case['fc'] else 0
            by_fc = 4 * N * N * P if case['fc'] and N <= 120 else 0
            return {'bytes': n * by + 4 * P * N * (2 * S + 2 * m) + by_fc,
                    'flops': n * fl + fc}
        if kind == 'logp':
            # frames, history values, and the sums' way back
            return {'bytes': n * (by + 4 * S * N * P) + 4 * N * P * 2,
                    'flops': n * 2 * fl}
        # forward, replay from checkpoints, reverse sweep; loss
        m = n // case['tavg']
        return {'bytes': n * (3 * by + 4 * (S + 1) * N * P * 2)
                + 4 * m * N * P * 4,
                'flops': n * 4 * fl + m * N * N * P * 3}
    if kind == 'subjects':
        subs, _ = _subject_inputs(case, 0)
        by = fl = 0
        for N, rows, cols, w, d, _ in subs:
            b1, f1 = _step_work(rows, cols, d, N, case['per_subject'], 4, 1,
                                2, 40)
            by, fl = by + b1, fl + f1
        return {'bytes': case['steps'] * by, 'flops': case['steps'] * fl}
    if kind in ('fcfit', 'fc'):
        n, N, P = case['n_sample'], case['n_node'], case['n_inst']
        x = 4 * n * N * P
        if kind == 'fc':
            return {'bytes': x + 4 * N * N * P, 'flops': n * N * (N + 1) * P}
        # samples read for the loss and for their gradient, gradient written
        return {'bytes': 3 * x, 'flops': n * N * (N + 1) * P
                + 2 * n * N * N * P}
    x = 4 * case['n_var'] * case['n_inst']
    return {'bytes': 2 * x * (case['n_vertex'] + case['n_region'])
            + 8 * case['n_vertex'],
            'flops': case['n_vertex'] * case['n_var'] * case['n_inst']}


# ---------------------------------------------------------------- in 64 bits

_M32 = 0xffffffff


def _mulhilo(a, b):
    "high and low words of a * b, a a 32-bit constant, b int64 words"
    lo = a * (b & 0xffff)
    hi = a * (b >> 16) + (lo >> 16)
    return hi >> 16, ((hi & 0xffff) << 16) | (lo & 0xffff)


def _normals(seed, n, N, p, S):
    """standard normals (S, N, P) of step n: Philox4x32-10 (Salmon et al.,
    2011) with counter (n, node, instance, 0) and the seed as key, then
    Box-Muller on 24-bit uniforms"""
    shape = (N, p.numel())
    i = torch.arange(N, device=p.device)[:, None].expand(shape)
    c = [torch.full(shape, n, dtype=torch.int64, device=p.device), i,
         p[None].expand(shape), torch.zeros(shape, dtype=torch.int64,
                                            device=p.device)]
    k0, k1 = seed & _M32, (seed >> 32) & _M32
    for _ in range(10):
        h0, l0 = _mulhilo(0xD2511F53, c[0])
        h1, l1 = _mulhilo(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & _M32, (k1 + 0xBB67AE85) & _M32
    u = ((c[0] >> 8) + 1).double() * 2.0 ** -24
    v = (c[1] >> 8).double() * 2.0 ** -24
    r = torch.sqrt(-2.0 * torch.log(u))
    z = [r * torch.cos(2 * math.pi * v), r * torch.sin(2 * math.pi * v)]
    return torch.stack(z[:S])


def _sigm(v, top, r, mid):
    return top / (1 + torch.exp(r * (mid - v)))


def _drift(model, x, c, par):
    if model == 'kuramoto':
        return torch.stack([par['m:omega'][:, None] + c])
    if model.startswith('g2do'):
        V, W = x
        return torch.stack([0.02 * (W - V ** 3 + 3.0 * V ** 2 + c),
                            0.02 * (-2.0 - 10.0 * V - W)])
    if model == 'mpr':
        r, V = x
        return torch.stack([1.0 / math.pi + 2 * r * V,
                            V ** 2 + par['m:eta'] + 15.0 * r + c
                            - (math.pi * r) ** 2])
    if model == 'rww':
        S = x[0]
        u = 0.270 * (0.6 * par['m:J'] * S + 0.33 + par['m:J'] * c) - 0.108
        z = u == 0
        h = u / (-torch.expm1(-154.0 * u) + z) + z / 154.0
        return torch.stack([-S / 100.0 + (1 - S) * h * 0.641])
    y0, y1, y2, y3, y4, y5 = x
    s = [_sigm(v, 0.005, 0.56, 5.52) for v in (y1 - y2, 135.0 * y0,
                                               33.75 * y0)]
    return torch.stack([
        y3, y4, y5, 0.325 * s[0] - 0.2 * y3 - 0.01 * y0,
        0.325 * (par['m:mu'] + 108.0 * s[1] + c) - 0.2 * y4 - 0.01 * y1,
        1.1 * (33.75 * s[2]) - 0.1 * y5 - 0.0025 * y2])


def _observed(model, x):
    return x[0] - x[1] if model == 'jr' else x[0]


class _Net:
    "delayed coupling sums of one network in 64 bits"

    def __init__(self, model, N, P, rows, cols, w, d, dev):
        self.model, self.N, self.P = model, N, P
        self.G = d.shape[0]
        self.H = int(d.max()) + 2 if d.size else 2
        t = lambda a: torch.as_tensor(a, device=dev)  # noqa: E731
        self.rows, self.cols = t(rows), t(cols)
        self.d = t(d).T.contiguous()                       # (nnz, G)
        self.w = t(w.astype(np.float64)).T[:, :, None]     # (nnz, G or 1, 1)
        self.g = torch.arange(self.G, device=dev)[None]
        self.ring = torch.zeros(self.H, N, self.G, P // self.G,
                                dtype=torch.float64, device=dev)

    def pre(self, y):
        if self.model == 'jr':
            return _sigm(y, 0.005, 1.0, 6.0)
        return _sigm(y, 1.0, 1.0, 0.0) if self.model == 'g2do' else y

    def write(self, n, y):
        self.ring[n % self.H] = y.reshape(self.N, self.G, -1)

    def sum(self, n):
        v = self.ring[(n - self.d) % self.H, self.cols[:, None], self.g]
        if self.model == 'kuramoto':
            v = torch.sin(v - self.ring[n % self.H][self.rows])
        else:
            v = self.pre(v)
        s = torch.zeros_like(self.ring[0])
        s.index_add_(0, self.rows, self.w * v)
        return s.reshape(self.N, self.P)


def _bold(state, x, dt):
    "one Euler step of Balloon-Windkessel on state [s, f, v, q]"
    s, f, v, q = state
    E0, V0, TE, nu, r0, eps, al = 0.4, 4.0, 0.04, 40.3, 25.0, 0.5, 0.32
    va = v ** (1 / al)
    ds = x - s / 0.65 - (f - 1) / 0.41
    dv = (f - va) / 0.98
    dq = (f * (1 - (1 - E0) ** (1 / f)) / E0 - va * (q / v)) / 0.98
    s, f, v, q = s + dt * ds, f + dt * s, v + dt * dv, q + dt * dq
    state[:] = [s, f, v, q]
    return V0 * (4.3 * nu * E0 * TE * (1 - q) + eps * r0 * E0 * TE
                 * (1 - q / v) + (1 - eps) * (1 - v))


def _corr(y):
    "(n, N, P) -> (P, N, N)"
    x = (y - y.mean(0)).permute(2, 1, 0).contiguous()
    c = torch.matmul(x, x.transpose(1, 2).contiguous())
    s = torch.sqrt(torch.diagonal(c, dim1=1, dim2=2))
    return c / (s[:, :, None] * s[:, None, :])


def _integrate(model, net, x, par, dt, steps, sigma, seed, p0=0, tavg=0,
               bold=False):
    "state after the steps and monitor samples, in 64 bits"
    p = torch.arange(p0, p0 + net.P, device=x.device)
    a = par['c:a']
    net.write(0, _observed(model, x))
    acc, samples = torch.zeros_like(x[0]), []
    hemo = [torch.zeros_like(x[0])] + [torch.ones_like(x[0])] * 3
    for n in range(steps):
        c = a * net.sum(n) / (net.N if model == 'kuramoto' else 1)
        if tavg:
            acc = acc + _observed(model, x)
        x = x + dt * _drift(model, x, c, par)
        if sigma is not None:
            x = x + math.sqrt(dt) * sigma * _normals(seed, n, net.N, p,
                                                     x.shape[0])
        if model == 'kuramoto':
            x = torch.where(x < 0, x + _PI2, torch.where(x > _PI2, x - _PI2,
                                                         x))
        net.write(n + 1, _observed(model, x))
        if tavg and (n + 1) % tavg == 0:
            out = acc / tavg
            samples.append(_bold(hemo, out, tavg * dt * 1e-3) if bold
                           else out)
            acc = torch.zeros_like(acc)
    return x, torch.stack(samples) if samples else None


def _loss(y, target):
    "1 - correlation of the upper triangles of FC(y) and of the target"
    iu = torch.triu_indices(y.shape[1], y.shape[1], 1, device=y.device)
    a = _corr(y)[:, iu[0], iu[1]]
    b = target[iu[0], iu[1]]
    a, b = a - a.mean(1, keepdim=True), b - b.mean()
    return 1 - (a * b).sum(1) / torch.sqrt((a * a).sum(1) * (b * b).sum())


def _blocks_loss(case, net, x, par, dt, sigma, seed, target):
    """the FC-fit loss, differentiable: steps in blocks of the smallest
    delay, whose coupling sums read earlier blocks only"""
    dev = x.device
    p = torch.arange(net.P, device=dev)
    B = int(net.d.min()) if net.d.numel() else case['steps']
    d, ys, acc, samples = net.d[:, 0], [x[0]], torch.zeros_like(x[0]), []
    past = torch.zeros(net.H, net.N, net.P, dtype=torch.float64, device=dev)
    for n0 in range(0, case['steps'], B):
        m = min(B, case['steps'] - n0)
        hist = torch.cat([past] + [torch.stack(ys)])  # steps -H .. n0
        k = net.H + n0 + torch.arange(m, device=dev)
        v = net.w[:, 0] * hist[k[:, None] - d, net.cols[None]]
        sums = torch.zeros(m, net.N, net.P, dtype=torch.float64, device=dev)
        sums = sums.index_add(1, net.rows, v)
        for j in range(m):
            acc = acc + x[0]
            x = x + dt * _drift('mpr', x, par['c:a'] * sums[j], par) + \
                math.sqrt(dt) * sigma * _normals(seed, n0 + j, net.N, p, 2)
            ys.append(x[0])
            if (n0 + j + 1) % case['tavg'] == 0:
                samples.append(acc / case['tavg'])
                acc = torch.zeros_like(acc)
    return _loss(torch.stack(samples), target)


def exact(case, seed):
    kind = case['kind']
    dev = torch.device('cuda' if torch.cuda.is_available() else 'cpu')
    up = lambda a: torch.as_tensor(a, device=dev).double()  # noqa: E731
    if kind == 'sweep':
        model = case['model']
        dt, _, sigma = _MODELS[model][:3]
        x0, par = _sweep_inputs(case, seed, model)
        net = _Net(model, case['n_node'], case['n_inst'],
                   *_network(case, seed, model), dev)
        x, y = _integrate(model, net, up(x0),
                          {k: up(v) for k, v in par.items()}, dt,
                          case['steps'], sigma, seed, tavg=case['tavg'],
                          bold=case['bold'])
        out = {'state': x}
        if case['tavg']:
            out['samples'] = y
        if case['fc'] and case['n_node'] <= 120:
            out['fc'] = _corr(y)
        elif case['fc']:
            N = case['n_node']
            w = np.random.default_rng([seed, 6]).random((N, N))
            sc = up(_f32(np.triu(w, 1)))
            iu = torch.triu_indices(N, N, 1, device=dev)
            out['error'] = torch.cat([
                ((_corr(y[:, :, k:k + 64])[:, iu[0], iu[1]]
                  - sc[iu[0], iu[1]]) ** 2).sum(1)
                for k in range(0, case['n_inst'], 64)])
        return out
    if kind == 'subjects':
        subs, par = _subject_inputs(case, seed)
        out, K = [], case['per_subject']
        for k, (N, rows, cols, w, d, x0) in enumerate(subs):
            q = {m: up(v[k * K:(k + 1) * K]) for m, v in par.items()}
            net = _Net('rww', N, K, rows, cols, w, d, dev)
            out.append(_integrate('rww', net, up(x0), q, 0.1, case['steps'],
                                  q['sigma'], seed, p0=k * K)[0])
        return out
    if kind in ('gradient', 'logp'):
        dt, _, sigma = _MODELS['mpr'][:3]
        x0, par = _sweep_inputs(case, seed, 'mpr')
        par = {k: up(v).requires_grad_() for k, v in par.items()}
        net = _Net('mpr', case['n_node'], case['n_inst'],
                   *_network(case, seed, 'mpr'), dev)
        if kind == 'gradient':
            loss = _blocks_loss(case, net, up(x0), par, dt, sigma, seed,
                                up(_target_fc(seed, case['n_node'])))
            out = {'loss': loss.detach()}
        else:
            tr = _trajectory(case, seed, dev).double()
            net.write(0, tr[0, 0])
            lp = torch.zeros(case['n_inst'], dtype=torch.float64, device=dev)
            for n in range(case['steps']):
                c = par['c:a'] * net.sum(n)
                r = tr[n + 1] - tr[n] - dt * _drift('mpr', tr[n], c, par)
                lp = lp - (r * r).sum((0, 1)) / (2 * dt * sigma ** 2)
                net.write(n + 1, tr[n + 1, 0])
            loss, out = lp, {'logp': lp.detach()}
        loss.sum().backward()
        return dict(out, a=par['c:a'].grad, eta=par['m:eta'].grad)
    if kind in ('fcfit', 'fc'):
        x = _signals(seed, case['n_sample'], case['n_node'], case['n_inst'],
                     dev).double()
        if kind == 'fc':
            return _corr(x)
        x.requires_grad_()
        loss = _loss(x, up(_target_fc(seed, case['n_node'])))
        loss.sum().backward()
        return {'loss': loss.detach(), 'grad': x.grad}
    rm = torch.as_tensor(_rmap(case, seed), device=dev).long()
    g = torch.Generator(device=dev).manual_seed(3000017 + seed)
    shape = (case['n_var'], case['n_inst'])
    node = torch.randn(case['n_vertex'], *shape, generator=g, device=dev)
    roi = torch.randn(case['n_region'], *shape, generator=g, device=dev)
    avg = torch.zeros(case['n_region'], *shape, dtype=torch.float64,
                      device=dev).index_add(0, rm, node.double())
    return avg, roi.double()[rm]
