"""Blocked launches with a workgroup per node and 16 instances (a pre() that
reads post_syn, few nodes and instances) against one step per launch, bit for
bit: rows of none, one, around 8 and 64, and past 128 edges, instance counts
around the 16 of a workgroup, delay groups, partial launches, the monitor,
noise, phases beyond the branch-free sine's range, two coupled observables,
and the transition log density.  Paced launches, which keep one wave per node
and 64 instances, must agree too."""

import numpy as np
import pytest

from tvb_hpc import coupling as CF
from tvb_hpc import model as M
from tvb_hpc import scheme as SC
from tvb_hpc.hip import Simulation
from tvb_hpc.network import CSR

pytestmark = pytest.mark.gpu


def _csr(N, deg, groups=1, dmin=6, seed=0):
    rng = np.random.default_rng(seed)
    rows = [np.sort(rng.choice(N, size=min(k, N), replace=False))
            for k in np.resize(deg, N)]
    row = np.concatenate([[0], np.cumsum([r.size for r in rows])])
    col = np.concatenate(rows)
    return CSR(N, row, col, rng.uniform(0.05, 0.5, col.size),
               rng.integers(dmin, dmin + 40, size=(groups, col.size)))


def _sim(model, cfun, csr, P, launch, scheme=None, **kw):
    m = getattr(M, model)()
    c = getattr(CF, cfun)(m)
    a = np.linspace(0.0, 1.0, P).astype(np.float32)
    gs = None if csr.n_group == 1 else -(-P // csr.n_group // 64) * 64
    return m, Simulation(m, c, scheme or SC.EulerStep(0.05), csr, P,
                         params={'c:a': a}, kinds={'c:a': 'inst'},
                         group_size=gs, horizon=60, **dict(launch, **kw))


SINGLE = dict(ipl=1, waves=2, node_block=2, steps_per_launch=1)


@pytest.mark.parametrize('model,cfun,N,deg,P,groups,L,noise,scale', [
    ('Kuramoto', 'Kuramoto', 5, (0, 1, 5), 1, 1, 7, False, 1.0),
    ('Kuramoto', 'Kuramoto', 11, (7, 8, 9), 15, 1, 2, True, 1.0),
    ('Kuramoto', 'Kuramoto', 70, (63, 64, 65), 17, 1, 5, False, 1.0),
    ('Kuramoto', 'Kuramoto', 140, (1, 139, 129, 0), 64, 1, 7, False, 1.0),
    ('Kuramoto', 'Kuramoto', 30, (12, ), 192, 3, 6, False, 1.0),
    ('Kuramoto', 'Kuramoto', 20, (9, ), 65, 1, 7, False, 1e6),
    ('Generic2dOscillator', 'Diff', 33, (16, 2), 33, 1, 4, False, 1.0),
    ('HMJE', 'Diff', 90, (8, 70), 18, 1, 5, False, 1.0),
    ('MontbrioPazoRoxin', 'Diff', 24, (20, 5), 80, 1, 7, True, 1.0)])
def test_split_launch_equals_single_steps(model, cfun, N, deg, P, groups, L,
                                          noise, scale):
    print('split', model, cfun, N, deg, P, groups, L, noise, flush=True)
    csr = _csr(N, deg, groups)
    steps = 3 * L + 1          # ends on a partial launch
    blocked = dict(ipl=1, waves=1, node_block=1, steps_per_launch=L)
    got = []
    for la in (SINGLE, blocked, dict(blocked, pace=1)):
        m, sim = _sim(model, cfun, csr, P, la, tavg_period=3, sample_slots=20,
                      scheme=SC.EulerMaryuyamaStep(0.05, sigma=0.02)
                      if noise else None)
        x0 = np.random.default_rng(5).uniform(0.1, 1.0,
                                              (sim.spec.S, N, P))
        sim.set_state((x0 * scale).astype(np.float32))
        sim.init_history('zeros')
        if noise:
            sim.set_noise(seed=3)
        sim.run(steps)
        got.append((sim.get_state(), sim.get_ring(), sim.samples()[0]))
    assert np.isfinite(got[0][0]).all()
    for other in got[1:]:
        for x, y in zip(got[0], other):
            assert np.array_equal(x, y)


def test_split_launch_log_density_equals_single_steps():
    csr = _csr(22, (9, 14, 0))
    P, T = 20, 30
    rng = np.random.default_rng(8)
    got = []
    for la in (SINGLE, dict(ipl=1, waves=1, node_block=1,
                            steps_per_launch=7)):
        m, sim = _sim('Kuramoto', 'Kuramoto', csr, P, la,
                      scheme=SC.EulerMaryuyamaStep(0.05, sigma=0.1))
        if not got:
            frames = rng.uniform(0, 6, (T + 1, sim.spec.S, 22, P)).astype('f')
        sim.set_state(frames[0])
        sim.init_history('zeros')
        got.append(np.asarray(sim.logp(frames)))
    assert np.array_equal(got[0], got[1])
