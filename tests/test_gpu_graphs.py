"""Captured windows of the launches that are more than one kernel, or a
workgroup per node (blocked, fewer than 8 steps: those are captured, see
test_host_graphs.py): replayed several times, with launches of their own and
copies between the replays, they give the state of direct launches bit for
bit after each."""

import numpy as np
import pytest

from tvb_hpc import coupling as CF
from tvb_hpc import model as M
from tvb_hpc import scheme as SC
from tvb_hpc.hip import Simulation
from tvb_hpc.network import CSR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('kind,N,deg,P,L,noise', [
    ('mfma', 24, 9, 128, 4, False),
    ('sums', 40, 17, 70, 4, True),
    ('sums', 70, 66, 64, 6, False),
    ('split', 22, 9, 40, 4, True),
    ('split', 200, 199, 30, 5, False)])
def test_windows_equal_direct_launches(kind, N, deg, P, L, noise):
    print(kind, N, deg, P, L, noise, flush=True)
    rng = np.random.default_rng(N)
    csr = CSR(N, np.arange(N + 1) * deg,
              np.concatenate([np.sort(rng.choice(N, deg, replace=False))
                              for _ in range(N)]),
              rng.uniform(0.05, 0.5, N * deg),
              rng.integers(8, 30, size=(1, N * deg)))
    if kind == 'split':
        m = M.Kuramoto()
        c, kw = CF.Kuramoto(m), dict(waves=1, node_block=1)
    else:
        m = M.JansenRit()
        c = CF.Sigmoidal(m)
        kw = dict(waves=4, node_block=4, ring_dtype='bf16', ring_scale=200.0) \
            if kind == 'mfma' else dict(waves=1, node_block=1)
    x0 = m.initial_state(N, P, rng)
    sims = []
    for graph in (False, True):
        sim = Simulation(m, c, SC.EulerMaryuyamaStep(0.05, sigma=0.01)
                         if noise else SC.EulerStep(0.05), csr, P,
                         params={'c:a': np.linspace(0, 1, P).astype('f')},
                         kinds={'c:a': 'inst'}, steps_per_launch=L,
                         horizon=48, **kw)
        if kind == 'mfma':
            sim.set_coupling('mfma')
        sim.set_state(x0)
        sim.init_history('zeros')
        if noise:
            sim.set_noise(seed=5)
        sim.set_exec(graph=graph, window=4 * L)
        sims.append(sim)
    for steps in (4 * L, 8 * L, 4 * L + 3, 12 * L, 1, 4 * L):
        for sim in sims:
            sim.run(steps)
        a, b = (s.get_state() for s in sims)
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
        assert np.array_equal(*(s.get_ring() for s in sims))
