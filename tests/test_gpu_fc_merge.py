"""The FC merge (k_fc_prep, k_fc_update) against numpy's corrcoef in float64:
node counts around the 16-node tiles, instance counts around the lane blocks
(ragged rows are read in place), few and many samples, and both instance
blocks of the merge kernel; a simulation's merges one after another, the
first into uninitialised co-moments, across the end of the sample ring."""

import numpy as np
import pytest

from tvb_hpc import coupling as CF
from tvb_hpc import model as M
from tvb_hpc import scheme as SC
from tvb_hpc.hip import Simulation
from tvb_hpc.network import CSR

pytestmark = pytest.mark.gpu

# float32 results in [-1, 1] of float64 sums: half an ulp, 6e-8
TOL = 1e-7


@pytest.mark.parametrize('n,N,P', [
    (2, 2, 1), (3, 15, 63), (5, 16, 64), (66, 17, 65), (17, 33, 100),
    (100, 84, 7), (7, 130, 900)])
def test_corr_of_ragged_samples(ctx, n, N, P):
    import torch
    rng = np.random.default_rng(n + N + P)
    x = (rng.standard_normal((n, N, P)) + rng.standard_normal((n, 1, P))
         + 5.0).astype(np.float32)
    d = torch.from_numpy(x).cuda()
    out = torch.full((P, N, N), float('nan'), device='cuda')
    torch.cuda.synchronize()
    ctx.corr_noalloc(d.data_ptr(), n, N, P, out.data_ptr())
    ctx.sync()
    got = out.cpu().numpy()
    assert np.array_equal(got, ctx.corr(x))
    for p in {0, P // 2, P - 1}:
        want = np.corrcoef(x[:, :, p].astype(np.float64).T)
        assert np.abs(got[p] - want).max() <= TOL


@pytest.mark.parametrize('slots', [3, 5, 64])
def test_successive_merges_of_a_simulation(slots):
    N, P, T = 35, 70, 4
    rng = np.random.default_rng(1)
    row = np.arange(N + 1) * 3
    csr = CSR(N, row, np.concatenate([rng.choice(N, 3, replace=False)
                                      for _ in range(N)]),
              rng.uniform(0.1, 0.4, 3 * N), rng.integers(6, 20, 3 * N))
    m = M.Generic2dOscillator()
    sim = Simulation(m, CF.Linear(m), SC.EulerMaryuyamaStep(0.1, 0.05), csr,
                     P, params={'c:a': np.full(P, 0.1, np.float32)},
                     tavg_period=T, fc=True, sample_slots=slots, waves=1,
                     node_block=1, steps_per_launch=4)
    sim.set_state(m.initial_state(N, P, rng))
    sim.init_history('zeros')
    sim.set_noise(seed=3)
    for _ in range(2):             # the second round after a reset
        ys = []
        for _ in range(9):         # one sample at a time, merged as slots fill
            sim.run(T)
            ys.append(sim.samples()[0][-1])
        got = sim.fc()
        assert sim.n_fc_samples == 9
        y = np.stack(ys).astype(np.float64)
        for p in (0, 33, P - 1):
            want = np.corrcoef(y[:, :, p].T)
            assert np.abs(got[p] - want).max() <= TOL
        sim.fc_reset()
