"""Blocked launches as two kernels (every coupling sum of the launch, then
the updates from them) against one step per launch, bit for bit, and against
the CPU oracle: node counts around the workgroup's and the XCDs' shares, rows
past 64 and 128 edges, partial launches, delay groups, and rings in 32, 16
and 8 bits.  The one-kernel blocked launch (taken with pacing on) must agree
too."""

import numpy as np
import pytest

from harness import oracle_for, scaled_err
from tvb_hpc import coupling as CF
from tvb_hpc import model as M
from tvb_hpc import scheme as SC
from tvb_hpc.hip import Simulation
from tvb_hpc.network import CSR

pytestmark = pytest.mark.gpu


def _csr(N, deg, groups=1, dmin=6, bins=0, seed=0):
    rng = np.random.default_rng(seed)
    rows = [np.sort(rng.choice(N, size=min(k, N), replace=False))
            for k in np.broadcast_to(deg, (N, ))]
    row = np.concatenate([[0], np.cumsum([r.size for r in rows])])
    col = np.concatenate(rows)
    d = rng.integers(dmin, dmin + 40, size=(groups, col.size))
    if bins:
        d = dmin + (d - dmin) // bins * bins
    return CSR(N, row, col, rng.uniform(0.05, 0.5, col.size), d)


def _sim(csr, P, ring, launch, **kw):
    m = M.JansenRit()
    c = CF.Sigmoidal(m)
    rs = 1.0 if ring == 'f32' else 1.0 / c.param['cmax']
    a = np.linspace(0.0, 1.0, P).astype(np.float32)
    gs = None if csr.n_group == 1 else -(-P // csr.n_group // 64) * 64
    sim = Simulation(m, c, SC.EulerStep(0.05), csr, P, params={'c:a': a},
                     kinds={'c:a': 'inst'}, ring_dtype=ring, ring_scale=rs,
                     group_size=gs, horizon=60, **dict(launch, **kw))
    x0 = m.initial_state(csr.nnode, P, np.random.default_rng(5))
    sim.set_state(x0)
    sim.init_history('zeros')
    return sim, x0, a, gs


@pytest.mark.parametrize('N,deg,P,groups,ring,ipl,L', [
    (2, 1, 1, 1, 'f32', 1, 2),
    (9, 5, 65, 1, 'f32', 1, 7),
    (33, 16, 130, 1, 'f32', 2, 5),
    (70, 66, 64, 1, 'bf16', 2, 7),
    (140, 139, 70, 1, 'f32', 4, 4),
    (31, 12, 192, 3, 'f32', 1, 6),
    (40, 17, 300, 1, 'u8', 4, 7),
    (65, 33, 129, 1, 'f16', 1, 7)])
def test_sums_ahead_equal_single_steps(N, deg, P, groups, ring, ipl, L):
    csr = _csr(N, deg, groups)
    steps = 3 * L + 1          # ends on a partial launch
    blocked = dict(ipl=ipl, waves=1, node_block=1, steps_per_launch=L)
    got = []
    for la in (dict(ipl=ipl, waves=2, node_block=2, steps_per_launch=1),
               blocked, dict(blocked, pace=1)):
        sim, x0, a, gs = _sim(csr, P, ring, la)
        sim.set_exec(graph=False)
        sim.run(steps)
        got.append((sim.get_state(), sim.get_ring()))
    for x, r in got[1:]:
        assert np.array_equal(x, got[0][0])
        assert np.array_equal(r, got[0][1])
    if ring == 'f32' and groups == 1:
        ref = oracle_for('JansenRit', 'Sigmoidal', csr, P, 60, 0.05, 'euler',
                         cparams={'a': a})
        ref.set_state(x0)
        ref.init_history('zeros')
        ref.run(steps)
        assert scaled_err(got[1][0], ref.get_state()) < 1e-5


def test_sums_ahead_where_values_are_reused():
    """2,600 waves with two delays (every value gathered many times): the
    launches are two kernels for the reuse, not for want of waves."""
    csr = _csr(260, 40, bins=20)
    got = []
    for la in (dict(ipl=1, waves=2, node_block=2, steps_per_launch=1),
               dict(ipl=1, waves=1, node_block=1, steps_per_launch=7)):
        sim, _, _, _ = _sim(csr, 640, 'f32', la)
        sim.run(20)
        got.append(sim.get_state())
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize('N,deg,P,groups,ipl,L,window', [
    (2, 1, 1, 1, 1, 2, 10),
    (9, 5, 65, 1, 1, 7, 20),
    (140, 139, 70, 1, 2, 4, 30),
    (31, 12, 192, 3, 1, 6, 15),
    (33, 20, 300, 1, 4, 7, 60)])
def test_reverse_sums_ahead_equal_single_steps(N, deg, P, groups, ipl, L,
                                               window):
    """The adjoint of blocked launches (transposed gathers ahead of the
    recursion) against one reverse step per launch, bit for bit."""
    csr = _csr(N, deg, groups)
    m = M.MontbrioPazoRoxin()
    rng = np.random.default_rng(2)
    x0 = m.initial_state(N, P, rng)
    par = {'c:a': rng.uniform(0, 0.1, P).astype(np.float32),
           'm:eta': -5 + rng.uniform(-.2, .2, (N, P)).astype(np.float32)}
    ds = rng.standard_normal((12, N, P)).astype(np.float32)
    gs = None if groups == 1 else P // groups
    got = []
    for la in (dict(ipl=ipl, waves=2, node_block=2, steps_per_launch=1),
               dict(ipl=ipl, waves=1, node_block=1, steps_per_launch=L)):
        sim = Simulation(m, CF.Linear(m), SC.EulerMaryuyamaStep(0.01, 0.01),
                         csr, P, params=par,
                         kinds={'c:a': 'inst', 'm:eta': 'ni'}, horizon=60,
                         group_size=gs, tavg_period=5, sample_slots=12,
                         adjoint=True, **la)
        sim.set_state(x0)
        sim.init_history('zeros')
        sim.set_noise(seed=4)
        sim.checkpoint_run(60, window)
        got.append(sim.adjoint(ds, 0))
    for key in ('c:a', 'm:eta'):
        assert np.isfinite(got[0][key]).all() and np.any(got[0][key])
        assert np.array_equal(got[0][key], got[1][key])
