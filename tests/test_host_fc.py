"""An FC merge whose work buffers cannot be allocated fails with an error and
leaves the simulation as it was: the next call sets up what is missing and
launches what an undisturbed simulation does."""

import pytest

from host_hip import run

CODE = r'''
m = M.Generic2dOscillator()
c = csr(20, 3, 6)
def sim():
    return hip.Simulation(m, CF.Linear(m), SC.EulerStep(0.1), c, 70,
                          params={'c:a': np.full(70, 0.1, np.float32)},
                          tavg_period=2, fc=True, sample_slots=64)
def step(s):
    s.set_state(m.initial_state(20, 70, np.random.default_rng(0)))
    s.init_history('zeros')
    s.run(20)
    log()
a, b = sim(), sim()
step(a)
a.fc()
want = log()
step(b)
H.host_hip_fail(FAIL)
try:
    b.fc()
    failed = False
except hip.TvbxError:
    failed = True
H.host_hip_fail(-1)
first = log()
b.fc()
print(json.dumps([failed, first, log(), want]))
'''


@pytest.mark.parametrize('k', [0, 1, 2, 3])
def test_merge_after_a_failed_allocation(k):
    failed, first, got, want = run(CODE.replace('FAIL', str(k)))
    assert failed and not any(n == 'k_fc_update' for n, _ in first)
    assert any(n == 'k_fc_tile_table' for n, _ in want)
    assert [n for n, _ in first + got] == [n for n, _ in want]
