"""The transposed connectome of the gradient is built as a whole or not at
all: after a call that found no memory for one of its arrays, the next one
builds it."""

from host_hip import run

CODE = r'''
m = M.MontbrioPazoRoxin()
c = csr(20, 4, 8)
ds = np.ones((12, 20, 64), np.float32)
def sim():
    s = hip.Simulation(m, CF.Linear(m), SC.EulerMaryuyamaStep(0.01, 0.01), c,
                       64, params={'c:a': np.full(64, 0.1, np.float32)},
                       kinds={'c:a': 'inst'}, tavg_period=5, sample_slots=12,
                       adjoint=True)
    s.set_state(m.initial_state(20, 64, np.random.default_rng(0)))
    s.init_history('zeros')
    s.checkpoint_run(60, 20)
    return s
out = []
for k in (-1, 0, 1, 2):
    held = H.host_hip_held()
    s = sim()
    failed = False
    if k >= 0:
        H.host_hip_fail_from(k)
        try:
            s.adjoint(ds, 0)
        except hip.TvbxError:
            failed = True
        H.host_hip_fail(-1)
    s.adjoint(ds, 0)
    out.append([failed, H.host_hip_held() - held])
    del s
print(json.dumps(out))
'''


def test_transpose_after_a_failed_allocation():
    out = run(CODE)
    assert [f for f, _ in out] == [False, True, True, True]
    # the same memory as undisturbed: no array is missing
    assert len({h for _, h in out}) == 1
