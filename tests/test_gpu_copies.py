"""Host copies of device arrays with and without padded instances, past one
piece of the staging workspace (32 MB), round trip bit for bit."""

import numpy as np
import pytest

from tvb_hpc import coupling as CF
from tvb_hpc import model as M
from tvb_hpc import scheme as SC
from tvb_hpc.hip import Simulation
from tvb_hpc.network import CSR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ring,P', [('f32', 100), ('f32', 128), ('bf16', 100),
                                    ('u8', 333)])
def test_ring_and_state_round_trip(ring, P):
    N, H = 60, 1500
    csr = CSR(N, np.arange(N + 1), np.arange(N)[::-1].copy(), np.ones(N),
              np.full(N, 3))
    m = M.JansenRit()
    c = CF.Sigmoidal(m)
    sim = Simulation(m, c, SC.EulerStep(0.05), csr, P, horizon=H,
                     params={'c:a': np.ones(P, np.float32)},
                     kinds={'c:a': 'inst'}, ring_dtype=ring,
                     ring_scale=1.0 if ring == 'f32' else 200.0)
    rng = np.random.default_rng(3)
    # values every ring type holds exactly
    r = {'u8': lambda z: z.astype(np.float32) / np.float32(255),
         'bf16': lambda z: (z / 256).astype(np.float32),
         'f32': lambda z: (z / 7).astype(np.float32)}[ring](
             rng.integers(0, 256, (H, 1, N, P)))
    assert 4 * r.size > 32 << 20
    sim.set_ring(r)
    assert np.array_equal(sim.get_ring(), r)
    x = rng.standard_normal((6, N, P)).astype(np.float32)
    sim.set_state(x)
    assert np.array_equal(sim.get_state(), x)


def test_threads_sharing_a_context_read_their_own_states():
    """Each thread's strided copies go through the context's one workspace."""
    import threading
    N, P = 50, 300
    csr = CSR(N, np.arange(N + 1), np.arange(N)[::-1].copy(), np.ones(N),
              np.full(N, 3))
    m = M.JansenRit()
    sims, xs, bad = [], [], []
    for k in range(4):
        sims.append(Simulation(m, CF.Sigmoidal(m), SC.EulerStep(0.05), csr, P,
                               horizon=8))
        xs.append(np.random.default_rng(k).standard_normal(
            (6, N, P)).astype(np.float32))
        sims[k].set_state(xs[k])

    def work(k):
        for _ in range(60):
            if not np.array_equal(sims[k].get_state(), xs[k]):
                bad.append(k)
            sims[k].set_state(xs[k])

    ts = [threading.Thread(target=work, args=(k, )) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
