"""Two-kernel launches that are chosen for repeated gathers, not for a small
history (a slot of 640 KB and more, few delays), against one step per launch,
bit for bit."""

import numpy as np
import pytest

from test_gpu_sums import _csr, _sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,deg,P,ring,ipl,dmin', [
    (260, 40, 640, 'f32', 1, 9), (260, 70, 1000, 'bf16', 2, 9),
    (300, 130, 2000, 'u8', 4, 8)])
def test_sums_ahead_where_values_are_reused(N, deg, P, ring, ipl, dmin):
    csr = _csr(N, deg, bins=20, dmin=dmin)
    got = []
    for la in (dict(ipl=ipl, waves=2, node_block=2, steps_per_launch=1),
               dict(ipl=ipl, waves=1, node_block=1, steps_per_launch=8)):
        sim, _, _, _ = _sim(csr, P, ring, la)
        if la['steps_per_launch'] > 1:
            assert sim.kernels() == 'tvbx_sums + tvbx_step_sums'
        sim.run(20)
        got.append((sim.get_state(), sim.get_ring()))
    for a, b in zip(*got):
        assert np.array_equal(a, b)
