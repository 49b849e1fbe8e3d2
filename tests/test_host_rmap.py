"""The index type of a region spread follows the larger of its two arrays:
with more regions than vertices that is the regions'."""

import pytest

from host_hip import run

CODE = r'''
V, R, C = %d, %d, %d
rm = hip.RegionMap(np.arange(V) %% R, R)
ptr = [ctypes.c_void_p() for _ in range(2)]
for p, n in zip(ptr, (R, V)):
    assert H.hipMalloc(ctypes.byref(p), ctypes.c_size_t(4 * n * C)) == 0
log()
hip.check(hip.lib().tvbx_rmap_from_avg(rm.h, 1, C, ptr[0], ptr[1]))
print(json.dumps(log()))
'''


# (65,536 columns; words of 16 bytes)
@pytest.mark.parametrize('V,R,wide', [
    (100, 80, False), (100, (1 << 18) - 1, False), (100, 1 << 18, True),
    (1 << 18, 100, True)])
def test_index_type_covers_both_arrays(V, R, wide):
    (name, _), = run(CODE % (V, R, 1 << 16))
    assert name.startswith('k_rmap_from_avg<ILi4E' + ('y' if wide else 'j'))


SUMS = r'''
V, R, C = %d, %d, %d
rm = hip.RegionMap(np.arange(V) %% R, R)
ptr = [ctypes.c_void_p() for _ in range(2)]
for p, n in zip(ptr, (V, R)):
    assert H.hipMalloc(ctypes.byref(p), ctypes.c_size_t(4 * n * C)) == 0
log()
hip.check(hip.lib().tvbx_rmap_to_avg(rm.h, 1, C, ptr[0], ptr[1]))
print(json.dumps(log()))
'''


# parcellations of a few hundred regions and finer ones
@pytest.mark.parametrize('V,R,C,short', [
    (20484, 148, 2, False), (20484, 200, 64, False), (20484, 1000, 2, True),
    (20484, 20000, 1, True), (515056, 400, 64, False), (515056, 1000, 2, False),
    (515056, 1000, 128, True), (515056, 100000, 16, True)])
def test_short_regions_take_a_wave_each(V, R, C, short):
    (name, _), = run(SUMS % (V, R, C))
    assert (name == 'k_rmap_to_avg_short') == short
    assert name.startswith('k_rmap_to_avg')
