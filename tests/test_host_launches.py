"""Which kernels a blocked launch runs as, on both sides of each line of the
rule: small slots, the launch's length, history values gathered several times,
rings far beyond the caches; and what never is split."""

import pytest

from host_hip import run

ONE, TWO = 'tvbx_step_blocked', 'tvbx_sums + tvbx_step_sums'

CODE = r'''
out = []
for N, deg, P, ring, ipl, L, bins, span in %r:
    m = M.JansenRit()
    c = CF.Sigmoidal(m)
    rng = np.random.default_rng(0)
    col = np.concatenate([rng.choice(N, deg, replace=False)
                          for _ in range(N)])
    d = rng.integers(0, span, col.size)
    if bins:
        d = d // (span // bins) * (span // bins)
    g = CSR(N, np.arange(N + 1) * deg, col, np.ones(col.size), 33 + d)
    s = hip.Simulation(m, c, SC.EulerStep(0.05), g, P,
                       params={'c:a': np.full(P, 0.1, np.float32)},
                       kinds={'c:a': 'inst'}, ring_dtype=ring,
                       ring_scale=1.0 if ring == 'f32' else 200.0, ipl=ipl,
                       waves=1, node_block=1, steps_per_launch=L,
                       horizon=34 + span + L)
    log()
    s.run(L)
    out.append([' + '.join(n for n, _ in log()), s.kernels()])
    del s
print(json.dumps(out))
'''

# N, edges a row, P, ring, instances a lane, steps, delay bins (0: exact),
# delay span -> kernels
RULE = [
    ((84, 20, 1024, 'f32', 1, 8, 0, 60), TWO),       # 344 KB a slot
    ((84, 20, 1024, 'f32', 1, 4, 0, 60), ONE),       # ... short launch
    ((84, 60, 1024, 'f32', 1, 4, 0, 60), TWO),       # ... of long rows
    ((84, 20, 256, 'f32', 1, 4, 0, 60), TWO),        # 86 KB
    ((84, 20, 256, 'f32', 1, 3, 0, 60), ONE),
    ((84, 60, 1024, 'f32', 1, 2, 0, 60), ONE),
    ((998, 100, 64, 'f32', 1, 32, 0, 400), TWO),     # 255 KB
    ((998, 100, 128, 'f32', 1, 32, 0, 400), ONE),    # 511 KB
    ((400, 40, 512, 'f32', 2, 32, 0, 60), ONE),      # 819 KB
    ((400, 80, 1024, 'f32', 1, 8, 15, 60), TWO),     # 4 edges a value, 2 MB
    ((400, 80, 1024, 'f32', 1, 7, 15, 60), ONE),
    ((998, 100, 256, 'f32', 1, 8, 25, 400), ONE),    # 4 edges a value, 6.5 MB
    ((998, 100, 1024, 'f32', 1, 8, 100, 400), TWO),  # 1.6, ring 1.8 GB
    ((998, 100, 1024, 'f32', 1, 4, 100, 400), ONE),
    ((998, 100, 1024, 'f32', 1, 4, 25, 400), TWO),   # 4, ring 1.8 GB
    ((998, 100, 1024, 'f32', 1, 32, 0, 400), ONE),   # 1.1
    ((998, 100, 1024, 'bf16', 2, 32, 100, 400), ONE),
    ((998, 100, 1024, 'bf16', 4, 8, 25, 400), TWO),
    ((998, 100, 1024, 'u8', 4, 8, 50, 400), ONE),    # 2.2, ring 0.45 GB
    ((998, 100, 2048, 'u8', 4, 16, 30, 400), ONE),   # 3.4, ring 0.9 GB
    ((998, 100, 2048, 'u8', 4, 32, 20, 400), TWO),   # 5
    ((400, 40, 2048, 'u8', 4, 8, 30, 60), ONE),      # 1.8 edges a value
    ((400, 80, 2048, 'u8', 4, 8, 15, 60), TWO),      # 4, 2 MB
]


def test_kernels_of_a_launch():
    got = run(CODE % ([r[0] for r in RULE], ))
    for (shape, want), (kernels, told) in zip(RULE, got):
        assert kernels == want and told == want, (shape, kernels, told)


SPLIT = r'''
out = []
for N, deg, P, L in %r:
    m = M.Kuramoto()
    s = hip.Simulation(m, CF.Kuramoto(m), SC.EulerStep(0.05), csr(N, deg, 12),
                       P, params={'c:a': np.full(P, 0.1, np.float32)},
                       kinds={'c:a': 'inst'}, waves=1, node_block=1,
                       steps_per_launch=L, horizon=300)
    log()
    s.run(L)
    out.append([n for n, _ in log()] + [s.kernels()])
print(json.dumps(out))
'''


@pytest.mark.parametrize('shape,split', [
    ((76, 22, 64, 10), True), ((256, 20, 64, 2), True),
    ((257, 20, 64, 8), False),                    # more than 256 pairs
    ((128, 20, 128, 8), True), ((129, 20, 128, 8), False),
    ((200, 5, 64, 8), True), ((200, 5, 64, 4), False),   # short rows
    ((128, 5, 64, 4), True), ((128, 5, 64, 3), False)])
def test_split_launches(shape, split):
    name = 'tvbx_step_split' if split else 'tvbx_step_blocked'
    assert run(SPLIT % ([shape], )) == [[name, name]]
