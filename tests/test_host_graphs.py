"""Which runs go in captured graph windows: launches of one step and blocked
ones of fewer than 8 steps, whatever kernels they are; not those of 8 steps
or more, nor with graphs off.  The GPU's test of the same launches
(test_gpu_graphs.py) relies on this for its windows to be captured."""

import pytest

from host_hip import run

CODE = r'''
N, P = 24, 64
out = []
for model, L, graph in %r:
    if model == 'Kuramoto':
        m = M.Kuramoto()
        c, kw = CF.Kuramoto(m), {}
    else:
        m = M.JansenRit()
        c, kw = CF.Sigmoidal(m), {}
        if model == 'mfma':
            kw = dict(ring_dtype='bf16', ring_scale=200.0)
    blk = 4 if model == 'mfma' else 1
    s = hip.Simulation(m, c, SC.EulerStep(0.05), csr(N, 5, 12), P,
                       params={'c:a': np.full(P, 0.1, np.float32)},
                       kinds={'c:a': 'inst'}, waves=blk, node_block=blk,
                       steps_per_launch=L, horizon=40, **kw)
    if model == 'mfma':
        s.set_coupling('mfma')
    s.set_exec(graph=graph, window=16)
    log()
    s.run(2 * 16 + L)
    out.append([n for n, _ in log()])
print(json.dumps(out))
'''

CASES = [('sums', 4, True), ('Kuramoto', 4, True), ('mfma', 4, True),
         ('sums', 8, True), ('Kuramoto', 8, True), ('mfma', 8, True),
         ('sums', 4, False), ('Kuramoto', 4, False), ('mfma', 4, False)]
KERNELS = {'sums': ['tvbx_sums', 'tvbx_step_sums'],
           'Kuramoto': ['tvbx_step_split'],
           'mfma': ['tvbx_mfma_sums', 'tvbx_step_sums']}


def test_captured_windows():
    for (model, L, graph), got in zip(CASES, run(CODE % (CASES, ))):
        k = KERNELS[model]
        direct = k * (1 if graph and L < 8 else 32 // L + 1)
        win = ['graph ' + n for n in k * (16 // L)] + ['graph k_tick']
        want = (win * 2 if graph and L < 8 else []) + direct
        assert got == want, (model, L, graph)
