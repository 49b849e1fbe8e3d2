"""The split blocked launch (a workgroup of three waves per node and 16
instances, edge terms and weights handed over through LDS) run on the host:
between two barriers the waves of a workgroup may run in any order, and the
result of a launch must be the same in all of them, and the oracle's.  Rows
of one, two and more blocks of 64 edges, ragged and full."""

import ctypes
import itertools
import os
import subprocess

import numpy as np
import pytest

from harness import oracle_for, scaled_err
from tvb_hpc import coupling as CF
from tvb_hpc import emit
from tvb_hpc import model as M
from tvb_hpc import scheme as SC
from tvb_hpc.network import CSR

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = '/opt/rocm/llvm/bin/clang++'


@pytest.fixture(scope='module')
def launch(tmp_path_factory):
    d = tmp_path_factory.mktemp('split')
    m = M.Kuramoto()
    spec = emit.KernelSpec(m, CF.Kuramoto(m), SC.EulerStep(0.05),
                           kinds={'c:a': 'inst'})
    src, lib = str(d / 'k.h'), str(d / 'k.so')
    with open(src, 'w') as fd:
        fd.write(spec.source())
    subprocess.check_call(
        [CLANG, '-std=c++17', '-O1', '-ffp-contract=off', '-mfma', '-w',
         '-shared', '-fPIC', '-DKERNEL_SRC="%s"' % src, '-o', lib,
         os.path.join(HERE, 'split_host.cpp')])
    return ctypes.CDLL(lib).split_launch


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize('deg', [(5, 64, 0), (65, 128), (129, 192),
                                 (193, 140, 1), (200, )])
def test_result_does_not_depend_on_the_order_of_the_waves(launch, deg):
    N, P, pitch, H, L, dt = 200, 16, 64, 30, 4, 0.05
    rng = np.random.default_rng(sum(deg))
    nodes = len(deg) + 1                # nodes with edges; the rest have none
    rows = [np.sort(rng.choice(N, size=k, replace=False))
            for k in (deg * 2)[:nodes]] + [np.zeros(0, int)] * (N - nodes)
    row = np.concatenate([[0], np.cumsum([r.size for r in rows])])
    col = np.concatenate(rows)
    csr = CSR(N, row, col, rng.uniform(0.05, 0.5, col.size),
              rng.integers(L - 1, H - L - 1, size=(1, col.size)))
    x0 = rng.uniform(0, 6, (1, N, P)).astype(np.float32)
    a = np.linspace(0.1, 1.0, P).astype(np.float32)
    ref = oracle_for('Kuramoto', 'Kuramoto', csr, P, H, dt, 'euler',
                     cparams={'a': a})
    ref.set_state(x0)
    ref.init_history('zeros')
    ref.run(L)

    cd = ((csr.delays[0].astype(np.uint32) << 16) | col).astype(np.uint32)
    w = csr.weight.astype(np.float32)
    pa = np.zeros(pitch, np.float32)
    pa[:P] = a
    omega = np.ones(N, np.float32)
    row = row.astype(np.int32)
    got = []
    for order in itertools.permutations(range(3)):
        for back in (0, 1):
            x = np.zeros((N, pitch), np.float32)
            x[:, :P] = x0[0]
            ring = np.zeros((H, N, pitch), np.float32)
            ring[0] = x
            bad = np.zeros(pitch, np.uint32)
            o = np.array(order, np.int32)
            uneven = launch(N, pitch, H, col.size, L, ctypes.c_float(dt),
                            _ptr(row), _ptr(cd), _ptr(w), _ptr(x), _ptr(ring),
                            _ptr(pa), _ptr(omega), _ptr(bad), _ptr(o), back)
            assert uneven == 0 and not bad.any()
            got.append((x, ring))
    for x, ring in got[1:]:
        assert np.array_equal(x, got[0][0])
        assert np.array_equal(ring, got[0][1])
    assert scaled_err(got[0][0][None, :, :P], ref.get_state()) < 1e-5
