"""libtvbx.so on the host's HIP runtime (host_hip.cpp), in a process of its
own: ``run(code)`` executes ``code`` after the prelude below and returns what
it printed as JSON on its last line."""

import atexit
import functools
import json
import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = '/opt/rocm/llvm/bin/clang++'

PRELUDE = r'''
import ctypes, json, os, re, subprocess, sys
sys.modules['torch'] = None         # its HIP runtime stays out
sys.path[:0] = [%(pkg)r, %(tests)r]
H = ctypes.CDLL(%(lib)r, ctypes.RTLD_GLOBAL)
H.host_hip_log.restype = ctypes.c_char_p
H.host_hip_held.restype = H.host_hip_left.restype = ctypes.c_long
H.host_hip_fail.argtypes = H.host_hip_fail_from.argtypes = [ctypes.c_long]
import numpy as np
from tvb_hpc import coupling as CF, hip, model as M, scheme as SC
from tvb_hpc.network import CSR


def _module(self, spec):
    src = subprocess.run([%(clang)r, '-E', '-P', '-x', 'c++', '-'],
                         input=spec.source(), capture_output=True, text=True,
                         check=True).stdout
    names = re.findall(r'\b(tvbx_\w+)\s*\(const tvbx_\w+_args ', src)
    img = (' '.join(names)).encode() + b'\0'
    buf, h = ctypes.create_string_buffer(img, len(img)), ctypes.c_void_p()
    hip.check(hip.lib().tvbx_module_load(self.h, buf, len(img),
                                         ctypes.byref(h)))
    return h


hip.Context.module = _module


def log():
    """The launches since the last call: [name, grid], names of the library's
    own kernels without their mangling."""
    out = []
    for line in H.host_hip_log().decode().splitlines():
        name, grid = line.rsplit(' ', 1)
        m = re.match(r'(graph )?_Z(\d+)(.*)', name)
        if m:
            name = (m[1] or '') + m[3][:int(m[2])] + \
                ('<' + m[3][int(m[2]):] if m[3][int(m[2])] == 'I' else '')
        out.append([name, grid])
    return out


def csr(N, deg, dmin, reuse=1, seed=0):
    "deg edges a row; every (delay, source) in about `reuse` of them"
    rng = np.random.default_rng(seed)
    col = np.concatenate([rng.choice(N, deg, replace=False)
                          for _ in range(N)])
    bins = max(1, deg // reuse)
    d = dmin + (np.arange(col.size) %% bins if reuse == 1
                else rng.integers(0, bins, col.size))
    return CSR(N, np.arange(N + 1) * deg, col, np.ones(col.size), d)
'''


@functools.lru_cache(None)
def _lib():
    d = tempfile.mkdtemp(prefix='tvbx_host_hip_')
    atexit.register(shutil.rmtree, d, True)
    so = os.path.join(d, 'libamdhip64.so.7')
    subprocess.check_call(
        [CLANG, '-std=c++17', '-O1', '-w', '-D__HIP_PLATFORM_AMD__',
         '-I/opt/rocm/include', '-shared', '-fPIC',
         '-Wl,-soname,libamdhip64.so.7',
         '-Wl,--version-script=' + os.path.join(HERE, 'host_hip.map'),
         '-o', so, os.path.join(HERE, 'host_hip.cpp')])
    return so


def run(code):
    pre = PRELUDE % dict(pkg=os.path.join(ROOT, 'tvb-hpc_amd'), tests=HERE,
                         lib=_lib(), clang=CLANG)
    r = subprocess.run([sys.executable, '-c', pre + code], cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads(r.stdout.strip().splitlines()[-1])
