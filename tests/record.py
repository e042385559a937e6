"""Launches of the library's host code, without a GPU: a snippet runs in a process of its own over a
HIP runtime that only writes launches down (native/record_hip.cpp)."""
import json
import os
import shutil
import subprocess
import sys

import pytest

from pned_amd import gpu

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, json, re, sys
rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
rec.record_take.restype = ctypes.c_char_p
rec.record_uploaded.restype = ctypes.c_size_t
sys.path.insert(0, sys.argv[2])
import numpy as np
from pned_amd import gpu, lattice, model
T = lattice.torus

def launches(f):
    "the kernels that f() launches: name, numeric template arguments, grid, block, LDS, LDS limit"
    rec.record_take()
    f()
    out = []
    for line in rec.record_take().decode().splitlines():
        name, *num = line.split()
        size = int(re.match("_ZN4pned([0-9]+)", name).group(1))
        at = 8 + len(str(size))
        m = re.match("I((?:[df]|L[ib][0-9]+E)*)E", name[at + size:])
        targs = [int(x) for x in re.findall("L[ib]([0-9]+)E", m.group(1))] if m else []
        out.append([name[at:at + size], targs] + [int(x) for x in num])
    return out

def offdiagonal(l1, l2, phi, field):
    "Kitaev-Heisenberg with symmetric off-diagonal exchange in a field: the most terms a bond can have"
    cl = T(l1, l2)
    c = model.set_lattice(20, phi)
    c.I11, c.I12, c.I11p, c.I12p, c.I11pp, c.I12pp = 0.21, 0.13, 0.21, 0.13, 0.21, 0.13
    H = model.bond_matrices(c, 2, "s12", field=field)
    mask, parity = model.local_mask(H, 2, "s12")
    return model.Operator(cl.n, 2, cl.ipair, cl.ibond_type, H, mask, parity, "s12", 0.0)

def general(n, seed):
    "all pairs of n sites, random Hermitian bond matrices: every term that two sites can have"
    rng = np.random.default_rng(seed)
    pairs = np.array([(a + 1, b + 1) for a in range(n) for b in range(a + 1, n)], dtype=np.int32)
    H = rng.standard_normal((9, 4, 4)) + 1j * rng.standard_normal((9, 4, 4))
    H = H + np.conj(np.transpose(H, (0, 2, 1)))
    return model.Operator(n, 2, pairs.reshape(-1), (np.arange(len(pairs)) % 9 + 1).astype(np.int32), H,
                          np.zeros(H.shape, dtype=bool), 1, "s12", 0.0)
"""


@pytest.fixture(scope="module")
def record(tmp_path_factory):
    """record(snippet): the JSON that the snippet prints as its last line."""
    cxx = shutil.which("g++") or shutil.which("c++")
    if not os.path.exists(gpu.LIB_PATH) or not cxx:
        pytest.skip("needs libpned_gpu.so and a C++ compiler")
    lib = str(tmp_path_factory.mktemp("record") / "librecord_hip.so")
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "native", "record_hip.cpp"), "-o",
                    lib], check=True)

    def run(snippet):
        r = subprocess.run([sys.executable, "-c", PRELUDE + snippet, lib, os.path.dirname(HERE)], capture_output=True,
                           text=True)
        assert r.returncode == 0, r.stdout + r.stderr
        return json.loads(r.stdout.splitlines()[-1])

    return run
