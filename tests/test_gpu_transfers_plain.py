"""Uploads, downloads and reductions of a process that gets no pinned memory: the
runtime's own copy, converted on the host."""
import os
import shutil
import subprocess
import sys
import textwrap

import numpy as np
import pytest

import test_gpu_transfers as big

pytestmark = pytest.mark.gpu
S = big.S


# hipHostMalloc as where the host has no memory left to pin
SHIM = "int calls; int hipHostMalloc(void** p, unsigned long n, unsigned f) { ++calls; *p = 0; return 2; }"
CHILD = """
    import ctypes, sys
    shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the library that calls it
    sys.path[:0] = sys.argv[2:]
    import numpy as np, swalbe as S
    import test_gpu_transfers as big
    for shape in ((7, 5), (300, 200), (513, 257), (1153, 911)):
        for T in (np.float64, np.float32):
            for host in (np.float64, np.float32):
                big.test_fields_cross_as_the_formula_says(S, shape, host, T)
    big.test_raw_round_trip_keeps_every_bit(S)
    st = S.HipState(30, 20)
    st.height = np.asfortranarray(np.random.default_rng(1).uniform(1, 2, (30, 20)))
    assert st.reduce()["max"] == st.get("height").max()
    sysc = S.SysConst_1D(5000, S.Taumucs())
    line = S.Sys(sysc)
    h = np.random.default_rng(1).uniform(1, 2, 5000)
    line.height = h
    assert np.array_equal(line.get("height"), h)
    assert ctypes.c_int.in_dll(shim, "calls").value > 20
    print("plain transfers", flush=True)
"""


def test_without_pinned_memory(S, tmp_path):
    if not shutil.which("gcc"):
        pytest.skip("no gcc for the shim")
    src, lib = tmp_path / "shim.c", tmp_path / "libshim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    pkg = os.path.dirname(os.path.dirname(os.path.abspath(S.__file__)))
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(CHILD), str(lib), pkg, here],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "plain transfers" in r.stdout, r.stdout + r.stderr
