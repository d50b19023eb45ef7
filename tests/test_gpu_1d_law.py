"""The two copies of the 1D several-steps kernel's loop (n = 9, m = 3, g = 0;
anything else) and its body force: FP64 bit for bit against the oracle at one
and at eight nodes per lane, FP32 as one launch per step."""
import numpy as np
import pytest

import oracle as O
from test_gpu_1d import _run_hip, _setup

pytestmark = pytest.mark.gpu

LAWS = {"usual": dict(), "gravity": dict(prm=dict(g=0.05)), "n32": dict(prm=dict(n=3, m=2)),
        "n63": dict(prm=dict(n=6, m=3)), "n92": dict(prm=dict(n=9, m=2)),
        "body": dict(body=(1e-5, 1.0)), "body_n32": dict(body=(1e-5, 1.0), prm=dict(n=3, m=2))}


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


@pytest.mark.parametrize("L,n", [(1021, 45), (700001, 19)])
@pytest.mark.parametrize("name", list(LAWS))
def test_fp64_bitwise(S, name, L, n):
    print(f"1D law {name} L={L}", flush=True)
    sysc, prm, st, ost, okw, hkw, args = _setup(S, L, n, LAWS[name])
    sysc.param.tdump = prm.tdump = 10 ** 9
    okw["mass"] = False
    O.time_loop_1d(ost, prm, n, **okw)
    _run_hip(S, sysc, st, hkw, args, LAWS[name].get("body"))
    for f in ("height", "vel", "fout", "pressure", "F"):
        assert np.array_equal(st.get(f), getattr(ost, f)), f


@pytest.mark.parametrize("name", list(LAWS))
def test_fp32_equals_one_launch_per_step(S, name):
    got = []
    for variant in (0, 1):
        sysc, prm, st, ost, okw, hkw, args = _setup(S, 5003, 45, LAWS[name], T=np.float32,
                                                    variant=variant)
        sysc.param.tdump = 10 ** 9
        _run_hip(S, sysc, st, hkw, args, LAWS[name].get("body"))
        got.append([st.get(k) for k in ("height", "vel", "fout", "pressure")])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
