"""Films that march in strips of short segments (3 rows and up; the middle
sizes): FP64 bit for bit against the oracle with the last segment cut or a
single row, strips narrower than a wave's columns, odd rows and every option."""
import numpy as np
import pytest

import oracle as O
from test_gpu_march import film

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


@pytest.mark.parametrize("shape", [(640, 700), (700, 640), (851, 849), (1024, 1024), (4000, 301),
                                   (3001, 97), (177, 4001)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["plain", "thermal", "gravity", "series"])
def test_fp64_bitwise(S, shape, opt):
    n = 4
    print(f"[march short] {shape} {opt}", flush=True)
    kw = {"thermal": dict(kbt=1e-4), "gravity": dict(g=0.002)}.get(opt, {})
    sysc, st, prm, ost = film(S, shape, n, **kw)
    th = opt == "thermal"
    dh = []
    out = O.time_loop(ost, prm, n, thermal=th, seed=21, dh=opt == "series")
    S.time_loop(sysc, st, *((dh,) if opt == "series" else ()), thermal=th, seed=21)
    for name in ("height", "velx", "vely", "pressure", "fout", "ftemp", "Fx"):
        got, want = st.get(name), getattr(ost, name)
        assert np.array_equal(got, want), (name, np.argwhere(got != want)[:3])
    if opt == "series":
        assert np.array_equal(np.array(dh), out["dh"])
    st.close()


@pytest.mark.parametrize("shape", [(640, 700), (851, 849), (4000, 301)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("th", [False, True], ids=["plain", "thermal"])
def test_fp32_equals_tiles(S, shape, th):
    """Strips against the LDS tiles (variant 2): each is within rel-L2 1e-5 of
    h and 1e-3 of the velocities of the FP64 step, so twice that of the other."""
    got = []
    for variant in (0, 2):
        sysc, st, _, _ = film(S, shape, 20, T=np.float32, kbt=1e-4 if th else 0.0)
        S.time_loop(sysc, st, thermal=th, seed=21, variant=variant)
        got.append([st.get(k) for k in ("height", "velx", "vely")])
        st.close()
    for a, b, tol in zip(*got, (2e-5, 2e-3, 2e-3)):
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
