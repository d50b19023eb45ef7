"""Large films whose loop writes f and p on its last step march in strips (one
wavefront per 58 columns and segment of rows): FP64 bit for bit against the
oracle, FP32 to its tolerance, on films whose last strip and segment are cut,
with an odd number of rows, and with the options and series of a step."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def film(S, shape, n, T=np.float64, g=0.0, kbt=0.0, amp=0.05, h0=1.0):
    Lx, Ly = shape
    h = O.init_normal(Lx, Ly, 5, h0, amp)
    rng = np.random.default_rng(Ly)
    ux, uy = (np.asfortranarray(rng.normal(0, 1e-3, shape)) for _ in range(2))
    ost = O.State(Lx, Ly)
    ost.height[...], ost.velx[...], ost.vely[...] = h, ux, uy
    sysc = S.SysConst(Lx, Ly, S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.01, g=g, kbt=kbt))
    st = S.Sys(sysc, "GPU", T=T)
    st.set_reference_height(h0, g)
    st.height, st.velx, st.vely = h, ux, uy
    return sysc, st, O.params(gamma=0.01, kbt=kbt, tdump=10 ** 9, g=g), ost


# the size rule: at least 24 rows of a strip per SIMD (1024 SIMDs)
SHAPES = [(1450, 1001), (5800, 251), (200, 6200), (64, 12500)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["plain", "thermal", "gravity", "theta", "body"])
def test_fp64_bitwise(S, shape, opt):
    n = 5
    print(f"[march] {shape} {opt}", flush=True)
    kw = {"thermal": dict(kbt=1e-4), "gravity": dict(g=0.002)}.get(opt, {})
    sysc, st, prm, ost = film(S, shape, n, **kw)
    th = opt == "thermal"
    okw, args = {}, ()
    if opt == "theta":
        th_f = np.asfortranarray(np.random.default_rng(4).uniform(1 / 18, 1 / 6, shape))
        okw, args = dict(theta_field=th_f), (th_f,)
    if opt == "body":
        okw, args = dict(body=(2e-5, -1e-5, 1.0)), (S.inclination, [2e-5, -1e-5])
    O.time_loop(ost, prm, n, thermal=th, seed=21, **okw)
    S.time_loop(sysc, st, *args, thermal=th, seed=21, final_outputs_only=True)
    for name in ("height", "velx", "vely", "pressure", "fout", "ftemp", "Fx"):
        got, want = st.get(name), getattr(ost, name)
        assert np.array_equal(got, want), (name, np.argwhere(got != want)[:3])
    st.close()


def test_series_and_masses(S):
    shape, n = (1450, 1001), 9
    sysc, st, prm, ost = film(S, shape, n, h0=0.06, amp=0.005)
    ref = O.time_loop(ost, prm, n, dh=True, wetted=0.055)
    dh = []
    S.time_loop(sysc, st, dh, final_outputs_only=True)
    assert np.array_equal(np.array(dh), ref["dh"])
    sysc, st, _, _ = film(S, shape, n, h0=0.06, amp=0.005)
    area = []
    S.time_loop(sysc, st, S.wetted, area, final_outputs_only=True)
    assert np.array_equal(np.array(area), ref["wetted"])


@pytest.mark.parametrize("shape", SHAPES[:2], ids=lambda s: f"{s[0]}x{s[1]}")
def test_fp32_tolerance_and_continuation(S, shape):
    """The bounds of the FP32 tiles (rel-L2 of h 1e-5, of its deviation and of ux 1e-3), and 4 + 4
    steps give the bits of 8."""
    n = 8
    print(f"[march] FP32 {shape}", flush=True)
    sysc, st, prm, ost = film(S, shape, n, T=np.float32, kbt=1e-6, amp=0.001)
    O.time_loop(ost, prm, n, thermal=True, seed=42)
    S.time_loop(sysc, st, thermal=True, seed=42, final_outputs_only=True)
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)  # noqa: E731
    h, ux = st.get("height", np.float64), st.get("velx", np.float64)
    assert rel(h, ost.height) <= 1e-5
    assert rel(h - h.mean(), ost.height - ost.height.mean()) <= 1e-3
    assert rel(ux, ost.velx) <= 1e-3
    sys2, two, _, _ = film(S, shape, n // 2, T=np.float32, kbt=1e-6, amp=0.001)
    for _ in range(2):
        S.time_loop(sys2, two, thermal=True, seed=42, final_outputs_only=True)
    for name in ("height", "velx", "fout", "pressure"):
        assert np.array_equal(two.get(name), st.get(name)), name
