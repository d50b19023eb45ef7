"""Small 2D films take several steps per launch (time_loop's default): FP64
bit for bit against the oracle, FP32 to its tolerance, on films whose tiles
are cut by the edge, smaller than a tile's halo, and of every tile shape the
size rule picks; with the options that change a step and with series, mass
records and snapshots between and inside launches."""
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


def films(S, shape, n, T=np.float64, tau=1.0, g=0.0, kbt=0.0, tdump=10 ** 9, h0=1.0, amp=0.05):
    Lx, Ly = shape
    rng = np.random.default_rng(Lx + 7 * Ly)
    h = O.init_normal(Lx, Ly, 5, h0, amp)
    ux, uy = (np.asfortranarray(rng.normal(0, 1e-3, shape)) for _ in range(2))
    prm = O.params(tau=tau, gamma=0.01, kbt=kbt, tdump=tdump, g=g)
    ost = O.State(Lx, Ly)
    ost.height[...], ost.velx[...], ost.vely[...] = h, ux, uy
    ost.feq[...], _ = O.equilibrium(h, ux, uy, g)
    ost.ftemp[...] = ost.feq
    sysc = S.SysConst(Lx, Ly, S.Taumucs(Tmax=n, tdump=tdump, τ=tau, γ=0.01, g=g, kbt=kbt))
    st = S.Sys(sysc, "GPU", T=T)
    st.set_reference_height(h0, g)
    st.height, st.velx, st.vely = h, ux, uy
    S.equilibrium(st, sysc)
    st.ftemp = ost.feq
    return sysc, st, prm, ost


def same(st, ost, names=("height", "velx", "vely", "pressure", "fout", "Fx", "feq")):
    for name in names:
        got, want = st.get(name), getattr(ost, name)
        assert np.array_equal(got, want), (name, np.argwhere(got != want)[:3])


# each tile shape of the FP64 rule, with tiles cut at the right and top edges
SHAPES = [(1, 2), (5, 31), (100, 100), (128, 161), (255, 250), (256, 256), (300, 299), (345, 328),
          (511, 505)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["plain", "gravity", "thermal", "tau", "tau_thermal"])
def test_fp64_bitwise(S, shape, opt):
    if shape[0] * shape[1] > 70000 and opt in ("gravity", "tau_thermal"):
        pytest.skip("covered by the smaller films")
    n = 14 if shape[0] * shape[1] > 70000 else 29
    print(f"[multi] {shape} {opt}", flush=True)
    kw = {"gravity": dict(g=0.002), "thermal": dict(kbt=1e-4), "tau": dict(tau=0.8, g=0.002),
          "tau_thermal": dict(tau=1.2, kbt=1e-4)}.get(opt, {})
    sysc, st, prm, ost = films(S, shape, n, **kw)
    th = "kbt" in kw
    O.time_loop(ost, prm, n, thermal=th, seed=21)
    S.time_loop(sysc, st, thermal=th, seed=21)
    same(st, ost)


@pytest.mark.parametrize("n", [0, 1, 2, 3, 4, 7])
def test_short_loops_theta_and_body(S, n):
    shape = (70, 45)
    theta = np.asfortranarray(np.random.default_rng(4).uniform(1 / 18, 1 / 6, shape))
    sysc, st, prm, ost = films(S, shape, n)
    O.time_loop(ost, prm, n, theta_field=theta)
    S.time_loop(sysc, st, theta)
    same(st, ost, ("height", "velx", "vely"))
    sysc, st, prm, ost = films(S, shape, n)
    O.time_loop(ost, prm, n, body=(2e-5, -1e-5, 1.0))
    S.time_loop(sysc, st, S.inclination, [2e-5, -1e-5])
    same(st, ost, ("height", "velx", "vely"))


@pytest.mark.parametrize("shape", [(9, 7), (130, 70), (256, 250)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_series_masses_and_snapshots(S, shape):
    n, dump = 31, 7
    sysc, st, prm, ost = films(S, shape, n, tdump=5)
    ref = O.time_loop(ost, prm, n, dh=True, mass=True)
    dh, mass, shots = [], [], {}
    S.time_loop(sysc, st, dh, mass=mass, snapshots=shots, snapshot_every=dump)
    same(st, ost)
    assert np.array_equal(np.array(dh), ref["dh"])
    assert len(mass) == n // 5 and np.allclose(mass, ref["mass"][:len(mass)], rtol=1e-13)
    _, _, prm, ost = films(S, shape, n, tdump=5)
    for k in range(n // dump):
        O.time_loop(ost, prm, dump, t0=k * dump)
        assert np.array_equal(shots[f"h_{(k + 1) * dump}"], ost.height), k
    sysc, st, prm, ost = films(S, shape, n, h0=0.06, amp=0.01)
    ref = O.time_loop(ost, prm, n, wetted=0.055)
    area = []
    S.time_loop(sysc, st, S.wetted, area)
    assert np.array_equal(np.array(area), ref["wetted"])


@pytest.mark.parametrize("shape", [(2, 3), (100, 101), (250, 256), (399, 400), (511, 500)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["thermal", "tau"])
def test_fp32_tolerance_and_continuation(S, shape, opt):
    """The bounds of the one-step FP32 kernels (rel-L2 of h 1e-5, of its deviation from the mean
    and of ux 1e-3), and 20 + 20 steps give the bits of 40."""
    n = 40
    kw = dict(kbt=1e-6) if opt == "thermal" else dict(tau=0.8)
    th = opt == "thermal"
    print(f"[multi] FP32 {shape} {opt}", flush=True)
    sysc, st, prm, ost = films(S, shape, n, T=np.float32, amp=0.001, **kw)
    O.time_loop(ost, prm, n, thermal=th, seed=42)
    S.time_loop(sysc, st, thermal=th, seed=42)
    rel = lambda a, b: np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)  # noqa: E731
    h, ux = st.get("height", np.float64), st.get("velx", np.float64)
    assert rel(h, ost.height) <= 1e-5
    assert rel(h - h.mean(), ost.height - ost.height.mean()) <= 1e-3
    assert rel(ux, ost.velx) <= 1e-3
    sys2, two, _, _ = films(S, shape, n // 2, T=np.float32, amp=0.001, **kw)
    for _ in range(2):
        S.time_loop(sys2, two, thermal=th, seed=42)
    for name in ("height", "velx", "fout", "pressure"):
        assert np.array_equal(two.get(name), st.get(name)), name
