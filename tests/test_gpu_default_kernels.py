"""The kernels that a loop takes by default, over the options that reach them:
FP32 strips and several steps per launch with a θ field, a body force, gravity,
noise and their series, within the bounds of the FP32 step; the FP64 shapes of
two steps per launch; strips on narrow films; FP32 against FP64 after 10^4 steps.
And with a tile named, the store modes and the last-step-only stores of the
one-step kernels, which the default no longer runs."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from test_gpu_loop_kernel import F32, F64, SEVERAL, STRIPS, TILES, kernel
from test_gpu_multi import films, same

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


OPTS = {"plain": {}, "thermal": dict(kbt=1e-6), "gravity": dict(g=0.002), "theta": {}, "body": {},
        "tau_theta": dict(tau=0.8), "tau_body": dict(tau=0.8, g=0.001)}


def extras(S, shape, opt):
    """(time_loop arguments, oracle keywords)"""
    if opt.endswith("theta"):
        th = np.asfortranarray(np.random.default_rng(4).uniform(1 / 18, 1 / 6, shape))
        return (th,), dict(theta_field=th)
    if opt.endswith("body"):
        return (S.inclination, [2e-5, -1e-5]), dict(body=(2e-5, -1e-5, 1.0))
    return (), {}


# FP32: 8x8, 16x16, 32x16 of 1024 threads, 32x16 and 24x16 tiles; strips
@pytest.mark.parametrize("shape,path", [((61, 50), SEVERAL), ((150, 131), SEVERAL),
                                        ((300, 299), SEVERAL), ((345, 340), SEVERAL),
                                        ((420, 411), SEVERAL), ((500, 401), SEVERAL),
                                        ((700, 641), STRIPS),
                                        ((851, 849), STRIPS), ((200, 6200), STRIPS)],
                         ids=lambda s: f"{s[0]}x{s[1]}" if isinstance(s, tuple) else str(s))
@pytest.mark.parametrize("opt", OPTS)
def test_fp32_options(S, shape, path, opt):
    if path == STRIPS and "tau" in opt:
        pytest.skip("strips are for tau = 1")
    kw, n, th = OPTS[opt], 20, opt == "thermal"
    got = kernel(S, shape, F32, n, tau=kw.get("tau", 1.0), thermal=th)
    print(f"[default f32] {shape} {opt} {got}", flush=True)
    assert got[0] == path, got
    args, okw = extras(S, shape, opt)
    sysc, st, prm, ost = films(S, shape, n, T=F32, amp=0.001, **kw)
    O.time_loop(ost, prm, n, thermal=th, seed=42, **okw)
    S.time_loop(sysc, st, *args, thermal=th, seed=42)
    h = st.get("height", F64)
    assert rel(h, ost.height) <= 1e-5
    assert rel(h - h.mean(), ost.height - ost.height.mean()) <= 1e-3
    for k in ("velx", "vely"):
        assert rel(st.get(k, F64), getattr(ost, k)) <= 1e-3, k
    assert rel(st.get("fout", F64), ost.fout) <= 1e-5
    st.close()


@pytest.mark.parametrize("shape,path", [((150, 131), SEVERAL), ((300, 299), SEVERAL),
                                        ((500, 401), SEVERAL), ((851, 849), STRIPS)],
                         ids=lambda s: f"{s[0]}x{s[1]}" if isinstance(s, tuple) else str(s))
def test_fp32_series(S, shape, path):
    n = 25
    assert kernel(S, shape, F32, n, thermal=True)[0] == path
    for series in ("dh", "wetted"):
        sysc, st, prm, ost = films(S, shape, n, T=F32, kbt=1e-6, h0=0.06, amp=0.005)
        ref = O.time_loop(ost, prm, n, thermal=True, seed=2, dh=True, wetted=0.055)
        out = []
        S.time_loop(sysc, st, *((out,) if series == "dh" else (S.wetted, out)), thermal=True, seed=2)
        want = np.asarray(ref[series])
        if series == "dh":
            assert np.all(np.abs(np.array(out) - want) <= 1e-7 + 1e-4 * want)
        else:  # differ only where h sits within FP32 rounding of the threshold
            assert np.max(np.abs(np.array(out) - want)) <= 3 + 1e-4 * shape[0] * shape[1]
        st.close()


def c_loop(S, sysc, st, n, **kw):
    o = S._lib.StepOpts()
    for k, v in kw.items():
        setattr(o, k, v)
    S._lib.check(S._lib.lib().swalbe_time_loop(st.handle, C.byref(sysc.param.cparams()), n,
                                               C.byref(o)), "time_loop")
    st.t += n


# FP64, two steps per launch, tau = 1: a C caller that does not ask for final outputs only
@pytest.mark.parametrize("shape", [(400, 399), (450, 451), (511, 505)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["plain", "gravity", "thermal", "thermal_gravity"])
def test_fp64_two_step_tiles(S, shape, opt):
    kw, n = {}, 9
    if "thermal" in opt:
        kw["kbt"] = 1e-4
    if "gravity" in opt:
        kw["g"] = 0.002
    th = "thermal" in opt
    got = kernel(S, shape, F64, n, thermal=th, final=False)
    print(f"[default f64] {shape} {opt} {got}", flush=True)
    assert got[0] == SEVERAL and got[2] == 2, got
    sysc, st, prm, ost = films(S, shape, n, **kw)
    O.time_loop(ost, prm, n, thermal=th, seed=21)
    c_loop(S, sysc, st, n, thermal=int(th), seed=21, materialize=1)
    same(st, ost)
    st.close()


@pytest.mark.parametrize("shape", [(70, 30000), (130, 9001)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("th", [False, True], ids=["plain", "thermal"])
def test_fp64_narrow_strips(S, shape, th):
    n = 4
    got = kernel(S, shape, F64, n, thermal=th)
    print(f"[narrow] {shape} {got}", flush=True)
    assert got[0] == STRIPS, got
    sysc, st, prm, ost = films(S, shape, n, kbt=1e-4 if th else 0.0)
    O.time_loop(ost, prm, n, thermal=th, seed=21)
    S.time_loop(sysc, st, thermal=th, seed=21)
    same(st, ost, ("height", "velx", "vely", "pressure", "fout", "Fx"))
    st.close()


@pytest.mark.parametrize("shape,path", [((256, 250), SEVERAL), ((2000, 1500), STRIPS),
                                        ((4096, 4096), STRIPS)],
                         ids=lambda s: f"{s[0]}x{s[1]}" if isinstance(s, tuple) else str(s))
def test_fp32_vs_fp64_after_1e4_steps(S, shape, path):
    """The bounds of the 4096^2 rupture film in tiles: rel-L2 of h 1e-5, of its deviation from
    the mean 1e-4."""
    n = 10_000
    assert kernel(S, shape, F32, n, thermal=True)[0] == path
    prm = S.Taumucs(Tmax=n, tdump=10 ** 9, kbt=1e-6, γ=0.01, δ=1.0, n=9, m=3, hmin=0.1,
                    hcrit=0.05, θ=1 / 9)
    init = S.film_init(S.INIT_NORMAL, seed=1234, base=1.0, amp=0.001, href=1.0)
    h = {}
    for T in (F64, F32):
        print(f"[default 1e4] {shape} {T.__name__}", flush=True)
        sysc = S.SysConst(*shape, prm)
        st = S.Sys(sysc, "GPU", T=T, kind="thermal")
        st.set_reference_height(init.href)
        st.init_height(init)
        S.equilibrium(st, sysc)
        S.time_loop(sysc, st, thermal=True, seed=7, materialize=False)
        h[T] = st.get("height", F64)
        st.close()
    e, dyn = rel(h[F32], h[F64]), rel(h[F32] - h[F32].mean(), h[F64] - h[F64].mean())
    print(f"[default 1e4] {shape}: rel-L2 h {e:.3e}, dynamics {dyn:.3e}", flush=True)
    assert e <= 1e-5 and dyn <= 1e-4


@pytest.mark.parametrize("T,tile", [(F64, 8), (F64, 16), (F32, 8), (F32, 16)],
                         ids=["f64-8", "f64-16", "f32-8", "f32-16"])
def test_last_step_only_stores(S, T, tile):
    """final_outputs_only of the one-step tiles: every field, series and snapshot as with every
    step's f and p written."""
    shape, n = (130, 66), 40
    assert kernel(S, shape, T, n, tile_y=tile)[0] == TILES
    got = []
    for final in (False, True):
        sysc, st, _, _ = films(S, shape, n, T=T, kbt=1e-6, tdump=10, amp=0.01)
        dh, mass, snaps = [], [], {}
        S.time_loop(sysc, st, dh, thermal=True, seed=3, tile_y=tile, mass=mass, snapshots=snaps,
                    snapshot_every=7, final_outputs_only=final)
        got.append(({k: st.get(k) for k in ("height", "velx", "vely", "pressure", "fout", "ftemp",
                                            "feq", "Fx", "Fy")}, dh, mass, snaps))
        st.close()
    (a, dha, ma, sa), (b, dhb, mb, sb) = got
    for k in a:
        assert np.array_equal(a[k], b[k]), k
    assert dha == dhb and ma == mb
    assert sa.keys() == sb.keys() and all(np.array_equal(sa[k], sb[k]) for k in sa)


@pytest.mark.parametrize("T,tile", [(F64, 8), (F64, 16), (F32, 8), (F32, 16)],
                         ids=["f64-8", "f64-16", "f32-8", "f32-16"])
@pytest.mark.parametrize("final", [0, 1], ids=["every", "last"])
@pytest.mark.parametrize("tau", [1.0, 0.8], ids=["tau1", "tau0.8"])
def test_store_modes(S, T, tile, final, tau):
    """nontemporal 0, 1 and 2 of the one-step tiles give the same bits."""
    shape, n = (200, 130), 25
    got = []
    for mode in (0, 1, 2):
        sysc, st, _, _ = films(S, shape, n, T=T, kbt=1e-6, tau=tau, amp=0.01)
        c_loop(S, sysc, st, n, thermal=1, seed=4, tile_y=tile, nontemporal=mode,
               final_outputs_only=final)
        got.append({k: st.get(k) for k in ("height", "velx", "vely", "pressure", "fout")})
        st.close()
    for g in got[1:]:
        for k in g:
            assert np.array_equal(g[k], got[0][k]), k
