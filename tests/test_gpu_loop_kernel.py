"""Which kernel a loop of a film takes (swalbe_loop_kernel), by its size, type,
options and length: short loops, and the steps that the kernels of several
steps per launch and the strips are slower at, take the one-step tiles.  FP64
has the same bits either way (against the oracle); a short FP32 loop has the
tiles' bits, a longer one stays within the bounds of the FP32 kernels."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from test_gpu_multi import films, same

pytestmark = pytest.mark.gpu
TILES, SEVERAL, STRIPS = 0, 1, 2


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def kernel(S, shape, T, n, tau=1.0, thermal=False, final=True, **kw):
    sysc = S.SysConst(*shape, S.Taumucs(Tmax=n, τ=tau, kbt=1e-6))
    st = S.Sys(sysc, "GPU", T=T)
    o = S._lib.StepOpts()
    o.thermal, o.final_outputs_only = int(thermal), int(final)
    for k, v in kw.items():
        setattr(o, k, v)
    out = (C.c_int32 * 4)()
    S._lib.check(S._lib.lib().swalbe_loop_kernel(st.handle, C.byref(sysc.param.cparams()), n,
                                                 C.byref(o), out), "loop_kernel")
    st.close()
    return tuple(out)


F64, F32 = np.float64, np.float32
PATHS = [
    # shape, type, steps, options, kernel
    ((64, 64), F64, 1, {}, SEVERAL),
    ((512, 512), F64, 40, dict(tau=0.8), SEVERAL),
    ((900, 700), F64, 40, dict(tau=0.8, thermal=True), TILES),
    ((560, 560), F64, 40, dict(tau=0.8, thermal=True), TILES),
    ((1450, 1001), F64, 1, {}, STRIPS),
    ((1450, 1001), F64, 40, dict(final=False), TILES),
    ((1450, 1001), F32, 1, {}, STRIPS),
    ((2048, 2000), F32, 16, {}, TILES),
    ((2048, 2000), F32, 17, {}, STRIPS),
    ((2050, 2000), F32, 1, {}, STRIPS),
    ((2048, 2000), F32, 40, dict(variant=2), TILES),
    ((2048, 2000), F32, 40, dict(tile_y=16), TILES),
    ((750, 750), F32, 3, dict(tau=0.8), TILES),
    ((750, 750), F32, 4, dict(tau=0.8), SEVERAL),
    ((1603, 1001), F32, 8, dict(tau=0.8), TILES),
    ((1603, 1001), F32, 9, dict(tau=0.8), SEVERAL),
]


@pytest.mark.parametrize("shape,T,n,opts,want", PATHS,
                         ids=[f"{s[0]}x{s[1]}-{T.__name__}-{n}-{'_'.join(o)}" for s, T, n, o, _ in PATHS])
def test_rule(S, shape, T, n, opts, want):
    got = kernel(S, shape, T, n, **opts)
    assert got[0] == want, got
    assert got[3] == int(T is F64 and (got[0] == STRIPS or got[0] == SEVERAL and got[2] == 2)), got


# FP64 films of two steps per launch or of strips, whose single or last steps take the tiles
@pytest.mark.parametrize("shape", [(400, 399), (450, 451), (511, 505)], ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["plain", "gravity", "tau", "tau_thermal"])
@pytest.mark.parametrize("n", [1, 2, 3, 8])
def test_fp64_single_steps(S, shape, opt, n):
    kw = {"gravity": dict(g=0.002), "tau": dict(tau=0.8, g=0.002),
          "tau_thermal": dict(tau=1.2, kbt=1e-4)}.get(opt, {})
    got = kernel(S, shape, F64, n, tau=kw.get("tau", 1.0), thermal="kbt" in kw)
    assert got[0] != TILES and got[3] == 1, got  # several steps per launch (tau != 1), or strips
    th = "kbt" in kw
    sysc, st, prm, ost = films(S, shape, n, tdump=3, **kw)
    ref = O.time_loop(ost, prm, n, thermal=th, seed=21, dh=True, mass=True)
    dh, mass, shots = [], [], {}
    S.time_loop(sysc, st, dh, thermal=th, seed=21, mass=mass, snapshots=shots, snapshot_every=4)
    same(st, ost)
    assert np.array_equal(np.array(dh), ref["dh"])
    assert len(mass) == n // 3 and np.allclose(mass, ref["mass"][:len(mass)], rtol=1e-13)
    assert sorted(shots) == [f"h_{t}" for t in range(1, n + 1) if t % 4 == 0]
    st.close()


def fields(st, names=("height", "velx", "vely", "pressure", "fout")):
    return {k: st.get(k) for k in names}


@pytest.mark.parametrize("shape,tau,short,longer",
                         [((2048, 2000), 1.0, 16, 17), ((750, 750), 0.8, 3, 4),
                          ((1603, 1001), 0.8, 8, 9)], ids=["strips", "several", "carried"])
def test_fp32_short_loops(S, shape, tau, short, longer):
    """Short loops (one step among them) have the bits of the tiles; the first longer one, of the
    other kernel, is within twice the FP32 bounds of them (rel-L2 of h 1e-5, of ux 1e-3 each)."""
    print(f"[short] {shape} tau {tau}", flush=True)
    for n in (1, short, longer):
        got = []
        for variant in (0, 2):
            sysc, st, _, _ = films(S, shape, n, T=F32, tau=tau, amp=0.001)
            S.time_loop(sysc, st, variant=variant)
            got.append(fields(st))
            st.close()
        a, b = got
        if n <= short:
            for k in a:
                assert np.array_equal(a[k], b[k]), (n, k)
            continue
        assert not np.array_equal(a["velx"], b["velx"])
        rel = lambda x, y: np.linalg.norm(x - y) / np.linalg.norm(y)  # noqa: E731
        assert rel(a["height"].astype(F64), b["height"].astype(F64)) <= 2e-5
        assert rel(a["velx"].astype(F64), b["velx"].astype(F64)) <= 2e-3


@pytest.mark.parametrize("th", [False, True], ids=["plain", "thermal"])
def test_fp32_carried(S, th):
    """tau != 1, two steps per launch: the FP32 bounds against the oracle, and 9 + 9 steps give
    the bits of 18."""
    shape, n = (1603, 1001), 18
    print(f"[carried] {shape} thermal {th}", flush=True)
    assert kernel(S, shape, F32, n // 2, tau=0.8, thermal=th)[0] == SEVERAL
    kw = dict(tau=0.8, g=0.001, kbt=1e-6 if th else 0.0)
    sysc, st, prm, ost = films(S, shape, n, T=F32, amp=0.001, **kw)
    O.time_loop(ost, prm, n, thermal=th, seed=42)
    S.time_loop(sysc, st, thermal=th, seed=42)
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)  # noqa: E731
    h, ux = st.get("height", F64), st.get("velx", F64)
    assert rel(h, ost.height) <= 1e-5
    assert rel(h - h.mean(), ost.height - ost.height.mean()) <= 1e-3
    assert rel(ux, ost.velx) <= 1e-3
    for k in range(9):
        assert rel(st.get("fout", F64)[..., k], ost.fout[..., k]) <= 1e-3
    sys2, two, _, _ = films(S, shape, n // 2, T=F32, amp=0.001, **kw)
    for _ in range(2):
        S.time_loop(sys2, two, thermal=th, seed=42)
    for k, v in fields(st).items():
        assert np.array_equal(two.get(k), v), k
    two.close()
    st.close()
