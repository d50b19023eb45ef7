"""FP64 loops over the whole range of the type: velocities down to the subnormals
(ahead of a front they fall off by about half per node and step, so that a flat
film some 900 nodes away holds them after as many steps), heights and velocities
that overflow, infinite ones.  The kernels of several steps per launch and the
strips have the bits of the one-step tiles, whose divisions are the compiler's."""
import numpy as np
import pytest

import oracle as O
from test_gpu_multi import films

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def tiny(shape, seed, top):
    """Signed magnitudes spread over 2^-1074 .. 2^top, and zeros."""
    rng = np.random.default_rng(seed)
    with np.errstate(under="ignore"):
        u = np.ldexp(rng.uniform(1, 2, shape) * rng.choice([-1.0, 1.0], shape),
                     rng.integers(-1075, top, shape))
    u[rng.random(shape) < 0.1] = 0.0
    return np.asfortranarray(u)


def same(got, want, what):
    for name in want:
        g, w = got[name], want[name]
        bad = (g != w) & ~(np.isnan(g) & np.isnan(w))
        assert not bad.any(), (what, name, int(bad.sum()), np.argwhere(bad)[:3], g[bad][:3], w[bad][:3])


def run2d(S, shape, n, h, u, v, thermal=False, tile_y=0, **kw):
    sysc, st, _, _ = films(S, shape, n, **kw)
    st.height, st.velx, st.vely = h, u, v
    S.equilibrium(st, sysc)
    st.copy("ftemp", "feq")
    S.time_loop(sysc, st, thermal=thermal, seed=5, tile_y=tile_y)
    out = {k: st.get(k) for k in ("height", "velx", "vely", "fout", "pressure", "Fx")}
    st.close()
    return out


def run1d(S, L, n, h, u, args=(), thermal=False, variant=0, **kw):
    par = {{"tau": "τ"}.get(k, k): v for k, v in kw.items()}
    sysc = S.SysConst_1D(L, S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.01, **par))
    st = S.Sys(sysc)
    st.height, st.vel = h, u
    S.equilibrium(st, sysc)
    st.ftemp = st.get("feq")
    S.time_loop(sysc, st, *args, thermal=thermal, seed=5, variant=variant)
    out = {k: st.get(k) for k in ("height", "vel", "fout", "pressure", "F")}
    st.close()
    return out


OPTS = {"thermal": dict(kbt=1e-320), "gravity": dict(g=1e-290), "tau": dict(tau=0.8)}


# several steps per launch, strips; the one-step tiles divide as the compiler does
@pytest.mark.parametrize("shape", [(100, 101), (257, 250), (700, 640), (1100, 301)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("opt", ["plain", "thermal", "gravity", "tau"])
@pytest.mark.parametrize("top", [-1040, -960, -880])
def test_tiny_velocities_2d(S, shape, opt, top):
    print(f"[range] {shape} {opt} {top}", flush=True)
    h = np.full(shape, 0.7, order="F")  # no pressure gradient: the velocities stay small
    u, v = tiny(shape, 2, top), tiny(shape, 3, top)
    kw = dict(thermal=opt == "thermal", **OPTS.get(opt, {}))
    want = run2d(S, shape, 7, h, u, v, tile_y=8, **kw)
    if opt in ("plain", "tau"):
        assert 0 < np.abs(want["velx"]).max() < 2.0 ** (top + 30)
    same(run2d(S, shape, 7, h, u, v, **kw), want, (shape, opt))


@pytest.mark.parametrize("shape", [(64, 50), (300, 256)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_tiny_velocities_oracle(S, shape):
    n = 6
    sysc, st, prm, ost = films(S, shape, n)
    u, v = tiny(shape, 2, -960), tiny(shape, 3, -960)
    for o in (st, ost):
        h = np.full(shape, 0.7, order="F")
        if o is st:
            st.height, st.velx, st.vely = h, u, v
        else:
            ost.height[...], ost.velx[...], ost.vely[...] = h, u, v
    with np.errstate(all="ignore"):
        O.time_loop(ost, prm, n)
    S.time_loop(sysc, st)
    same({k: st.get(k) for k in ("height", "velx", "fout")},
         {k: getattr(ost, k) for k in ("height", "velx", "fout")}, shape)
    st.close()


@pytest.mark.parametrize("L", [64, 1000, 70000, 300000, 2000000])
@pytest.mark.parametrize("opt", ["plain", "thermal", "gravity", "tau", "theta"])
@pytest.mark.parametrize("top", [-1040, -960, -880])
def test_tiny_velocities_1d(S, L, opt, top):
    print(f"[range] {L} {opt} {top}", flush=True)
    h, u = np.full(L, 0.7), tiny(L, 2, top)
    kw = dict(thermal=opt == "thermal", **OPTS.get(opt, {}))
    if opt == "theta":
        kw["args"] = (np.full(L, 1 / 9),)
    want = run1d(S, L, 13, h, u, variant=1, **kw)
    if opt not in ("thermal", "gravity"):
        assert 0 < np.abs(want["vel"]).max() < 2.0 ** (top + 30)
    same(run1d(S, L, 13, h, u, **kw), want, (L, opt))


# heights and velocities beyond the range that the shared reciprocal covers
VALUES = [(np.inf, 0.0), (-np.inf, 0.0), (np.nan, 0.0), (1e200, 1e-3), (1e-310, 1e-3), (0.0, 1e-3),
          (-0.05, 1e-3), (1.0, 1e280), (1.0, np.inf), (-1e-9, 1e250)]


@pytest.mark.parametrize("hv,uv", VALUES, ids=[f"{a}_{b}" for a, b in VALUES])
def test_extreme_values(S, hv, uv):
    rng = np.random.default_rng(6)
    for n in (1, 2, 4):
        for g in (0.0, 0.001):
            for shape in ((60, 50), (700, 640)):
                h = np.asfortranarray(1 + 0.01 * rng.standard_normal(shape))
                u, v = (np.asfortranarray(1e-3 * rng.standard_normal(shape)) for _ in range(2))
                h[30, 20], u[30, 20] = hv, uv
                want = run2d(S, shape, n, h, u, v, g=g, tile_y=8)
                same(run2d(S, shape, n, h, u, v, g=g), want, (shape, g, n))
            for L in (300, 90000):
                h, u = 1 + 0.01 * rng.standard_normal(L), 1e-3 * rng.standard_normal(L)
                h[200], u[200] = hv, uv
                want = run1d(S, L, n, h, u, g=g, variant=1)
                same(run1d(S, L, n, h, u, g=g), want, (L, g, n))
