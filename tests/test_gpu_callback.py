"""time_loop with a callback runs a step in two kernels around it: every field
of the state has the bits that the single ops leave, before the callback and
after the last step, on one-node, thin, ragged and cut films (tiles of 64 x 8),
with the callback changing the state and the parameters."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SCALARS = ("height", "velx", "vely", "vsq", "pressure", "Fx", "Fy", "slipx", "slipy",
           "hgradpx", "hgradpy")
DISTS = ("fout", "ftemp", "feq")


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def film(S, shape, T, steps, **kw):
    Lx, Ly = shape
    rng = np.random.default_rng(Lx + 7 * Ly)
    sysc = S.SysConst(Lx, Ly, S.Taumucs(Tmax=steps, tdump=10 ** 9, γ=0.01, **kw))
    st = S.Sys(sysc, "GPU", T=T, kind="thermal")
    st.height = np.asfortranarray(1.0 + 0.1 * rng.normal(size=shape))
    st.velx, st.vely = (np.asfortranarray(1e-3 * rng.normal(size=shape)) for _ in range(2))
    st.ftemp = np.asfortranarray(0.1 + 0.01 * rng.normal(size=shape + (9,)))
    return sysc, st


def bits(st, thermal):
    names = SCALARS + DISTS + (("kbtx", "kbty") if thermal else ())
    return {k: np.array(st.get(k)) for k in names}


def touch(S, log, sysc, thermal):
    """A callback that logs, pushes the film and raises the viscosity."""
    def f(measure, st):
        measure.append(st.reduce()["sum"])
        log.append(bits(st, thermal))
        st.Fx = np.asfortranarray(st.get("Fx") + 1e-5)
        sysc.param.μ *= 1.25
    return f


def ops(S, sysc, st, f, measure, thermal, seed):
    from swalbe._lib import check, lib
    P = sysc.param
    for t in range(1, P.Tmax + 1):
        S.filmpressure(st, sysc)
        S.h_grad_p(st)
        S.slippage(st, sysc)
        if thermal:
            check(lib().swalbe_thermal(st.handle, P.kbt, P.μ, P.δ, seed, t), "thermal")
        S.force_sum(st, thermal)
        f(measure, st)
        S.equilibrium(st, sysc)
        S.BGKandStream(st, sysc)
        S.moments(st)


@pytest.mark.parametrize("T", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", [(1, 1), (2, 3), (5, 1), (63, 7), (64, 8), (65, 9), (131, 25)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("kw", [dict(), dict(τ=0.8, g=0.002), dict(kbt=1e-4, n=3, m=2),
                                dict(n=4, m=2, hmin=0.07, hcrit=0.02)],
                         ids=["default", "tau_g", "thermal32", "n4m2"])
def test_bits(S, T, shape, kw):
    print(f"[callback] {T.__name__} {shape} {kw}", flush=True)
    thermal, n = "kbt" in kw, 3
    out = []
    for run in ("loop", "ops"):
        sysc, st = film(S, shape, T, n, **kw)
        log, measure = [], []
        f = touch(S, log, sysc, thermal)
        if run == "loop":
            S.time_loop(sysc, st, f, measure, thermal=thermal, seed=9)
        else:
            ops(S, sysc, st, f, measure, thermal, 9)
        log.append(bits(st, thermal))
        out.append((log, measure))
        st.close()
    (a, ma), (b, mb) = out
    assert ma == mb and len(a) == len(b) == n + 1
    for k, (x, y) in enumerate(zip(a, b)):
        for name in x:
            assert np.array_equal(x[name], y[name], equal_nan=True), (k, name)
