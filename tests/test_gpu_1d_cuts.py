"""1D films whose mass records or snapshots come every few steps, on both sides of
the rule that steps them in LDS instead of in registers: the fields of the other
kernels and of the oracle bit for bit, and the oracle's records."""
import ctypes as C

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


@pytest.mark.parametrize("L", [3, 64, 513, 1500, 2600])
@pytest.mark.parametrize("every", [1, 2, 3, 4, 7])
@pytest.mark.parametrize("kind", ["mass", "snapshots", "both"])
@pytest.mark.parametrize("th", [False, True], ids=["plain", "thermal"])
def test_cuts(S, L, every, kind, th):
    n = 23
    h = 0.5 + 0.05 * np.sin(np.arange(L) / 5)
    kbt = 1e-5 if th else 0.0
    tdump = every if kind != "snapshots" else 10 ** 9
    prm = O.params(gamma=0.01, kbt=kbt, tdump=tdump)
    ost = O.State1D(L)
    ost.height[...] = h
    ref = O.time_loop_1d(ost, prm, n, thermal=th, seed=5, mass=True, dh=True)
    for variant in (0, 1):
        sysc = S.SysConst_1D(L, S.Taumucs(Tmax=n, tdump=tdump, γ=0.01, kbt=kbt))
        st = S.Sys(sysc)
        st.height = h
        shots = np.zeros((n // every, L))
        kw = dict(snapshots=shots, dumping=every) if kind != "mass" else {}
        mass, dh = [], []
        S.time_loop(sysc, st, dh, thermal=th, seed=5, mass=mass, variant=variant, **kw)
        for name in ("height", "vel", "pressure", "fout", "F"):
            assert np.array_equal(st.get(name), getattr(ost, name)), (variant, name)
        assert np.array_equal(dh, ref["dh"])
        assert len(mass) == n // tdump and np.allclose(mass, ref["mass"][:len(mass)], rtol=1e-13)
        if kind != "mass":
            o2 = O.State1D(L)
            o2.height[...] = h
            for k in range(n // every):
                O.time_loop_1d(o2, prm, every, thermal=th, seed=5, t0=k * every)
                assert np.array_equal(shots[k], o2.height), (variant, k)
        st.close()


WAVE, RESIDENT = 1, 2
RULE = [
    # length, type, steps between mass records and between snapshots (0: none), noise, kernel
    (64, np.float64, 0, 0, False, WAVE),
    (64, np.float64, 1, 0, False, RESIDENT),
    (64, np.float64, 2, 0, False, RESIDENT),
    (64, np.float64, 50, 0, False, WAVE),
    (64, np.float32, 0, 4, False, RESIDENT),
    (64, np.float64, 0, 10, False, WAVE),
    (64, np.float64, 0, 50, False, WAVE),
    (1000, np.float64, 1, 0, False, RESIDENT),
    (1000, np.float64, 3, 0, False, WAVE),
    (2500, np.float64, 1, 0, True, WAVE),
    (3300, np.float64, 0, 1, False, RESIDENT),
    (3500, np.float64, 1, 1, False, WAVE),
]


@pytest.mark.parametrize("L,T,tdump,snap,th,want", RULE)
def test_rule(S, L, T, tdump, snap, th, want):
    n = 200
    sysc = S.SysConst_1D(L, S.Taumucs(Tmax=n, tdump=tdump or 10 ** 9, kbt=1e-6))
    st = S.Sys(sysc, T=T)
    o = S._lib.StepOpts1D()
    o.thermal = int(th)
    mass, shots = np.zeros(n), np.zeros((n, L))
    if tdump:
        o.mass_series = mass.ctypes.data_as(C.POINTER(C.c_double))
    if snap:
        o.snap_every, o.snap_series = snap, shots.ctypes.data_as(C.POINTER(C.c_double))
    out = C.c_int32(-1)
    S._lib.check(S._lib.lib().swalbe1d_loop_kernel(st.handle, C.byref(sysc.param.cparams()), n,
                                                   C.byref(o), C.byref(out)), "loop_kernel")
    assert out.value == want
    st.close()
