"""Series of short loops, whose device memory is kept with the film: many calls of
different lengths, with and without a series between them and beyond the kept
length, give the series of one long loop; and a loop that fails leaves nothing
behind."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from test_gpu_multi import films

pytestmark = pytest.mark.gpu
CUTS = [1, 2, 1, 64, 65, 3, 1, 100, 7]


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


@pytest.mark.parametrize("shape", [(70, 45), (450, 451), (700, 641)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_2d(S, shape):
    cuts = CUTS if shape[0] == 70 else [1, 2, 1, 5]
    n = sum(cuts)
    _, st0, prm, ost = films(S, shape, n, h0=0.06, amp=0.005)
    st0.close()
    ref = O.time_loop(ost, prm, n, dh=True, wetted=0.055)
    sysc, st, _, _ = films(S, shape, n, h0=0.06, amp=0.005)
    done = 0
    for i, k in enumerate(cuts):
        sysc.param.Tmax = k
        out = []
        if i % 3 == 2:
            S.time_loop(sysc, st)  # no series in between
        elif i % 3:
            S.time_loop(sysc, st, S.wetted, out)
            assert np.array_equal(out, ref["wetted"][done:done + k]), (i, k)
        else:
            S.time_loop(sysc, st, out)
            assert np.array_equal(out, ref["dh"][done:done + k]), (i, k)
        done += k
    assert np.array_equal(st.get("height"), ost.height)
    st.close()


def test_1d(S):
    L, n = 500, sum(CUTS)
    h = 0.06 + 0.005 * np.sin(np.arange(L) / 7)
    ost, prm = O.State1D(L), O.params(gamma=0.01, tdump=10 ** 9)
    ost.height[...] = h
    ref = O.time_loop_1d(ost, prm, n, dh=True, wetted=0.055)
    sysc = S.SysConst_1D(L, S.Taumucs(tdump=10 ** 9, γ=0.01))
    st = S.Sys(sysc)
    st.height = h
    done = 0
    for i, k in enumerate(CUTS):
        sysc.param.Tmax = k
        out = []
        S.time_loop(sysc, st, *((S.wetted, out) if i % 2 else (out,)))
        assert np.array_equal(out, ref["wetted" if i % 2 else "dh"][done:done + k]), (i, k)
        done += k
    st.close()


def test_after_an_error(S):
    """An option that is refused once the series have been set up."""
    shape = (40, 30)
    sysc, st, prm, ost = films(S, shape, 2)
    dh = np.zeros(2)
    o = S._lib.StepOpts()
    o.dh_series = dh.ctypes.data_as(C.POINTER(C.c_double))
    ms = C.c_double()
    rc = S._lib.lib().swalbe_time_loop_timed(st.handle, C.byref(sysc.param.cparams()), 2,
                                             C.byref(o), C.byref(ms))
    assert rc != 0
    ref = O.time_loop(ost, prm, 2, dh=True)
    for _ in range(2):
        out = []
        S.time_loop(sysc, st, out)
        if _ == 0:
            assert np.array_equal(out, ref["dh"])
    st.close()
