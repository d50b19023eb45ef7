"""Δh, maximum-height and wet-count series of films that hold NaN heights.  The
one-step kernels pass over NaN in max and min (all NaN: max -inf, min inf, so
Δh = -inf), and the kernels that take several steps per launch give the same
series."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def heights(shape, which):
    h = np.asfortranarray(1.0 + 0.01 * np.random.default_rng(3).standard_normal(shape))
    flat = h.reshape(-1, order="F")  # a view
    if which == "one":
        flat[flat.size // 2] = np.nan
    elif which == "negative":  # NaN with the sign bit
        flat[5] = -np.nan
    else:
        flat[:] = np.nan
    return h


def run2d(S, shape, which, T, n, series, **kw):
    sysc = S.SysConst(*shape, S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.01))
    st = S.Sys(sysc, "GPU", T=T)
    st.set_reference_height(1.0)
    st.height = heights(shape, which)
    out, top = [], []
    if series == "dh":
        S.time_loop(sysc, st, out, **kw)
    else:
        S.time_loop(sysc, st, S.wetted, out, maxheight=top, **kw)
    st.close()
    return np.array(out, dtype=float), np.array(top)


@pytest.mark.parametrize("which", ["one", "negative", "all"])
@pytest.mark.parametrize("shape", [(9, 7), (100, 101), (300, 299)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("T", [np.float64, np.float32], ids=["f64", "f32"])
def test_2d(S, shape, which, T):
    n = 4
    print(f"[nan] {shape} {which}", flush=True)
    h = heights(shape, which).astype(T).astype(np.float64)
    for series in ("dh", "wetted"):
        got, top = run2d(S, shape, which, T, n, series)
        want, wtop = run2d(S, shape, which, T, n, series, tile_y=8)
        # FP32 kernels agree to rounding: heights of order 1, a few steps
        tol = dict(rtol=0, atol=0 if T is np.float64 else 1e-5)
        np.testing.assert_allclose(got, want, **tol)
        np.testing.assert_allclose(top, wtop, **tol)
        if series == "dh":
            first = np.nanmax(h) - np.nanmin(h) if which != "all" else -np.inf
            np.testing.assert_allclose(got[0], first, rtol=0, atol=0 if T is np.float64 else 1e-6)
            assert not np.isnan(got).any()


@pytest.mark.parametrize("which", ["one", "negative", "all"])
@pytest.mark.parametrize("L", [9, 1024, 2000])
@pytest.mark.parametrize("T", [np.float64, np.float32], ids=["f64", "f32"])
def test_1d(S, L, which, T):
    """Against the kernel that holds the film in LDS (variant 2): every step's series."""
    n = 30
    got = []
    for variant in (2, 0):
        sysc = S.SysConst_1D(L, S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.01))
        st = S.Sys(sysc, T=T)
        st.height = heights((L,), which)
        dh = []
        S.time_loop(sysc, st, dh, variant=variant)
        got.append(np.array(dh))
        st.close()
    assert np.array_equal(*got) and not np.isnan(got[0]).any(), got
