"""Per-step series past one chunk of steps (1024) and with more workgroups
than slots (32): extremes and counts of every step equal the oracle's, from
the loops that take one and several steps per launch, 2D and 1D."""
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


@pytest.mark.parametrize("n", [1023, 1024, 1025, 2060])
@pytest.mark.parametrize("tile_y", [0, 8], ids=["several", "one"])
def test_film_series_past_a_chunk(S, n, tile_y):
    Lx, Ly = 50, 21
    print(f"[series] n={n} tile_y={tile_y}", flush=True)
    h0 = O.init_normal(Lx, Ly, 8, 1.0, 0.05)
    ost = O.State(Lx, Ly)
    ost.height[...] = h0
    ref = O.time_loop(ost, O.params(gamma=0.01, tdump=10 ** 9), n, dh=True)
    sysc = S.SysConst(Lx, Ly, S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.01))
    st = S.Sys(sysc, "GPU")
    st.height = h0
    S.equilibrium(st, sysc)
    dh, top = [], []
    S.time_loop(sysc, st, dh, maxheight=top, tile_y=tile_y)
    assert np.array_equal(np.array(dh), ref["dh"])
    assert len(top) == n and top[0] == h0.max()


@pytest.mark.parametrize("T", [np.float64, np.float32])
def test_more_workgroups_than_slots(S, T):
    """One step of a 1300 x 1290 film (hundreds of tiles): the input's own extremes and count."""
    h0 = np.asfortranarray(0.06 + 0.01 * np.random.default_rng(1).standard_normal((1300, 1290)))
    for n in (1, 3):
        sysc = S.SysConst(1300, 1290, S.Taumucs(Tmax=n, tdump=10 ** 9))
        st = S.Sys(sysc, "GPU", T=T)
        st.set_reference_height(0.06)
        st.height = h0
        h = st.get("height", np.float64)
        dh, area = [], []
        S.time_loop(sysc, st, dh)
        assert len(dh) == n and dh[0] == h.max() - h.min()
        st.height = h0
        S.time_loop(sysc, st, S.wetted, area)
        assert len(area) == n and area[0] == int((h > 0.055).sum())


@pytest.mark.parametrize("variant", [0, 1])
def test_line_series_past_a_chunk(S, variant):
    L, n = 1500, 1100
    h = 1.0 + 0.05 * np.sin(2 * np.pi * 3 * np.arange(L) / L)
    ost = O.State1D(L)
    ost.height[...] = h
    ref = O.time_loop_1d(ost, O.params(gamma=0.01, tdump=10 ** 9), n, dh=True, wetted=0.055)
    sysc = S.SysConst_1D(L, S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.01))
    st = S.Sys(sysc)
    st.height = h
    dh = []
    S.time_loop(sysc, st, dh, variant=variant)
    assert np.array_equal(np.array(dh), ref["dh"])
