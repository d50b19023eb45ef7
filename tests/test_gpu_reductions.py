"""Reductions over several workgroups and their finishing wave, at the sizes
where the number of partials changes (2D: one per 1024 nodes, at most 1024,
64 lanes; 1D: one per 4096 nodes, at most 256).  max, min and count are exact;
the sum of n positive terms in any tree order is within (log2 n + 64) ulp of
the exact sum (a lane adds at most 64 terms in a row here per 4096 nodes)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def check(got, h, thresh, terms):
    assert got["max"] == h.max() and got["min"] == h.min()
    assert got["count"] == int((h > thresh).sum())
    want = math.fsum(h.ravel())
    tol = (terms + 64) * np.finfo(float).eps * math.fsum(np.abs(h).ravel())
    assert abs(got["sum"] - want) <= tol, (got["sum"], want)


@pytest.mark.parametrize("shape", [(3, 1), (64, 64), (64, 129), (512, 513), (520, 513),
                                   (2048, 2049)], ids=lambda s: f"{s[0]}x{s[1]}")
def test_film_reduction(S, shape):
    h = np.asfortranarray(0.06 + 0.02 * np.random.default_rng(5).standard_normal(shape))
    st = S.HipState(*shape)
    st.height = h
    print(f"[reduce] {shape}", flush=True)
    check(st.reduce("height", 0.055), h, 0.055, 64)
    m = S.measure(st, 0.055, surface=False)
    assert m["count"] == int((h > 0.055).sum()) and m["max"] == h.max()
    st.close()


@pytest.mark.parametrize("L", [3, 4096, 4097, 8193, 262145, 1048576, 1048577, 3000001])
def test_line_reduction(S, L):
    h = 0.06 + 0.02 * np.random.default_rng(6).standard_normal(L)
    st = S.HipState1D(L)
    st.height = h
    print(f"[reduce] L={L}", flush=True)
    check(st.reduce("height", 0.055), h, 0.055, max(64, L // (256 * 256) + 1))
    inter = (np.random.default_rng(7).random(L) < 0.3).astype(float)
    st.set("interior", inter)
    got = st.reduce("height", 0.055, interior=True)["sum"]
    w = h - inter * h
    assert abs(got - math.fsum(w)) <= 256 * np.finfo(float).eps * math.fsum(np.abs(w))
    st.close()
