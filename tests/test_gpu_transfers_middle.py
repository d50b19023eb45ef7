"""Fields around the sizes where a transfer changes its way: a workgroup and its
flag per 1024 elements, 16 of them from 16384, one chunk beyond 65536 and several
beyond a chunk; and doubles of an FP32 film, converted on the host beyond 1024."""
import threading

import numpy as np
import pytest

import test_gpu_transfers as big

pytestmark = pytest.mark.gpu
S = big.S


@pytest.mark.parametrize("shape", [(1024, 1), (1025, 1), (113, 1), (114, 1), (16384, 1), (16385, 1),
                                   (1820, 1), (1821, 1), (512, 128), (65537, 1), (7281, 1),
                                   (7282, 1), (131073, 1), (14565, 2)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("host", [np.float64, np.float32], ids=["h64", "h32"])
@pytest.mark.parametrize("T", [np.float64, np.float32], ids=["d64", "d32"])
def test_values(S, shape, host, T):
    big.test_fields_cross_as_the_formula_says(S, shape, host, T)


def test_special_values(S):
    """Infinities, NaN, subnormals and overflow of the FP32 type, on both sides of 1024."""
    for n in (900, 3000):
        a = np.ones((n, 1), order="F")
        a[:8, 0] = [np.inf, -np.inf, np.nan, 1e-40, -1e-46, 1e39, -0.0, 3.4028235e38]
        st = S.HipState(n, 1, T=np.float32)
        st.set("velx", a)
        with np.errstate(over="ignore"):
            want = a.astype(np.float32)
        assert np.array_equal(st.get("velx", np.float32), want, equal_nan=True)
        assert np.array_equal(st.get("velx", np.float64), want.astype(np.float64), equal_nan=True)
        assert np.array_equal(np.signbit(st.get("velx", np.float64)), np.signbit(want))
        st.close()


def test_threads(S):
    """Buffers change hands between transfers of one and of sixteen flags."""
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        films = [S.HipState(n, 3, T=T) for n, T in ((50 + k, np.float64), (2000 + k, np.float32),
                                                    (9000, np.float64))]
        for i in range(40):
            st = films[i % 3]
            a = np.asfortranarray(rng.normal(size=(st.Lx, 3)).astype(np.float32).astype(np.float64))
            st.set("velx", a)
            if not np.array_equal(st.get("velx", np.float64), a):
                bad.append((k, i))
        for st in films:
            st.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
