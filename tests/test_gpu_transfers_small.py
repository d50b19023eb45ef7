"""Fields of at most 4096 elements cross in one workgroup that tells the host by
a flag: the formula's values around that size and with nine planes, from many
threads at once, behind work that takes longer than the host polls for, and
reductions beside them."""
import threading

import numpy as np
import pytest

import test_gpu_transfers as big

pytestmark = pytest.mark.gpu
S = big.S


@pytest.mark.parametrize("shape", [(64, 64), (63, 65), (64, 65), (21, 21), (22, 22), (3, 1)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("host", [np.float64, np.float32], ids=["h64", "h32"])
@pytest.mark.parametrize("T", [np.float64, np.float32], ids=["d64", "d32"])
def test_values(S, shape, host, T):
    big.test_fields_cross_as_the_formula_says(S, shape, host, T)


def test_threads(S):
    bad = []

    def work(k):
        st = S.HipState(17 + k, 9, T=np.float64)
        rng = np.random.default_rng(k)
        for _ in range(100):
            a = np.asfortranarray(rng.normal(size=(17 + k, 9)))
            st.set("height", a)
            if not np.array_equal(st.get("height"), a):
                bad.append(k)
            r = st.reduce()
            if r["max"] != a.max() or r["min"] != a.min():
                bad.append((k, "reduce"))
        st.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_behind_long_work(S):
    """A loop of some milliseconds is queued before the download starts."""
    sysc = S.SysConst(40, 30, S.Taumucs(Tmax=4000, tdump=10 ** 9, γ=0.01))
    a, b = S.Sys(sysc), S.Sys(sysc)
    h = np.asfortranarray(1 + 0.01 * np.random.default_rng(1).normal(size=(40, 30)))
    a.height, b.height = h, h
    S.time_loop(sysc, a)
    S.time_loop(sysc, b)
    got, mx = a.get("height"), b.reduce()["max"]
    assert np.array_equal(got, b.get("height")) and mx == got.max()
    a.close()
    b.close()
