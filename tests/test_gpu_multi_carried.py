"""Larger FP32 films with tau != 1 take two steps per launch: the bounds of the
one-step FP32 kernels against the oracle, on films whose tiles are cut at the
right and top edges, and the same bits however the run is cut."""
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


@pytest.mark.parametrize("shape", [(1603, 1001), (1001, 1607), (1600, 1008)],
                         ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("th", [False, True], ids=["plain", "thermal"])
def test_fp32(S, shape, th):
    n = 8
    print(f"[multi carried] {shape} thermal {th}", flush=True)
    kw = dict(tau=0.8, g=0.001, kbt=1e-6 if th else 0.0)
    sysc, st, prm, ost = films(S, shape, n, T=np.float32, amp=0.001, **kw)
    O.time_loop(ost, prm, n, thermal=th, seed=42)
    S.time_loop(sysc, st, thermal=th, seed=42)
    rel = lambda a, b: np.linalg.norm(a - b) / np.linalg.norm(b)  # noqa: E731
    h, ux = st.get("height", np.float64), st.get("velx", np.float64)
    assert rel(h, ost.height) <= 1e-5
    assert rel(h - h.mean(), ost.height - ost.height.mean()) <= 1e-3
    assert rel(ux, ost.velx) <= 1e-3
    for k in range(9):
        f = st.get("fout", np.float64)[..., k]
        assert rel(f, ost.fout[..., k]) <= 1e-3
    sys2, two, _, _ = films(S, shape, n // 2, T=np.float32, amp=0.001, **kw)
    for _ in range(2):
        S.time_loop(sys2, two, thermal=th, seed=42)
    for name in ("height", "velx", "vely", "fout", "pressure"):
        assert np.array_equal(two.get(name), st.get(name)), name
    two.close()
    st.close()
