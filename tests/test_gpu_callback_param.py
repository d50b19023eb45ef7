"""time_loop with a callback that replaces sys.param: the ops that follow take
the new parameters, as the single ops do, in the same step (g, τ) and the
next (γ, μ, θ)."""
import numpy as np
import pytest

from test_gpu_callback import bits, film, ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


@pytest.mark.parametrize("thermal", [False, True], ids=["plain", "thermal"])
@pytest.mark.parametrize("field", [False, True], ids=["scalar", "theta"])
def test_replaced_parameters(S, thermal, field):
    shape, n = (65, 9), 3
    theta = np.asfortranarray(np.random.default_rng(4).uniform(1 / 18, 1 / 6, shape))
    out = []
    for run in ("loop", "ops"):
        kw = dict(kbt=1e-4) if thermal else {}
        sysc, st = film(S, shape, np.float64, n, **kw)
        log = []

        def f(measure, state):
            measure.append(state.reduce()["sum"])
            log.append(bits(state, thermal))
            if len(measure) == 1:
                sysc.param = S.Taumucs(Tmax=n, tdump=10 ** 9, γ=0.02, μ=0.2, τ=0.9, g=0.001, δ=0.7,
                                       kbt=3e-4, θ=1 / 12)
                if field:
                    sysc.param.θ = theta
        if run == "loop":
            S.time_loop(sysc, st, f, [], thermal=thermal, seed=9)
        else:
            ops(S, sysc, st, f, [], thermal, 9)
        log.append(bits(st, thermal))
        out.append(log)
        st.close()
    a, b = out
    assert len(a) == len(b) == n + 1
    assert not np.array_equal(a[1]["slipx"], a[2]["slipx"])
    for k, (x, y) in enumerate(zip(a, b)):
        for name in x:
            assert np.array_equal(x[name], y[name]), (k, name)
