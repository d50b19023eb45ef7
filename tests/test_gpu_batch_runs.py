"""A batch's step(n) writes the distributions and pressure of tau = 1 films on
the last of its n steps: after any cut of a run into calls and graph replays
every field has the bits of the same film stepped one step per call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("height", "velx", "vely", "pressure", "fout")


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def specs(S):
    T, fi = S.Taumucs, S.film_init
    return [(70, 33, T(Tmax=1, kbt=1e-6, γ=0.01), fi(S.INIT_NORMAL, thermal=True, seed=3, base=1.0,
                                                     amp=1e-3, href=1.0), 40),
            (96, 64, T(Tmax=1, τ=0.8, γ=0.01), fi(S.INIT_NORMAL, seed=4, base=1.0, amp=1e-3,
                                                  href=1.0), 40),
            (64, 16, T(Tmax=1, γ=0.01), fi(S.INIT_NORMAL, seed=5, base=1.0, amp=1e-3, href=1.0), 12),
            (130, 20, T(Tmax=1, γ=0.01), fi(S.INIT_NORMAL, seed=6, base=1.0, amp=1e-3, href=1.0),
             0)]


@pytest.mark.parametrize("graph", [0, 1, 3, 8])
@pytest.mark.parametrize("mix", [True, False], ids=["mixed", "tau1"])
def test_any_cut_of_a_run(S, graph, mix):
    films = [s for s in specs(S) if mix or s[2].τ == 1.0]
    a, b = S.Batch(64 << 20, 8, graph_steps=graph), S.Batch(64 << 20, 8)
    sa, sb = ([x.add(p, Lx, Ly, i, n) for Lx, Ly, p, i, n in films] for x in (a, b))
    for n in (1, 2, 9, 5, 16, 1, 17):
        print(f"[batch run] graph {graph} mixed {mix} step({n})", flush=True)
        a.step(n)
        for _ in range(n):
            b.step(1)
        for u, v in zip(sa, sb):
            assert a.status(u) == b.status(v)
            for name in FIELDS:
                assert np.array_equal(a.get(u, name), b.get(v, name)), (n, u, name)
    a.close()
    b.close()
