"""The 1D loop that takes several steps per launch in registers (the default
of time_loop): FP64 bit for bit against the oracle over the model's options,
at lengths where its windows wrap the film many times (3 nodes and up), end
inside a lane, and change their nodes per lane (1, 2, 4 and 8), with series,
mass records and snapshots falling between and inside launches."""
import numpy as np
import pytest

import oracle as O
from test_gpu_1d import CONFIGS, _run_hip, _setup

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import swalbe
    if swalbe.device_count() < 1:
        pytest.skip("no GPU")
    return swalbe


def same(st, ost, names=("height", "vel", "fout", "pressure", "F", "feq")):
    for name in names:
        got, want = st.get(name), getattr(ost, name)
        assert np.array_equal(got, want), (name, np.flatnonzero(got != want)[:5])


@pytest.mark.parametrize("L", [16, 65, 1021])
@pytest.mark.parametrize("name", list(CONFIGS))
def test_every_option_bitwise(S, name, L):
    cfg, n = CONFIGS[name], 57  # tdump 5: launches of five steps at most while masses are recorded
    print(f"1D wave {name} L={L}", flush=True)
    sysc, prm, st, ost, okw, hkw, args = _setup(S, L, n, cfg)
    out = O.time_loop_1d(ost, prm, n, **okw)
    body = cfg.get("body")
    dh = _run_hip(S, sysc, st, hkw, args, body)
    same(st, ost)
    if body is None and not args:
        assert np.array_equal(np.array(dh), out["dh"])


@pytest.mark.parametrize("L,n", [(3, 41), (4, 7), (7, 41), (511, 33), (20001, 36), (100003, 29),
                                 (400001, 27), (3000001, 14)])
def test_lengths_bitwise(S, L, n):
    """No mass records (tdump past the end), so launches take their full step count."""
    print(f"1D wave L={L} steps={n}", flush=True)
    for name in ("plain", "tau") if L < 200000 else ("plain",):
        sysc, prm, st, ost, okw, hkw, args = _setup(S, L, n, CONFIGS[name])
        sysc.param.tdump = 10 ** 9
        O.time_loop_1d(ost, prm, n)
        S.time_loop(sysc, st)
        same(st, ost)


@pytest.mark.parametrize("n", [0, 1, 2, 3])
def test_short_loops(S, n):
    sysc, prm, st, ost, okw, hkw, args = _setup(S, 300, n, CONFIGS["thermal"])
    O.time_loop_1d(ost, prm, n, thermal=True, seed=11)
    S.time_loop(sysc, st, thermal=True, seed=11)
    same(st, ost, ("height", "vel"))


def test_snapshots_masses_and_wetted_between_launches(S):
    L, n, dump = 300, 120, 7
    sysc, prm, st, ost, okw, hkw, args = _setup(S, L, n, CONFIGS["walls"])
    sysc.param.tdump = prm.tdump = 11
    shots, mass = np.zeros((n // dump, L)), []
    S.time_loop(sysc, st, snapshots=shots, dumping=dump, mass=mass)
    kw = dict(borders=okw["borders"], interior=okw["interior"])
    ref = _setup(S, L, n, CONFIGS["walls"])[3]
    out = O.time_loop_1d(ref, prm, n, mass=True, **kw)
    same(st, ref)
    assert np.allclose(mass, out["mass"][:len(mass)], rtol=1e-13) and len(mass) == n // 11
    for k in range(n // dump):
        O.time_loop_1d(ost, prm, dump, t0=k * dump, **kw)
        assert np.array_equal(shots[k], ost.height), k
    sysc, prm, st, ost, okw, hkw, args = _setup(S, L, n, CONFIGS["plain"])
    sysc.param.tdump = 10 ** 9
    area = []
    S.time_loop(sysc, st, S.wetted, area)
    want = O.time_loop_1d(ost, prm, n, wetted=0.055)
    assert np.array_equal(np.array(area), want["wetted"])


@pytest.mark.parametrize("name", ["plain", "walls", "tau", "thermal", "gamma_plus"])
def test_fp32_equals_one_launch_per_step(S, name):
    """No FP32 oracle: the same bits as the per-step kernel, which is held to it."""
    got = []
    for variant in (0, 1):
        sysc, prm, st, ost, okw, hkw, args = _setup(S, 5003, 45, CONFIGS[name], T=np.float32,
                                                    variant=variant)
        sysc.param.tdump = 10 ** 9
        S.time_loop(sysc, st, *args, **hkw)
        got.append([st.get(k) for k in ("height", "vel", "fout", "pressure")])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_ensemble_intermediates_equal_each_film_alone(S):
    """One launch writes the last step's intermediates of every film of an ensemble (longer and
    shorter than a workgroup, with noise, walls, ∇γ, τ ≠ 1; one film without them)."""
    specs = [(300, "thermal"), (77, "walls"), (700, "gamma_minus"), (256, "tau"), (16, "plain")]
    n, films, alone = 40, [], []
    for L, name in specs:
        for keep in (films, alone):
            sysc, prm, st, ost, okw, hkw, args = _setup(S, L, n, CONFIGS[name])
            keep.append((sysc, st, hkw))
    for sysc, st, hkw in alone:
        S.time_loop(sysc, st, **hkw)
    S.ensemble_time_loop([f[0] for f in films], [f[1] for f in films], n,
                         thermal=[f[2]["thermal"] for f in films], seed=11,
                         γ=[f[2].get("γ") for f in films],
                         grad_gamma_sign=[f[2].get("grad_gamma_sign", 0) for f in films])
    for (_, a, _), (_, b, _), spec in zip(films, alone, specs):
        for name in ("height", "vel", "fout", "pressure", "hgradp", "slip", "kbt", "F", "feq"):
            assert np.array_equal(a.get(name), b.get(name)), (spec, name)
