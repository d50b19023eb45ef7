"""Timed cases of the thin-film solver, called as a user's program calls it.

Five kinds of work, each through the package's public entry points:

* "film":  one 2D film through `time_loop` (FP64 or FP32; noise, contact-angle
  field, gravity, body force, tau != 1, per-step series, final outputs only).
  flow "go on" is one output interval of a running simulation (advance by
  `steps`, read the fields back); flow "solve" is a whole `run_*` driver: the
  initial film goes up, the loop runs, the film comes back.
* "watch": one 2D film with the user's own callback on every step.
* "line":  one 1D film through the 1D `time_loop` (a solve with snapshots under
  a surface-tension gradient, or an interval of a long film).
* "scan":  many 1D films of one length in one `ensemble_time_loop`.
* "sweep": many FP32 2D films of different sizes in one `Batch`.

A case's outputs are what its driver hands back (the height; also the
velocities for a driven film, the populations where tau != 1 carries them on;
the series that were asked for).
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "swalbe.jl_amd"))

import swalbe as S  # noqa: E402

PRECURSOR = 0.05  # hmin - hcrit: the thickness at which the disjoining pressure vanishes


def _film(name, Lx, Ly, dtype, steps, shape, flow="go on", noise=False, theta=False, tau=1.0,
          g=0.0, body=False, series="", final=False):
    c = {"kind": "film", "Lx": Lx, "Ly": Ly, "dtype": dtype, "steps": steps, "shape": shape,
         "flow": flow, "noise": noise, "theta": theta, "tau": tau, "g": g, "body": body,
         "series": series, "final": final}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a droplet relaxing on the default lattice (256 x 256, Float64) with its wetted area of
        # every step, as run_dropletrelax records it: the call most first scripts make
        _film("relax_256_f64", 256, 256, "f64", 500, "drop", series="wetted"),
        # the hanging film of the Rayleigh-Taylor driver: small, whole solve, extremes every step
        _film("hanging_100_f64", 100, 100, "f64", 1000, "rough", flow="solve", g=-0.001,
              series="dh"),
        # a droplet on a patterned substrate: a contact-angle field goes up with the film
        _film("patterned_1024_f64", 1024, 1024, "f64", 300, "drop", flow="solve", theta=True),
        # the headline: rupture with thermal noise, 4096 x 4096, FP32, every step's outputs
        _film("rupture_4096_f32", 4096, 4096, "f32", 500, "rough", noise=True),
        # the same physics in FP64 on a ragged film (odd rows: no pair of rows shares a draw)
        _film("rupture_2501_f64", 2500, 2501, "f64", 200, "rough", noise=True),
        # a long deterministic FP32 run that only wants its last state
        _film("longrun_2000x1500_f32", 2000, 1500, "f32", 1000, "rough", final=True),
        # a driven film under gravity with tau != 1: the populations are carried from step to step
        _film("driven_1000x1031_f32", 1000, 1031, "f32", 400, "rough", tau=0.8, g=0.001,
              body=True),
        # the user's own measurement on every step: the op-by-op loop
        {"name": "watch_512_f64", "kind": "watch", "Lx": 512, "Ly": 512, "dtype": "f64",
         "steps": 50},
        # coalescence of two droplets on a line under a surface-tension gradient, with snapshots
        {"name": "gamma_line_1024_f64", "kind": "line", "L": 1024, "dtype": "f64", "steps": 5000,
         "shape": "drops", "dump": 500},
        # a long undulated line, one output interval
        {"name": "long_line_3m_f64", "kind": "line", "L": 3_000_001, "dtype": "f64",
         "steps": 1000, "shape": "rough", "dump": 0},
        # a parameter scan: surface tension and contact angle over 512 lines at once
        {"name": "scan_512x1024_f64", "kind": "scan", "films": 512, "L": 1024, "dtype": "f64",
         "steps": 1000},
        # a sweep of droplet pairs on films of different sizes, heights back at the end
        {"name": "sweep_32_f32", "kind": "sweep", "films": 32, "lo": 128, "hi": 768,
         "steps": 200},
    ]


def draw(rng):
    def size(lo, hi, odd=0.4):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        if rng.random() < odd:
            return n | 1
        return max(lo, n // 8 * 8)

    def sides(lo, hi):
        a = size(lo, hi)
        b = min(hi, max(lo, int(a * math.exp(rng.uniform(-0.5, 0.5)))))
        return a, b

    kind = rng.choice(["small", "small", "middle", "large64", "large32", "large32", "carried",
                       "watch", "line", "long", "scan", "sweep"])
    if kind == "small":
        Lx, Ly = sides(48, 400)
        dtype = rng.choice(["f64", "f64", "f32"])
        return _film("", Lx, Ly, dtype, rng.randrange(300, 900), rng.choice(["drop", "rough"]),
                     flow=rng.choice(["go on", "solve"]), theta=rng.random() < 0.3,
                     series=rng.choice(["", "wetted", "dh"] if dtype == "f64" else ["", "dh"]))
    if kind == "middle":
        Lx, Ly = sides(500, 1400)
        return _film("", Lx, Ly, rng.choice(["f64", "f32"]), rng.randrange(150, 350),
                     rng.choice(["drop", "rough"]), flow=rng.choice(["go on", "solve"]),
                     theta=rng.random() < 0.4, final=rng.random() < 0.3)
    if kind == "large64":
        Lx, Ly = sides(1500, 2600)
        return _film("", Lx, Ly, "f64", rng.randrange(100, 200), "rough",
                     noise=rng.random() < 0.7, final=rng.random() < 0.3)
    if kind == "large32":
        Lx, Ly = sides(1500, 4000)
        return _film("", Lx, Ly, "f32", rng.randrange(200, 500), "rough",
                     noise=rng.random() < 0.6, final=rng.random() < 0.5)
    if kind == "carried":
        Lx, Ly = sides(200, 1400)
        return _film("", Lx, Ly, rng.choice(["f64", "f32"]), rng.randrange(150, 400), "rough",
                     tau=round(rng.uniform(0.7, 1.3), 3), g=0.001, body=rng.random() < 0.5)
    if kind == "watch":
        Lx, Ly = sides(64, 800)
        return {"kind": "watch", "Lx": Lx, "Ly": Ly, "dtype": rng.choice(["f64", "f32"]),
                "steps": rng.randrange(30, 80)}
    if kind == "line":
        return {"kind": "line", "L": size(200, 3000), "dtype": "f64",
                "steps": rng.randrange(1500, 5000), "shape": "drops", "dump": 500}
    if kind == "long":
        return {"kind": "line", "L": size(20_000, 4_000_000),
                "dtype": rng.choice(["f64", "f64", "f32"]), "steps": rng.randrange(300, 1000),
                "shape": "rough", "dump": 0}
    if kind == "scan":
        return {"kind": "scan", "films": size(32, 768), "L": size(256, 1500), "dtype": "f64",
                "steps": rng.randrange(400, 1000)}
    return {"kind": "sweep", "films": rng.randrange(12, 40), "lo": 128,
            "hi": rng.choice([384, 512, 768]), "steps": rng.randrange(120, 240)}


# ---------------------------------------------------------------- inputs


def _np(dtype):
    return np.float64 if dtype == "f64" else np.float32


def _normal(seed, *shape):
    """Standard normals of a seed as a host array, drawn on the GPU (quick at every size)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    return torch.randn(*shape, generator=gen, dtype=torch.float64, device=dev).cpu().numpy()


def _cap(r, R, theta):
    """Height of a spherical cap (a circle in 1D) at distance r from its axis."""
    s = np.minimum(r / R, 1.0)
    return np.where(r <= R, (np.sqrt(1.0 - s * s) - math.cos(math.pi * theta)) * R, 0.0)


def _film_inputs(c, seed):
    rng = np.random.default_rng(seed)
    Lx, Ly = c["Lx"], c["Ly"]
    if c.get("shape", "rough") == "drop":
        # the scheme stays finite for caps with gamma H up to about 0.4
        R = min(rng.uniform(0.2, 0.28) * min(Lx, Ly), 0.35 / (0.01 * (1 - math.cos(math.pi / 6))))
        cx, cy = rng.uniform(0.4, 0.6) * Lx, rng.uniform(0.4, 0.6) * Ly
        i, j = np.arange(1, Lx + 1)[:, None], np.arange(1, Ly + 1)[None, :]
        h = np.maximum(_cap(np.sqrt((i - cx) ** 2 + (j - cy) ** 2), R, 1 / 6), PRECURSOR)
    else:
        h = 1.0 + 0.001 * _normal(seed, Ly, Lx).T
    theta = None
    if c.get("theta"):  # stripes of two contact angles
        w = max(4, Lx // int(rng.integers(6, 12)))
        theta = np.where((np.arange(Lx)[:, None] // w) % 2 == 0, 1 / 9, 1 / 6) + np.zeros((1, Ly))
        theta = np.asfortranarray(theta)
    return {"h": np.asfortranarray(h), "theta": theta,
            "body": [2e-5, -1e-5] if c.get("body") else None, "noise_seed": int(seed) % 100003}


def _taumucs(c, steps=None):
    return S.Taumucs(Tmax=c["steps"] if steps is None else steps, tau=c.get("tau", 1.0),
                     g=c.get("g", 0.0), gamma=0.0005 if c.get("g", 0.0) < 0 else 0.01,
                     kbt=1e-6 if c.get("noise") else 0.0, theta=1 / 9)


def _line_inputs(c, seed):
    rng = np.random.default_rng(seed)
    L = c["L"]
    i = np.arange(1, L + 1, dtype=float)
    if c["shape"] == "drops":
        R = rng.uniform(0.4, 0.48) * L
        b = R * math.sin(math.pi / 9)
        h = sum(np.maximum(_cap(np.abs(i - x), R, 1 / 9), PRECURSOR) for x in (L / 2 - b, L / 2 + b))
        gam = 1e-4 * (1.0 + 0.1 * np.tanh((i - L / 2) / rng.uniform(5.0, 60.0)))
        return {"h": h - PRECURSOR, "gamma": gam}
    k = int(rng.integers(3, 9))
    return {"h": 1.0 + 0.01 * np.sin(2 * math.pi * k * i / L) + 0.001 * _normal(seed, L),
            "gamma": None}


def _scan_inputs(c, seed):
    rng = np.random.default_rng(seed)
    n, L = c["films"], c["L"]
    i = np.arange(1, L + 1, dtype=float)
    gam, th = rng.uniform(5e-5, 2e-4, n), rng.uniform(1 / 12, 1 / 7, n)
    R = 0.45 * L
    b = R * math.sin(math.pi / 9)
    h = sum(np.maximum(_cap(np.abs(i - x), R, 1 / 9), PRECURSOR) for x in (L / 2 - b, L / 2 + b))
    h = (h - PRECURSOR)[None, :] * (1.0 + 0.01 * rng.uniform(-1, 1, (n, 1)))
    return {"h": h, "gamma": gam, "theta": th}


def _sweep_inputs(c, seed):
    """Two tangent caps per film: (Lx, Ly, gamma, theta, R) of each."""
    rng = np.random.default_rng(seed)
    wide = np.random.default_rng(c["films"] * 1000 + c["hi"])  # the sizes are the case's own
    films = []
    for _ in range(c["films"]):
        Lx = int(wide.integers(c["lo"], c["hi"] + 1))
        Ly = int(Lx * wide.uniform(0.4, 0.8))
        gam, th = rng.uniform(0.005, 0.02), rng.uniform(1 / 18, 1 / 6)
        R = min(rng.uniform(0.15, 0.3) * Ly, 0.4 / (gam * (1 - math.cos(math.pi * th))))
        films.append((Lx, Ly, gam, th, R))
    return films


def _caps_centres(Lx, Ly, R, theta):
    b = R * math.sin(math.pi * theta)
    return (Lx / 2 + 0.5 - b, Ly / 2 + 0.5), (Lx / 2 + 0.5 + b, Ly / 2 + 0.5)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("film", "watch"):
        x = _film_inputs(c, seed)
        sysc = S.SysConst(c["Lx"], c["Ly"], _taumucs(c))
        state = S.Sys(sysc, "GPU", T=_np(c["dtype"]), kind="thermal" if c.get("noise") else "simple")
        # the rest film that FP32 states store their deviations from (no effect in FP64)
        state.set_reference_height(PRECURSOR if c.get("shape") == "drop" else 1.0, c.get("g", 0.0))
        state.height = x["h"]
        S.equilibrium(state, sysc)
        if c.get("tau", 1.0) != 1.0:
            state.copy("ftemp", "feq")
        return {"case": c, "in": x, "sys": sysc, "state": state}
    if kind == "line":
        x = _line_inputs(c, seed)
        sysc = S.SysConst_1D(c["L"], S.Taumucs(Tmax=c["steps"], gamma=1e-4 if c["dump"] else 0.01))
        state = S.Sys(sysc, T=_np(c["dtype"]), kind="gamma" if c["dump"] else "simple")
        state.height = x["h"]
        S.equilibrium(state, sysc)
        if c["dump"]:
            state.set("gamma", x["gamma"])
            S.grad_gamma(state)
        return {"case": c, "in": x, "sys": sysc, "state": state}
    if kind == "scan":
        x = _scan_inputs(c, seed)
        systems, states = [], []
        for k in range(c["films"]):
            sysc = S.SysConst_1D(c["L"], S.Taumucs(Tmax=c["steps"], gamma=x["gamma"][k],
                                                   theta=x["theta"][k]))
            st = S.Sys(sysc, T=_np(c["dtype"]))
            st.height = x["h"][k]
            systems.append(sysc)
            states.append(st)
        return {"case": c, "systems": systems, "states": states}
    films = []
    need = 0
    for Lx, Ly, gam, th, R in _sweep_inputs(c, seed):
        c1, c2 = _caps_centres(Lx, Ly, R, th)
        init = S.film_init(S.INIT_TWO_CAPS, precursor=0.1, href=0.1, cap1=(R, th) + c1,
                           cap2=(R, th) + c2, clamp=True)
        films.append((S.Taumucs(Tmax=c["steps"], gamma=gam, theta=th), Lx, Ly, init))
        need += S.film_bytes(Lx, Ly)
    return {"case": c, "films": films, "batch": S.Batch(need + (1 << 20), len(films))}


# ---------------------------------------------------------------- one pass


def run(state):
    c = state["case"]
    return {"film": _run_film, "watch": _run_watch, "line": _run_line, "scan": _run_scan,
            "sweep": _run_sweep}[c["kind"]](c, state)


def _run_film(c, s):
    sysc, st, x = s["sys"], s["state"], s["in"]
    if c["flow"] == "solve":
        st.height = x["h"]
        st.velx = 0.0
        st.vely = 0.0
        S.equilibrium(st, sysc)
    out = {}
    args = ()
    if c["series"] == "wetted":
        out["wetted"] = []
        args = (S.wetted, out["wetted"])
    elif c["series"] == "dh":
        out["dh"] = []
        args = (out["dh"],)
    elif c["theta"]:
        args = (x["theta"],)
    elif c["body"]:
        args = (S.inclination, x["body"])
    S.time_loop(sysc, st, *args, thermal=c["noise"], seed=x["noise_seed"],
                final_outputs_only=c["final"])
    out = {k: np.asarray(v, dtype=st.T if k == "dh" else None) for k, v in out.items()}
    out["height"] = st.get("height")
    if c["body"]:
        out["velx"], out["vely"] = st.get("velx"), st.get("vely")
    if c["tau"] != 1.0:
        out["fout"] = st.get("fout")
    return out


def _highest(measure, st):
    measure.append(st.reduce("height", 0.055)["max"])


def _run_watch(c, s):
    seen = []
    S.time_loop(s["sys"], s["state"], _highest, seen)
    return {"seen": np.asarray(seen, dtype=_np(c["dtype"])), "height": s["state"].get("height"),
            "velx": s["state"].get("velx")}


def _run_line(c, s):
    sysc, st, x = s["sys"], s["state"], s["in"]
    if not c["dump"]:
        S.time_loop(sysc, st)
        return {"height": st.get("height")}
    st.height = x["h"]
    st.vel = 0.0
    st.t = 0
    S.equilibrium(st, sysc)
    shots = np.zeros((c["steps"] // c["dump"], c["L"]))
    S.time_loop(sysc, st, γ=x["gamma"], grad_gamma_sign=-1, snapshots=shots, dumping=c["dump"])
    return {"snapshots": shots, "height": st.get("height")}


def _run_scan(c, s):
    S.ensemble_time_loop(s["systems"], s["states"], nsteps=c["steps"])
    return {"height": np.stack([st.get("height") for st in s["states"]])}


def _run_sweep(c, s):
    b = s["batch"]
    slots = [b.add(prm, Lx, Ly, init, c["steps"]) for prm, Lx, Ly, init in s["films"]]
    b.step(c["steps"])
    out = {"film %02d" % k: b.get(slot, "height", dtype=np.float32) for k, slot in enumerate(slots)}
    for slot in slots:
        b.remove(slot)
    return out


# ---------------------------------------------------------------- what a pass cannot do without


# operations per node and step, counted in the model's formulas: film pressure 25, h grad p 27,
# slip 14, force sum 4, equilibrium 72, force term 20, streaming and moments 20; noise: half a
# 10-round counter draw and one pair of normals; 1D: pressure 22, force 16, equilibrium 13,
# collision and moments 8
_OPS_2D, _OPS_NOISE, _OPS_1D = 182, 110, 59


def work(case):
    c, kind = case, case["kind"]
    if kind == "sweep":
        nodes = sum(f[0] * f[1] for f in _sweep_inputs(c, 0))
        # initial heights are made on the GPU; h, ux, uy, p and nine populations written once
        return {"bytes": 4.0 * nodes * 14, "flops": float(_OPS_2D * nodes * c["steps"])}
    e = 8.0 if c["dtype"] == "f64" else 4.0
    if kind in ("line", "scan"):
        n = c["L"] * c.get("films", 1)
        shots = (c["steps"] // c["dump"]) * c["L"] * 8.0 if c.get("dump") else 0.0
        # h, u in; h, u, p and three populations out; the height back to the host
        return {"bytes": e * n * 9 + shots, "flops": float(_OPS_1D * n * c["steps"])}
    n = c["Lx"] * c["Ly"]
    ops = _OPS_2D + (_OPS_NOISE if c.get("noise") else 0)
    if kind == "watch":
        # the callback may look at every field of every step: p, h grad p, slip, F, feq, |u|^2, f
        # and the moments are written each step, the moments and F read
        return {"bytes": e * n * (2 + c["steps"] * (3 + 2 + 28)), "flops": float(ops * n * c["steps"])}
    planes = 3 + 13 + 1 + (2 if c["body"] else 0) + (18 if c["tau"] != 1.0 else 0)
    planes += (1 if c["flow"] == "solve" else 0) + (1 if c["theta"] else 0)
    return {"bytes": e * n * planes, "flops": float(ops * n * c["steps"])}


# ---------------------------------------------------------------- the same in plain 64-bit torch


_C = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)]


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_dev(), torch.float64)


def _sh(a, x, y):
    """a at (i - x, j - y), periodic."""
    return torch.roll(a, (x, y), (0, 1))


def _kappa(theta, n, m, hmin):
    return (1.0 - np.cos(np.pi * np.asarray(theta, dtype=float))) * (n - 1) * (m - 1) / ((n - m) * hmin)


def _normals_2d(Lx, Ly, seed, step):
    """The counter-based pair of normals of every node: Philox 4x32-10 on the counter
    {x + Lx (y // 2), 0, step}, words 0-1 for even rows, 2-3 for odd ones, Box-Muller."""
    dev, M = _dev(), 0xFFFFFFFF
    x = torch.arange(Lx, device=dev, dtype=torch.int64)[:, None]
    q = torch.arange((Ly + 1) // 2, device=dev, dtype=torch.int64)[None, :]
    c = [(x + Lx * q) & M, torch.zeros((), dtype=torch.int64, device=dev),
         torch.full((), step & M, dtype=torch.int64, device=dev),
         torch.full((), step >> 32, dtype=torch.int64, device=dev)]
    k0, k1 = seed & M, seed >> 32

    def mul(a, b):  # 32 x 32 bits: high and low words
        lo = a * (b & 0xFFFF)
        hi = a * (b >> 16) + (lo >> 16)
        return hi >> 16, ((hi & 0xFFFF) << 16) | (lo & 0xFFFF)

    for r in range(10):
        h0, l0 = mul(c[0], 0xD2511F53)
        h1, l1 = mul(c[2], 0xCD9E8D57)
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
    z = torch.empty(2, Lx, Ly, device=dev, dtype=torch.float64)
    for b in range(2):
        u1, u2 = ((w.double() + 0.5) * 2.0 ** -32 for w in c[2 * b:2 * b + 2])
        rad = torch.sqrt(-2.0 * torch.log(u1)).expand(Lx, -1)
        n = (Ly + 1 - b) // 2
        z[0, :, b::2] = (rad * torch.cos(2 * math.pi * u2))[:, :n]
        z[1, :, b::2] = (rad * torch.sin(2 * math.pi * u2))[:, :n]
    return z


def _steps_2d(h, steps, gamma, theta, tau=1.0, g=0.0, kbt=0.0, seed=0, body=None, dh=None, top=None):
    """`steps` steps of the D2Q9 model from rest in 64 bits: h, ux, uy, f."""
    n, m, hmin, hcrit, delta, mu = 9, 3, 0.1, 0.05, 1.0, (1 / 3) * (tau - 0.5)
    Lx, Ly = h.shape
    ux, uy = torch.zeros_like(h), torch.zeros_like(h)
    kap = torch.as_tensor(_kappa(theta, n, m, hmin), dtype=torch.float64, device=h.device)

    def feq(k, h, ux, uy, usq):
        if k == 0:
            return h * (1.0 - (5 / 6) * g * h - (2 / 3) * usq)
        a = _C[k][0] * ux + _C[k][1] * uy
        return (1 / 9 if k < 5 else 1 / 36) * h * (1.5 * g * h + (3.0 + 4.5 * a) * a - 1.5 * usq)

    usq = ux * ux + uy * uy
    ft = [feq(k, h, ux, uy, usq) for k in range(9)] if tau != 1.0 else None
    for it in range(steps):
        if dh is not None:
            dh.append(h.max() - h.min())
        axis = _sh(h, 1, 0) + _sh(h, -1, 0) + _sh(h, 0, 1) + _sh(h, 0, -1)
        diag = _sh(h, 1, 1) + _sh(h, -1, 1) + _sh(h, 1, -1) + _sh(h, -1, -1)
        lap = (2 / 3) * axis + (1 / 6) * diag - (10 / 3) * h
        a = hmin / (h + hcrit)
        a3 = a * a * a
        p = -gamma * (kap * (a3 * a3 * a3 - a3)) - gamma * lap
        xm, xp = _sh(p, 1, 0), _sh(p, -1, 0)
        ym, yp = _sh(p, 0, 1), _sh(p, 0, -1)
        mm, pm, pp, mp = _sh(p, 1, 1), _sh(p, -1, 1), _sh(p, -1, -1), _sh(p, 1, -1)
        gx = (xp - xm) / 3 + (pm - mm + pp - mp) / 12
        gy = (yp - ym) / 3 + (mp - mm + pp - pm) / 12
        den = 2 * h * h + 6 * delta * h + 3 * delta * delta
        Fx, Fy = -h * gx - 6 * mu * h * ux / den, -h * gy - 6 * mu * h * uy / den
        if kbt:
            amp = torch.sqrt(2 * kbt * mu * 6 * h / den)
            z = _normals_2d(Lx, Ly, seed, it + 1)
            Fx, Fy = Fx - z[0] * amp, Fy - z[1] * amp
        if body is not None:
            Fx, Fy = Fx + h * body[0], Fy + h * body[1]
        if top is not None:
            top.append(h.max())
        usq = ux * ux + uy * uy
        f = []
        for k in range(9):
            fo = feq(k, h, ux, uy, usq) / tau
            if ft is not None:
                fo = fo + (1 - 1 / tau) * ft[k]
            if k:
                fo = fo + (1 / 3 if k < 5 else 1 / 24) * (_C[k][0] * Fx + _C[k][1] * Fy)
            f.append(_sh(fo, *_C[k]) if k else fo)
        h = sum(f[1:], f[0])
        ux = sum(_C[k][0] * f[k] for k in range(9) if _C[k][0]) / h
        uy = sum(_C[k][1] * f[k] for k in range(9) if _C[k][1]) / h
        if ft is not None:
            ft = f
    return h, ux, uy, f


def _steps_1d(h, steps, gamma, theta, grad_gamma=None, dump=0, shots=None):
    """`steps` steps of the D1Q3 model from rest in 64 bits along the last axis."""
    n, m, hmin, hcrit, delta, mu = 9, 3, 0.1, 0.05, 1.0, 1 / 6
    u = torch.zeros_like(h)
    kap = torch.as_tensor(_kappa(theta, n, m, hmin), dtype=torch.float64, device=h.device)
    if kap.ndim == 1:
        kap = kap[:, None]
    for it in range(1, steps + 1):
        a = hmin / (h + hcrit)
        a3 = a * a * a
        p = -gamma * (kap * (a3 * a3 * a3 - a3))
        p = p - gamma * (torch.roll(h, 1, -1) - 2 * h + torch.roll(h, -1, -1))
        F = -h * 0.5 * (torch.roll(p, -1, -1) - torch.roll(p, 1, -1))
        F = F - 6 * mu * h * u / (2 * h * h + 6 * delta * h + 3 * delta * delta)
        if grad_gamma is not None:
            F = F - grad_gamma
        uu = u * u
        f0 = h * (1.0 - uu)
        f1 = torch.roll(h * (0.5 * u + 0.5 * uu) + 0.5 * F, 1, -1)
        f2 = torch.roll(h * (0.5 * uu - 0.5 * u) - 0.5 * F, -1, -1)
        h = f0 + f1 + f2
        u = (f1 - f2) / h
        if dump and it % dump == 0:
            shots.append(h)
    return h


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "film":
        x, p = _film_inputs(c, seed), _taumucs(c)
        dh = [] if c["series"] == "dh" else None
        theta = x["theta"] if c["theta"] and not c["series"] else p.θ
        h, ux, uy, f = _steps_2d(_t(x["h"]), c["steps"], p.γ, theta, p.τ, p.g, p.kbt,
                                 x["noise_seed"], x["body"], dh=dh)
        out = {"height": h}
        if dh is not None:
            out["dh"] = torch.stack(dh)
        if c["series"] == "wetted":
            out["wetted"] = None
        if c["body"]:
            out["velx"], out["vely"] = ux, uy
        if c["tau"] != 1.0:
            out["fout"] = torch.stack(f, dim=-1)
        return out
    if kind == "watch":
        x, p, top = _film_inputs(c, seed), _taumucs(c), []
        h, ux, _, _ = _steps_2d(_t(x["h"]), c["steps"], p.γ, p.θ, top=top)
        return {"seen": torch.stack(top), "height": h, "velx": ux}
    if kind == "line":
        x, shots = _line_inputs(c, seed), []
        if not c["dump"]:
            return {"height": _steps_1d(_t(x["h"]), c["steps"], 0.01, 1 / 9)}
        gam = _t(x["gamma"])
        gg = -0.75 * (torch.roll(gam, 1) - torch.roll(gam, -1))
        h = _steps_1d(_t(x["h"]), c["steps"], gam, 1 / 9, gg, c["dump"], shots)
        return {"snapshots": torch.stack(shots), "height": h}
    if kind == "scan":
        x = _scan_inputs(c, seed)
        return {"height": _steps_1d(_t(x["h"]), c["steps"], _t(x["gamma"])[:, None], x["theta"])}
    out = {}
    for k, (Lx, Ly, gam, th, R) in enumerate(_sweep_inputs(c, seed)):
        i, j = np.arange(1, Lx + 1)[:, None], np.arange(1, Ly + 1)[None, :]
        caps = [np.where(d <= R, _cap(d, R, th), 0.1) for d in
                (np.sqrt((i - a) ** 2 + (j - b) ** 2) for a, b in _caps_centres(Lx, Ly, R, th))]
        caps = [np.where(q < 0, 0.1, q) for q in caps]
        h = np.maximum(caps[0] + caps[1] - 0.1, 0.1)
        out["film %02d" % k] = _steps_2d(_t(h), c["steps"], gam, th)[0]
    return out
