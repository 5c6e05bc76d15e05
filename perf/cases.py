"""The work a user of this framework has it do, as cases that can be timed.

Every case goes through the public entry points (raishinsource_amd.native and,
for reading a state into the caller's own arrays, the C entry
raishin_model_get_state) the way a program calls them: put a state into a
resident model, advance it some steps, read it back.  Grids, schemes and
parameters are those of this repository's configurations, or the same with
other sizes.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) grid, resident models, initial data, result arrays
    run(state)          one pass; returns the new state, time and last dt
    work(case)          bytes and operations one pass cannot do without
    exact(case, seed)   the result in 64 bits by plain numpy, where it has one
"""
import ctypes
import math
from dataclasses import replace

import numpy as np

from raishinsource_amd import configs, native

PI = math.pi
# stored cells times steps of the largest listed case; draw() stays below it
LARGEST = 256 * 128 * 128 * 24
TORUS_2D = ((64, 64), (128, 128), (256, 128), (512, 256))


def listed():
    return [
        # the time-step limit alone, as a driver asks for it before planning
        # its outputs (one reduction over a resident state)
        {"name": "cfl_kerr", "kind": "cfl", "ni": 192, "nj": 96, "nk": 110, "irec": 5, "spin": 0.9375},
        # a restart: primitives from the host, conserved variables on the
        # device, both read back
        {"name": "load_kerr", "kind": "load", "ni": 100, "nj": 41, "nk": 67, "irec": 5, "spin": 0.9},
        # the smallest 2D torus, graph-stepped: launches and latency
        {"name": "torus2d_64_graph", "kind": "torus", "ni": 64, "nj": 11, "nk": 64, "irec": 5, "irkt": 2, "icha": 2,
         "iwvec": 1, "cfl": 0.4, "spin": 0.9375, "mixed": False, "graph": True, "steps": 100},
        # the reference's own 2D configuration, stepped one call after another
        {"name": "torus2d_128", "kind": "torus", "ni": 128, "nj": 11, "nk": 128, "irec": 5, "irkt": 2, "icha": 2,
         "iwvec": 1, "cfl": 0.4, "spin": 0.9375, "mixed": False, "graph": False, "steps": 100},
        # a served 3D torus request
        {"name": "torus3d_64", "kind": "torus", "ni": 64, "nj": 64, "nk": 64, "irec": 5, "irkt": 3, "icha": 2,
         "iwvec": 1, "cfl": 0.5, "spin": 0.9375, "mixed": False, "graph": True, "steps": 60},
        # one GPU's subdomain at its real shape (the benchmark's), FP64
        {"name": "torus3d_256", "kind": "torus", "ni": 256, "nj": 128, "nk": 128, "irec": 5, "irkt": 3, "icha": 2,
         "iwvec": 1, "cfl": 0.5, "spin": 0.9375, "mixed": False, "graph": False, "steps": 24},
        # the same with reconstruction and face fluxes in FP32
        {"name": "torus3d_256_mixed", "kind": "torus", "ni": 256, "nj": 128, "nk": 128, "irec": 5, "irkt": 3,
         "icha": 2, "iwvec": 1, "cfl": 0.5, "spin": 0.9375, "mixed": True, "graph": False, "steps": 24},
        # the reference's 3D torus scheme set (MC, Leismann speeds, recov2,
        # RK3) on a ragged grid
        {"name": "torus3d_mc_recov2", "kind": "torus", "ni": 151, "nj": 50, "nk": 83, "irec": 1, "irkt": 3, "icha": 1,
         "iwvec": 2, "cfl": 0.3, "spin": 0.9375, "mixed": False, "graph": False, "steps": 24},
        # smooth flow in flat space with the fifth-order reconstructions
        {"name": "box_mp5", "kind": "box", "ni": 96, "nj": 72, "nk": 64, "irec": 6, "irkt": 3, "cfl": 0.5,
         "mixed": False, "steps": 24},
        {"name": "box_weno5", "kind": "box", "ni": 131, "nj": 37, "nk": 59, "irec": 7, "irkt": 3, "cfl": 0.5,
         "mixed": False, "steps": 24},
        # independent 2D tori of uneven size and precision, one batch
        {"name": "ensemble_12", "kind": "ensemble", "members": 12, "largest": 3, "mixed": True, "steps": 100},
        # Riemann tubes advanced together, as the serving loop does
        {"name": "tubes_8", "kind": "tubes", "members": 8, "zones": 1024, "steps": 96},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("cfl", "load", "torus2d", "torus2d", "torus3d", "torus3d", "torus3d", "box", "ensemble", "tubes"))
    if kind in ("cfl", "load"):
        c = {"kind": kind, "ni": _log(rng, 40, 256), "nj": _log(rng, 16, 128), "nk": _log(rng, 30, 128),
             "irec": rng.choice((1, 5, 6)), "spin": round(rng.uniform(0.0, 0.99), 4)}
        if kind == "load":  # the state crosses the host boundary three times
            c["ni"], c["nj"] = min(c["ni"], 160), min(c["nj"], 64)
        return c
    if kind == "torus2d":
        irec = rng.choice((1, 5, 5, 5))
        ni, nk = _log(rng, 64, 512), _log(rng, 64, 256)
        return {"kind": "torus", "ni": ni, "nj": 7 if irec == 1 else 11, "nk": nk, "irec": irec,
                "irkt": rng.choice((2, 3)), "icha": rng.choice((0, 1, 2)) if irec == 1 else 2,
                "iwvec": rng.choice((1, 1, 2)), "cfl": 0.3, "spin": round(rng.uniform(0.0, 0.99), 4),
                "mixed": rng.random() < 0.4, "graph": rng.random() < 0.5, "steps": 2 * rng.randint(10, 50)}
    if kind == "torus3d":
        irec = rng.choice((1, 5, 5, 5))
        ni, nj, nk = _log(rng, 48, 256), _log(rng, 24, 128), _log(rng, 40, 128)
        steps = 2 * rng.randint(4, 30)
        while ni * nj * nk * steps > LARGEST:
            steps -= 2
        return {"kind": "torus", "ni": ni, "nj": nj, "nk": nk, "irec": irec, "irkt": 3 if irec == 5 else rng.choice((2, 3)),
                "icha": rng.choice((0, 1)) if irec == 1 else 2, "iwvec": rng.choice((1, 1, 2)), "cfl": 0.3,
                "spin": round(rng.uniform(0.0, 0.99), 4), "mixed": rng.random() < 0.4, "graph": rng.random() < 0.5,
                "steps": steps}
    if kind == "box":
        return {"kind": "box", "ni": _log(rng, 30, 140), "nj": _log(rng, 20, 100), "nk": _log(rng, 20, 100),
                "irec": rng.choice((5, 6, 7)), "irkt": rng.choice((2, 3)), "cfl": 0.4, "mixed": rng.random() < 0.4,
                "steps": 2 * rng.randint(4, 15)}
    if kind == "ensemble":
        return {"kind": "ensemble", "members": rng.randint(3, 16), "largest": rng.randint(1, 3),
                "mixed": rng.random() < 0.5, "steps": 2 * rng.randint(15, 60)}
    return {"kind": "tubes", "members": rng.randint(1, 10), "zones": _log(rng, 128, 1024), "steps": 2 * rng.randint(10, 50)}


# -- configurations ---------------------------------------------------------

def _pram(c):
    """The run configuration of a case with one grid."""
    kind = c["kind"]
    if kind == "box":
        # flat space, copy boundaries in x1 and x3, periodic x2, unit cube
        return configs.Pram("box", c["ni"], c["nj"], c["nk"], irec=c["irec"], irkt=c["irkt"], cfl=c["cfl"],
                            gam=5.0 / 3.0, model=2, metric=1, ix1=1, xmin=1.0, xmax=2.0, ymin=0.0, ymax=1.0,
                            zmin=0.0, zmax=1.0, iboux1in=(5,) * 9, iboux1ot=(5,) * 9, iboux2in=(1,) * 9,
                            iboux2ot=(1,) * 9, iboux3in=(5,) * 9, iboux3ot=(5,) * 9)
    if kind in ("cfl", "load"):
        return configs.Pram(kind, c["ni"], c["nj"], c["nk"], irec=c["irec"], irkt=3, cfl=0.5, akm=c["spin"])
    return configs.Pram("torus", c["ni"], c["nj"], c["nk"], irec=c["irec"], irkt=c["irkt"], icha=c["icha"],
                        iwvec=c["iwvec"], cfl=c["cfl"], akm=c["spin"])


def _members(c, seed):
    """The tori of an ensemble: sizes in turn over the first `largest` of
    TORUS_2D, spin, field strength and inner edge from the seed."""
    rng = np.random.default_rng(1000 + seed)
    out = []
    for q in range(c["members"]):
        ni, nk = TORUS_2D[q % c["largest"]]
        p = configs.Pram("ens%d" % q, ni, 11, nk, irec=5, irkt=2, cfl=0.4, akm=float(rng.uniform(0.0, 0.99)))
        rin = float(rng.uniform(6.0, 10.0))
        out.append((p, {"rin": rin, "rmax": rin + 6.0, "beta": float(rng.choice([10.0, 100.0, 1000.0])),
                        "seed": int(seed) * 64 + q}))
    return out


# -- a smooth magnetised state on a Kerr-Schild grid, by numpy alone ---------

def _kerr_grid(p):
    """Logarithmic r, theta cells over (0, pi) and uniform phi, ghosts beyond."""
    ni, nj, nk, g = p.imax, p.jmax, p.kmax, p.nm1
    x1 = p.xmin * (p.xmax / p.xmin) ** (np.arange(ni) / (ni - 1))
    x2 = (np.arange(nj) - g + 0.5) * (2 * PI / (nj - 2 * g))
    x3 = (np.arange(nk) - g + 0.5) * (PI / (nk - 2 * g))
    grid = {"x1": x1, "x2": x2, "x3": x3}
    for q, x in (("1", x1), ("2", x2), ("3", x3)):
        d = np.empty_like(x)
        d[:-1] = x[1:] - x[:-1]
        d[-1] = d[-2]
        grid["dx%sb" % q] = d
        grid["x%sa" % q] = x + 0.5 * d
    return grid


def _smooth(shape, r, seed, flat):
    """Primitives (9, ni, nj, nk): density, u^1..u^3, pressure, unused, B^1..B^3."""
    ni, nj, nk = shape
    rng = np.random.default_rng(seed)
    i = np.arange(ni)[:, None, None] / ni
    j = np.arange(nj)[None, :, None] / nj
    k = np.arange(nk)[None, None, :] / nk
    a = 2 * PI * rng.random(6)
    w = np.zeros((9,) + tuple(shape), order="F")
    s = 1.0 if flat else 1.0 / r[:, None, None]  # angular components fall off as 1/r
    f = 1.0 if flat else r[:, None, None] ** -1.5
    w[0] = f * (1.0 + 0.3 * np.sin(2 * PI * (i + j) + a[0]) * np.cos(PI * k) + 0.02 * rng.random(shape))
    w[1] = 0.1 * np.sin(2 * PI * (i + k) + a[1])
    w[2] = s * (0.05 + 0.05 * np.cos(2 * PI * (j + i) + a[2]))
    w[3] = s * 0.05 * np.sin(2 * PI * (k - j) + a[3])
    w[4] = 0.3 * w[0] * (1.0 + 0.2 * np.cos(2 * PI * (j - k) + a[4]) + 0.02 * rng.random(shape))
    b = np.sqrt(f)
    w[6] = 0.1 * b * np.cos(2 * PI * k + a[5])
    w[7] = 0.1 * b * s * np.sin(2 * PI * i + a[0])
    w[8] = 0.1 * b * s * np.sin(2 * PI * j + a[1])
    return w


# -- prepare and run ----------------------------------------------------------

def _arrays(p):
    return [np.zeros((9, p.imax, p.jmax, p.kmax), order="F") for _ in range(2)]


def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    s = {"case": c}
    if kind in ("ensemble", "tubes"):
        s["models"], s["init"] = [], []
        rng = np.random.default_rng(2000 + seed)
        if kind == "ensemble":
            for p, init in _members(c, seed):
                p = p.resolved()
                m = native.Model.from_grid(p, native.setup_grid(p))
                m.set_precision(c["mixed"] and len(s["models"]) % 2 == 1)
                s["models"].append(m)
                s["init"].append(init)
        else:
            p = configs.tube("tube", c["zones"]).resolved()
            g = native.setup_grid(p)
            for _ in range(c["members"]):
                left, right = native.random_tube_states(rng)
                s["models"].append(native.Model.from_grid(p, g))
                s["init"].append(native.setup_tube(p, left, right))
        s["out"] = [_arrays(m.p) for m in s["models"]]
        for q, m in enumerate(s["models"]):
            _start(s, kind, m, s["init"][q])
        s["batch"] = native.Batch(s["models"])
        return s
    p = _pram(c).resolved()
    if kind in ("cfl", "load"):
        g = _kerr_grid(p)
        s["init"] = _smooth((p.imax, p.jmax, p.kmax), g["x1"], seed, False)
    else:
        g = native.setup_grid(p)
        s["init"] = (_smooth((p.imax, p.jmax, p.kmax), None, seed, True) if kind == "box"
                     else {"rin": 6.0, "rmax": 12.0, "beta": 100.0, "seed": int(seed)})
    m = s["model"] = native.Model.from_grid(p, g)
    if c.get("mixed"):
        m.set_precision(True)
    if kind == "cfl":
        m.set_state(s["init"])
    else:
        s["out"] = _arrays(p)
    return s


def _start(s, kind, m, init):
    """The initial state into the model: tori are built on the device."""
    if kind in ("torus", "ensemble"):
        m.set_torus(**init)
    else:
        m.set_state(init)


def _read(m, out):
    """The state into the caller's arrays; returns the time."""
    t = ctypes.c_double(0.0)
    native.lib().raishin_model_get_state(m.h, out[0].ctypes.data, out[1].ctypes.data, ctypes.byref(t))
    native.check()
    return t.value


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind in ("ensemble", "tubes"):
        for m, init in zip(state["models"], state["init"]):
            _start(state, kind, m, init)
        state["batch"].step_graph(c["steps"] // 2)
        times = state["batch"].times()
        for m, out in zip(state["models"], state["out"]):
            _read(m, out)
        return {"times": np.array(times), "states": state["out"]}
    m = state["model"]
    if kind == "cfl":
        return list(m.cdtcfl4())
    _start(state, kind, m, state["init"])
    if kind == "load":
        _read(m, state["out"])
        return state["out"]
    t, dt = m.step_graph(c["steps"] // 2) if c.get("graph") else m.step(c["steps"])
    _read(m, state["out"])
    return {"state": state["out"], "time": t, "dt": dt}


# -- what a pass cannot do without ------------------------------------------

def _grid_work(p, steps):
    """Steps of one model: every RK stage reads primitives and conserved
    variables (and those of the step's start from the second stage on) and
    writes both, 72 bytes each, and reads the (r, theta) metric tables once;
    about 6000 additions and multiplications per zone and stage (three
    interface fluxes with their reconstruction, sources, recovery, floors).
    Then the state is read out."""
    zi, zj, zk = p.interior
    zones = zi * zj * zk
    cells = p.imax * p.jmax * p.kmax
    b = steps * (zones * (288 + 360 * (p.irkt - 1)) + 824 * p.irkt * zi * zk) + 2 * 72 * cells
    return b, 6000 * p.irkt * zones * steps


def work(case):
    c = dict(case)
    kind = c["kind"]
    if kind in ("cfl", "load"):
        n = c["ni"] * c["nj"] * c["nk"]
        if kind == "cfl":
            return {"bytes": 72 * n + 264 * c["ni"] * c["nk"], "flops": 250 * n}
        return {"bytes": 3 * 72 * n + 264 * c["ni"] * c["nk"], "flops": 200 * n}
    if kind == "ensemble":
        parts = [_grid_work(p, c["steps"]) for p, _ in _members(c, 0)]
    elif kind == "tubes":
        parts = [_grid_work(configs.tube("tube", c["zones"]), c["steps"])] * c["members"]
    else:
        parts = [_grid_work(_pram(c), c["steps"])]
    return {"bytes": sum(x[0] for x in parts), "flops": sum(x[1] for x in parts)}


# -- 64-bit results by numpy --------------------------------------------------

def _kerr_schild(a, r, th):
    """Covariant and contravariant Kerr-Schild metric and sqrt(-g) on (r, theta);
    index order t, r, phi, theta."""
    s2, c2 = np.sin(th) ** 2, np.cos(th) ** 2
    sig = r * r + a * a * c2
    z = np.zeros_like(sig)
    h = 2 * r / sig
    g = [[h - 1, h, -a * h * s2, z], [h, 1 + h, -a * s2 * (1 + h), z],
         [-a * h * s2, -a * s2 * (1 + h), s2 * (sig + a * a * s2 * (1 + h)), z], [z, z, z, sig + z]]
    gi = [[-1 - h, h, z, z], [h, (r * r - 2 * r + a * a) / sig, a / sig, z], [z, a / sig, 1 / (sig * s2), z],
          [z, z, z, 1 / sig]]
    return g, gi, sig * np.abs(np.sin(th))


def _state_vectors(w, p, g, gi):
    """Enthalpy, Lorentz factor, u^mu, u_mu, b^mu, b_mu, b^2."""
    rho, pr = w[0], w[4]
    al = 1 / np.sqrt(-gi[0][0])
    usq = sum(g[m][n] * w[m] * w[n] for m in range(1, 4) for n in range(1, 4))
    gf = np.sqrt(1 + usq)
    uc = [gf / al] + [w[m] - gf * al * gi[0][m] for m in range(1, 4)]
    ud = [sum(g[m][n] * uc[n] for n in range(4)) for m in range(4)]
    B = [None, w[6], w[7], w[8]]
    b0 = sum(B[m] * ud[m] for m in range(1, 4))
    b = [b0] + [(B[m] + b0 * uc[m]) / uc[0] for m in range(1, 4)]
    bd = [sum(g[m][n] * b[n] for n in range(4)) for m in range(4)]
    return rho + p.gam / (p.gam - 1) * pr, gf, uc, ud, b, bd, sum(b[m] * bd[m] for m in range(4)), al


def exact(case, seed):
    # A stepped state is 64-bit arithmetic throughout already, and its
    # restatement in numpy takes minutes at these sizes.
    c = dict(case)
    if c["kind"] not in ("cfl", "load"):
        return None
    p = _pram(c).resolved()
    grid = _kerr_grid(p)
    g, gi, detg = _kerr_schild(p.akm, grid["x1"][:, None, None], grid["x3"][None, None, :])
    w = _smooth((p.imax, p.jmax, p.kmax), grid["x1"], seed, False)
    h, gf, uc, ud, b, bd, bsq, al = _state_vectors(w, p, g, gi)
    if c["kind"] == "load":
        u = np.zeros_like(w)
        u[0] = w[0] * uc[0]
        for q in range(1, 4):
            u[q] = (h + bsq) * uc[0] * ud[q] - b[0] * bd[q]
        u[4] = (h + bsq) * uc[0] * ud[0] + w[4] + 0.5 * bsq - b[0] * bd[0] + w[0] * uc[0]
        u[5] = w[0] * (w[4] / w[0] ** p.gam) * uc[0]
        u[6:9] = w[6:9]
        return [w, u * detg]
    # fast speeds of the three directions at the cell centres (Del Zanna et
    # al. 2007) and the smallest crossing time of the cells off the outer layer
    v = [None] + [w[m] / gf for m in range(1, 4)]
    vsq = sum(g[m][n] * v[m] * v[n] for m in range(1, 4) for n in range(1, 4))
    va = bsq / (h + bsq)
    om = va + p.gam * w[4] / h * (1 - va)
    out = []
    for q in range(1, 4):
        gqq = gi[q][q] + (al * gi[0][q]) ** 2
        root = np.sqrt(om * (1 - vsq) * ((1 - vsq * om) * gqq - (1 - om) * v[q] ** 2))
        speed = np.zeros(w.shape[1:])
        for sign in (1, -1):
            lam = al * (v[q] * (1 - om) + sign * root) / (1 - vsq * om) - al * al * gi[0][q]
            speed = np.maximum(speed, np.minimum(np.abs(lam), 1.0))
        dx = grid["dx%db" % q].reshape([-1 if ax == q - 1 else 1 for ax in range(3)])
        dt = np.abs(dx / (speed + 1e-12))[1:-1, 1:-1, 1:-1]
        out.append(min(1.0, float(dt.min())) if w.shape[q] > 3 * p.nm1 - 1 else 1.0)
    return [min(out)] + out
