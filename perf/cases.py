"""What a program that uses gpuvh has it do, as cases to be timed and compared.

Kinds of case, each through the public entry points of gpuvh:

  steps      a context that evolves: a stretch of KT steps, then the ten hydro
             fields of a snapshot (e, u^i, the five spatial pi, Pi)
  loop       one freeze-out window of the run loop: per step the history
             record, the termination count and the KT step, then the window's
             surface search and its rows
  find       the surface search of a recorded window alone
  setup      the initial state of an event with flow, shear and bulk from
             primitive fields, and the T^{tau mu} that it gives
  batch      a whole call of the batched engine: submit, run to the end, rows
             and final energy densities of every event
  cornelius  surface elements of independent cells on device buffers
  validity   the Knudsen and inverse Reynolds fields of a state

An evolving context goes on from where its last pass left it, as the run loop
does, and starts its event again once it is over.  The mixed precision forms
carry pi, Pi and all fluxes in FP32, and a program that picks them keeps what
it reads in FP32: their outputs are returned so.
"""
import ctypes
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gpu-vh_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

HBARC = 0.197326938
FOFREQ = 10
EOS = {"conformal": 0, "wb": 1, "table": 2}
PRECISION = {"fp64": 0, "mixed": 1, "mixed_f64_roots": 2}
# fields of a snapshot in the order of the history ring, as gpuvh numbers them
SNAPSHOT = {"ux": 18, "uy": 19, "un": 20, "e": 15, "pixx": 8, "pixy": 9, "pixn": 10, "piyy": 11,
            "piyn": 12, "Pi": 14}
VALIDITY = ["kn_taupi", "kn_taubulk", "re_pi", "re2_pi", "re_bulk", "re2_bulk", "taupi", "dxux",
            "dyuy", "theta", "regulations"]
# most cell-steps (a 3+1D one counts twice) and cells of cornelius whose exact
# values take numpy less than about 20 seconds
EXACT_CELL_STEPS = 700_000
EXACT_CELLS_4D = 2_000
EXACT_CELLS_3D = 12_000


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest event in use, 2+1D and conformal: launches and latency
        dict(name="steps_2d_conformal", kind="steps", nx=61, ny=61, nz=1, h=0.1, dt=0.002,
             steps=20, eos="conformal", bulk=False, precision="fp64", t_reg=0.0),
        # an ordinary 2+1D event with everything switched on, in the fast form
        dict(name="steps_2d_table_mixed", kind="steps", nx=261, ny=261, nz=1, h=0.1, dt=0.002,
             steps=10, eos="table", bulk=True, precision="mixed", t_reg=0.05),
        # an ordinary 3+1D event
        dict(name="steps_3d_table", kind="steps", nx=101, ny=101, nz=51, h=0.15, dt=0.002,
             steps=20, eos="table", bulk=True, precision="fp64", t_reg=0.05),
        # the library's default equation of state and bulk setting, odd sizes
        dict(name="steps_3d_wb", kind="steps", nx=87, ny=93, nz=25, h=0.15, dt=0.002, steps=20,
             eos="wb", bulk=True, precision="fp64", t_reg=0.0),
        # the mixed form with FP64 root-finds, shear only
        dict(name="steps_3d_f64_roots", kind="steps", nx=121, ny=117, nz=31, h=0.15, dt=0.002,
             steps=20, eos="table", bulk=False, precision="mixed_f64_roots", t_reg=0.0),
        # the headline lattice in the run loop, in both forms: the largest work
        dict(name="loop_3d_large", kind="loop", nx=201, ny=201, nz=101, h=0.1, dt=0.01,
             eos="table", bulk=True, precision="fp64", t_reg=0.0),
        dict(name="loop_3d_large_mixed", kind="loop", nx=201, ny=201, nz=101, h=0.1, dt=0.01,
             eos="table", bulk=True, precision="mixed", t_reg=0.0),
        # the search of a 3+1D window by itself
        dict(name="find_3d", kind="find", nx=121, ny=121, nz=61, h=0.15, dt=0.01, eos="table",
             bulk=True, precision="fp64", t_reg=0.0),
        # a 3+1D event that starts with flow, shear and bulk from a pre-equilibrium stage
        dict(name="setup_3d", kind="setup", nx=101, ny=101, nz=51, h=0.15, dt=0.01, eos="table",
             bulk=True, precision="fp64", t_reg=0.0),
        # serving: many small events of several sizes together, surfaces on
        dict(name="batch_2d", kind="batch", events=12, nx=101, ny=101, nz=1, spread=20, h=0.2,
             dt=0.02, nt=60, eos="table", bulk=True, precision="fp64", t_reg=0.0),
        # elements of as many hypercubes as one call takes
        dict(name="cornelius_4d", kind="cornelius", dim=4, cells=16384),
        # the diagnostics of a 3+1D state
        dict(name="validity_3d", kind="validity", nx=151, ny=151, nz=41, h=0.15, dt=0.01,
             eos="table", bulk=True, precision="fp64", t_reg=0.0),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "loop", "find", "setup", "batch", "cornelius",
                       "validity"])
    if kind == "cornelius":
        return dict(kind=kind, dim=rng.choice([3, 4]), cells=_log(rng, 64, 16384))
    eos = rng.choice(["table", "table", "wb", "conformal"])
    bulk = rng.random() < 0.7 and eos != "conformal"
    precision = rng.choice(["fp64", "mixed"] if kind == "batch" else
                           ["fp64", "fp64", "mixed", "mixed_f64_roots"])
    case = dict(kind=kind, h=round(rng.uniform(0.1, 0.2), 3), dt=0.01, eos=eos, bulk=bulk,
                precision=precision, t_reg=rng.choice([0.0, 0.05]))
    if kind == "batch":
        flat = rng.random() < 0.6
        n = _log(rng, 41, 121) if flat else _log(rng, 31, 61)
        return dict(case, events=rng.randint(2, 12 if flat else 6), nx=n, ny=n + rng.randint(-8, 8),
                    nz=1 if flat else rng.randint(9, 31), spread=rng.randint(0, 10),
                    nt=rng.randint(20, 60))
    if rng.random() < 0.4 and kind != "validity":
        nx = _log(rng, 41, 301)
        case.update(nx=nx, ny=max(41, nx + rng.randint(-20, 20)), nz=1)
    else:
        nx = _log(rng, 41, 151)
        case.update(nx=nx, ny=max(41, nx + rng.randint(-20, 20)), nz=_log(rng, 11, 81))
    if kind == "steps":
        case.update(dt=0.002, steps=rng.randint(5, 25))
    return case


# ------------------------------------------------------------------ inputs

def _axis(n, h):
    return (np.arange(n) - (n - 1) / 2.0) * h


def _energy(case, seed, nx=None, ny=None):
    """Seeded energy density [fm^-4]: a broad transverse Gaussian with
    hotspots on it, falling off smoothly in eta and dense up to the lattice's
    edge, so that the viscous evolution is a stable one."""
    r = np.random.default_rng(seed)
    nx, ny, nz, h = nx or case["nx"], ny or case["ny"], case["nz"], case["h"]
    x, y = _axis(nx, h)[:, None], _axis(ny, h)[None, :]
    half = 0.5 * (min(nx, ny) - 1) * h
    e = r.uniform(12.0, 18.0) * np.exp(-(x * x + y * y) / (2.0 * (0.42 * half) ** 2))
    for _ in range(int(r.integers(20, 60))):
        rad, phi = 0.45 * half * np.sqrt(r.random()), 2 * np.pi * r.random()
        xk, yk = rad * np.cos(phi), rad * np.sin(phi)
        e = e + r.uniform(0.0, 5.0) * np.exp(-((x - xk) ** 2 + (y - yk) ** 2) / (2 * 0.7 ** 2))
    eta = _axis(nz, 0.1)
    e = (e / HBARC)[:, :, None] * np.exp(-0.5 * (eta / 6.0) ** 2)[None, None, :]
    return np.asfortranarray(e + 1e-3)


def _flow(case, seed, e, p):
    """Flow, shear and bulk of a pre-equilibrium stage: radial and
    longitudinal velocities that grow outwards with seeded ripples, a small
    pi^{mu nu} transverse to the flow and traceless, and Pi."""
    r = np.random.default_rng(seed + 1_000_003)
    nx, ny, nz, h, t0 = case["nx"], case["ny"], case["nz"], case["h"], 0.5
    x, y = _axis(nx, h)[:, None, None], _axis(ny, h)[None, :, None]
    eta = _axis(nz, 0.1)[None, None, :]
    k = r.uniform(0.5, 1.5, 3)
    half = 0.5 * (min(nx, ny) - 1) * h
    ux = 0.3 * x / half + 0.02 * np.sin(k[0] * y) + 0.0 * eta
    uy = 0.3 * y / half + 0.02 * np.sin(k[1] * x) + 0.0 * eta
    un = (0.05 * np.tanh(eta) * np.cos(k[2] * x) + 0.0 * y) if nz > 1 else 0.0 * ux
    ut = np.sqrt(1 + ux ** 2 + uy ** 2 + (t0 * un) ** 2)
    # pi from three spatial amplitudes: the projector's u^mu u^nu part keeps
    # it transverse to first order, which is what such input files hold
    a, b = 0.05 * (e + p), 0.02 * (e + p)
    pixx, piyy = a * np.cos(k[0] * x), -a * np.cos(k[0] * x) + b
    pinn = -b / t0 ** 2
    pixy, pixn, piyn = b * np.sin(k[1] * y), 0.1 * b * np.sin(k[2] * x), 0.1 * b + 0.0 * x
    pitx = (pixx * ux + pixy * uy + t0 ** 2 * pixn * un) / ut
    pity = (pixy * ux + piyy * uy + t0 ** 2 * piyn * un) / ut
    pitn = (pixn * ux + piyn * uy + t0 ** 2 * pinn * un) / ut
    pitt = (pitx * ux + pity * uy + t0 ** 2 * pitn * un) / ut
    pi10 = [pitt, pitx, pity, pitn, pixx, pixy, pixn, piyy, piyn, pinn]
    f = lambda v: np.asfortranarray(np.broadcast_to(v, e.shape), dtype=np.float64)  # noqa: E731
    return [f(v) for v in (ut, ux, uy, un)], [f(v) for v in pi10], f(-0.02 * p)


def _options(case):
    import gpuvh
    return gpuvh.options(EOS[case["eos"]], case["bulk"], PRECISION[case["precision"]],
                         0.16 / HBARC)


def _hydro(case):
    import gpuvh
    return gpuvh.hydro(0.5, 0.16, T_fo_GeV=0.15, T_reg_GeV=case["t_reg"])


def _context(case):
    import gpuvh
    L = gpuvh.lattice(case["nx"], case["ny"], case["nz"], case["h"], case["h"], 0.1, case["dt"])
    return gpuvh.Context(L, _hydro(case), _options(case))


def _rest(ctx, e):
    """Initial fields of an event at rest with no viscous stress."""
    z = np.zeros(e.shape, order="F")
    p = ctx.equilibrium_pressure(e.ravel(order="F")).reshape(e.shape, order="F")
    return [e, p, np.ones(e.shape, order="F"), z, z, z]


def _row_buffer(case, nx, ny):
    """A buffer for the rows of any surface of the case: the surfaces of these
    events are rings around the fluid, so their elements go with the perimeter."""
    n = 40 * (nx + ny) * (case["nt"] // 8 if case["kind"] == "batch" else 1)
    rows = np.zeros((max(1024, n * max(1, case["nz"] - 1)), 20))
    return rows, (rows if case["precision"] == "fp64"
                  else torch.zeros(rows.shape, dtype=torch.float32))


def _keep_rows(bufs, last, n, read):
    """The n rows that read(pointer) gives into the buffers; what an earlier,
    longer surface left behind them is cleared.  Returns what the program
    keeps."""
    buf, keep = bufs
    if n > len(buf):
        raise RuntimeError("%d rows, a buffer of %d" % (n, len(buf)))
    if n and read(buf.ctypes.data_as(ctypes.POINTER(ctypes.c_double))):
        raise RuntimeError("reading the rows failed")
    if keep is not buf:
        keep[:n].copy_(torch.from_numpy(buf[:n]))
    keep[n:last] = 0
    return keep


def _search(s, n, t):
    """The window search at loop index n; its rows into the state's buffer."""
    import gpuvh
    count, ctx = ctypes.c_longlong(), s["ctx"]
    if gpuvh.lib().gvh_freezeout_find(ctx.h, n, t, ctypes.byref(count)):
        raise RuntimeError(gpuvh.lib().gvh_last_error())
    rows = _keep_rows(s["rows"], s["nrows"], count.value,
                      lambda p: gpuvh.lib().gvh_freezeout_rows(ctx.h, p, count.value))
    s["nrows"] = count.value
    return rows


def _start(s):
    s["ctx"].set_initial_state(0.5, *s["fields"])
    s["n"] = 0


def prepare(case, seed):
    import gpuvh
    if case["kind"] == "cornelius":
        dim, n = case["dim"], case["cells"]
        g = torch.Generator().manual_seed(seed)
        # corner values of a linear field with a random gradient and some
        # roughness, placed so that the iso-value cuts it: surface cells
        grad = torch.randn(n, dim, generator=g, dtype=torch.float64)
        bits = torch.tensor([[(c >> (dim - 1 - k)) & 1 for k in range(dim)]
                             for c in range(1 << dim)], dtype=torch.float64)
        v = (bits - 0.5) @ grad.T
        v = v.T + 0.1 * torch.randn(n, 1 << dim, generator=g, dtype=torch.float64)
        v = 2.0 + v + 0.3 * torch.randn(n, 1, generator=g, dtype=torch.float64)
        dx = np.array([0.1, 0.15, 0.15, 0.1][:dim])
        return dict(case=case, corners=v.contiguous().cuda(), dx=dx,
                    counts=torch.zeros(n, dtype=torch.int32, device="cuda"),
                    cen=torch.zeros(n, 10, dim, dtype=torch.float64, device="cuda"),
                    nrm=torch.zeros(n, 10, dim, dtype=torch.float64, device="cuda"))
    if case["kind"] == "batch":
        events = []
        for k in range(case["events"]):
            nx, ny = case["nx"] + (k % 3) * case["spread"], case["ny"] + (k % 3) * case["spread"]
            L = gpuvh.lattice(nx, ny, case["nz"], case["h"], case["h"], 0.1, case["dt"],
                              nt=case["nt"] + 2 * (k % 5))
            events.append((L, _energy(case, 1000 * seed + k, nx, ny)))
        batch = gpuvh.Batch(_options(case), max_events=16, fofreq=FOFREQ, autotune=False)
        bufs = [_row_buffer(case, e.shape[0], e.shape[1]) for _, e in events]
        return dict(case=case, batch=batch, events=events, hydro=_hydro(case), rows=bufs,
                    nrows=[0] * len(bufs))
    e = _energy(case, seed)
    ctx = _context(case)
    s = dict(case=case, ctx=ctx, fields=_rest(ctx, e))
    if case["kind"] == "setup":
        u, pi10, Pi = _flow(case, seed, e, s["fields"][1])
        s["fields"] = [e, s["fields"][1]] + u + [pi10, Pi if case["bulk"] else None]
        return s
    _start(s)
    if case["kind"] in ("loop", "find"):
        s["e_fo"] = ctx.energy_density_of_T(0.15 / HBARC)
        ctx.freezeout_init(FOFREQ, s["e_fo"])
        s["rows"], s["nrows"] = _row_buffer(case, case["nx"], case["ny"]), 0
    if case["kind"] == "find":  # the history of steps 1..19: a full window
        for n in range(1, 2 * FOFREQ):
            ctx.freezeout_record(n)
            ctx.step(0.5 + (n - 1) * case["dt"])
    if case["kind"] == "validity":
        u, pi10, Pi = _flow(case, seed, e, s["fields"][1])
        ctx.set_initial_state(0.5, e, s["fields"][1], *u, pi10, Pi if case["bulk"] else None)
        ctx.validity_enable()
    ctx.synchronize()
    return s


# ------------------------------------------------------------------ a pass

def _out(case, v):
    return v if case["precision"] == "fp64" else v.astype(np.float32)


def run(state):
    import gpuvh
    case = state["case"]
    kind = case["kind"]
    if kind == "cornelius":
        dx = state["dx"]
        rc = gpuvh.lib().gvh_cornelius_cells_noalloc(
            case["dim"], case["cells"], state["corners"].data_ptr(),
            dx.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 2.0, state["counts"].data_ptr(),
            state["cen"].data_ptr(), state["nrm"].data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError(gpuvh.lib().gvh_last_error())
        return dict(counts=state["counts"], centroids=state["cen"], normals=state["nrm"])
    if kind == "batch":
        b = state["batch"]
        ids = [b.submit(L, state["hydro"], e, surface=True, keep_state=True)
               for L, e in state["events"]]
        b.run()
        done = {r["id"]: r for r in b.poll()}
        out = []
        for k, i in enumerate(ids):
            if done[i]["status"]:
                raise RuntimeError("event status %d" % done[i]["status"])
            n = done[i]["surface_rows"]
            rows = _keep_rows(state["rows"][k], state["nrows"][k], n,
                              lambda p: gpuvh.lib().gvh_batch_rows(b.h, i, p, n))
            state["nrows"][k] = n
            out.append(dict(rows=rows, count=n, e=_out(case, b.field(i, gpuvh.E))))
            b.release(i)
        return out
    ctx = state["ctx"]
    if kind == "setup":
        ctx.set_initial_state(0.5, *state["fields"])
        return {k: _out(case, ctx.get(f)) for k, f in
                (("ttt", gpuvh.TTT), ("ttx", gpuvh.TTX), ("tty", gpuvh.TTY), ("ttn", gpuvh.TTN))}
    if kind == "find":
        n = 2 * FOFREQ - 1
        rows = _search(state, n, 0.5 + (n - 1) * case["dt"])
        return dict(rows=rows, count=state["nrows"])
    if kind == "validity":
        ctx.check_validity(0.5)
        return {k: _out(case, ctx.get_validity(f)) for f, k in enumerate(VALIDITY)
                if case["bulk"] or "bulk" not in k}
    dt = case["dt"]
    if kind == "steps":
        if state["n"] + case["steps"] > 1000:  # the event is over: the next one
            _start(state)
        ctx.steps(0.5, state["n"], case["steps"])
        state["n"] += case["steps"]
        return {k: _out(case, ctx.get(f)) for k, f in SNAPSHOT.items() if case["bulk"] or k != "Pi"}
    if state["n"] + FOFREQ > 300:
        _start(state)
    above = 0
    for n in range(state["n"] + 1, state["n"] + FOFREQ + 1):
        ctx.freezeout_record(n)
        if n % FOFREQ == FOFREQ - 1:
            rows = _search(state, n, 0.5 + (n - 1) * dt)
        above = ctx.count_above(state["e_fo"])
        ctx.step(0.5 + (n - 1) * dt)
    state["n"] += FOFREQ
    return dict(rows=rows, count=state["nrows"], above=above)


# ------------------------------------------------------------------ work

def _cell_step(case):
    """Bytes and operations of one cell in one KT step, each value read and
    written once per Runge-Kutta stage: stage 1 reads q^n, e, p, u, u_prev and
    writes q, e, p, u; stage 2 reads those, q^n and u again and writes the new
    state.  About 2500 additions, multiplications and FMAs per stage."""
    nv = 15 if case["bulk"] else 14
    q = 8 * nv if case["precision"] == "fp64" else 32 + 4 * (nv - 4)
    dims = 1.0 if case["nz"] > 1 else 0.7
    return 5 * q + 8 * 32, 2 * 2500 * dims


def work(case):
    kind = case["kind"]
    if kind == "cornelius":
        n, d = case["cells"], case["dim"]
        return dict(bytes=n * (8 * (1 << d) + 4 + 2 * 8 * d), flops=n * (4000 if d == 4 else 300))
    cells = case["nx"] * case["ny"] * case["nz"]
    item = 8 if case["precision"] == "fp64" else 4
    rec = cells * (4 * 8 + 6 * item + 80)  # ten values read and ten written to the history
    b, f = _cell_step(case)
    if kind == "batch":
        total = dict(bytes=0, flops=0)
        for k in range(case["events"]):
            c = (case["nx"] + (k % 3) * case["spread"]) * (case["ny"] + (k % 3) * case["spread"])
            c *= case["nz"]
            steps = case["nt"] + 2 * (k % 5) + 1
            total["bytes"] += steps * c * (b + 4 * 8 + 6 * item + 80) + 16 * c
            total["flops"] += steps * c * f
        return total
    if kind == "setup":
        return dict(bytes=cells * 8 * (17 + 4), flops=cells * 20)
    if kind == "find":
        return dict(bytes=cells * 8 * (FOFREQ + 1), flops=cells * FOFREQ * 16)
    if kind == "validity":
        return dict(bytes=cells * (10 * 8 + 11 * item + 11 * 8), flops=cells * 600)
    if kind == "steps":
        n = len(SNAPSHOT) if case["bulk"] else len(SNAPSHOT) - 1
        return dict(bytes=cells * (case["steps"] * b + 8 * n), flops=cells * case["steps"] * f)
    return dict(bytes=FOFREQ * (cells * (b + 8) + rec) + cells * 8 * (FOFREQ + 1),
                flops=FOFREQ * cells * f)


# ------------------------------------------------------------------ exact
# The same in numpy and 64 bits: Kurganov-Tadmor with the generalised minmod
# limiter (theta = 2), Heun's two stages, Newton root-finds from the owning
# cell's energy density, second-order viscous sources (Bazow, Heinz &
# Strickland, arXiv:1608.06577), and cornelius (Huovinen & Petersen,
# arXiv:1206.3371).

class _Eos:
    def __init__(self, kind):
        self.kind = kind
        if kind == "table":
            path = os.path.join(PKG, "data", "eos_qcdlike_2000.dat")
            with open(path) as f:
                tok = next(ln for ln in f if ln.startswith("# nodes")).split()
            self.M, self.emin = int(tok[4]), int(tok[6])
            self.e, self.p, self.c, self.T = np.loadtxt(path).T

    def _at(self, e):
        n, M = len(self.e), self.M
        with np.errstate(invalid="ignore"):
            m, x = np.frexp(e)
            f = (2 * m - 1) * M
            j = np.where(np.isfinite(f), f, 0).astype(np.int64)
            k, r = (x - 1 - self.emin) * M + j, f - j
            r = np.where(k > n - 2, r + 1.0, r)
            k = np.clip(k, 0, n - 2)
            hi, lo = e >= self.e[-1], ~(e >= self.e[0])
        k = np.where(hi, n - 2, np.where(lo, 0, k))
        r = np.where(hi, (e - self.e[-2]) / (self.e[-1] - self.e[-2]),
                     np.where(lo, (e - self.e[0]) / (self.e[1] - self.e[0]), r))
        return k, r

    def p_cs2(self, e):
        if self.kind == "conformal":
            return e / 3.0, np.zeros_like(e)
        if self.kind == "table":
            k, r = self._at(e)
            return (self.p[k] + r * (self.p[k + 1] - self.p[k]),
                    self.c[k] + r * (self.c[k + 1] - self.c[k]))
        a = np.polynomial.polynomial.polyval
        return a(e, WB_P[0]) / a(e, WB_P[1]), a(e, WB_CS2[0]) / a(e, WB_CS2[1])

    def temperature(self, e):
        if self.kind == "conformal":
            return (e / 13.8997) ** 0.25
        if self.kind == "table":
            k, r = self._at(e)
            return self.T[k] + r * (self.T[k + 1] - self.T[k])
        a = np.polynomial.polynomial.polyval
        return a(e, WB_T[0]) / a(e, WB_T[1])

    def e_of_T(self, T):
        if self.kind == "conformal":
            return 13.8997 * T ** 4
        if self.kind == "table":
            if T <= self.T[0]:
                return 0.0 if T <= 0 else self.e[0] * (T / self.T[0]) ** 4
            k = min(int(np.searchsorted(self.T, T, side="right")) - 1, len(self.T) - 2)
            return self.e[k] + (T - self.T[k]) / (self.T[k + 1] - self.T[k]) * (
                self.e[k + 1] - self.e[k])
        a = np.polynomial.polynomial.polyval
        return a(T, WB_E[0]) / a(T, WB_E[1])


# Wuppertal-Budapest fits of the default equation of state: numerator and
# denominator coefficients in rising powers
WB_P = (
    [-0.25181736420168666, 9737.845799644809, 1.077580993288114e6, 3.1729694865420084e6,
     1.6357487344679043e6, 334334.4309240126, 41913.439282708554, 6340.448389300905,
     141.5073484468774, 0.7158279081255019, 0.0009417586777847889, 3.1188455176941583e-7,
     1.9531729608963267e-11],
    [45829.44617893836, 4.0574329080826794e6, 2.0931169138134286e7, 1.3512402226067686e7,
     1.7851642641834426e6, 278581.2989342773, 26452.34905933697, 499.04919730607065,
     2.3405487982094204, 0.002962497695527404, 9.601103399348206e-7, 5.928138360995685e-11,
     3.2581066229887368e-18])
WB_CS2 = (
    [5.191934309650155e-32, 4.123605749683891e-23, 3.1955868410879504e-16,
     1.4170364808063119e-10, 6.087136671592452e-6, 0.02969737949090831, 15.382615282179595,
     460.6487249985994, 1612.4245252438795, 275.0492627924299, 58.60283714484669,
     6.504847576502024, 0.03009027913262399, 8.189430244031285e-6],
    [1.4637868900982493e-30, 6.716598285341542e-22, 3.5477700458515908e-15,
     1.1225580509306008e-9, 0.00003551782901018317, 0.13653226327408863, 60.85769171450653,
     1800.5461219450308, 15190.225535036281, 590.2572000057821, 293.99144775704605,
     21.461303090563028, 0.09301685073435291, 0.000024810902623582917])
WB_T = (
    [1.510073201405604e-29, 8.014062800678687e-18, 2.4954778310451065e-10, 0.000063810382643387,
     0.4873490574161924, 207.48582344326206, 6686.07424325115, 14109.766109389702,
     1471.6180520527757, 14.055788949565482, 0.015421252394182246, 1.5780479034557783e-6],
    [7.558667139355393e-28, 1.3686372302041508e-16, 2.998130743142826e-9, 0.0005036835870305458,
     2.316902328874072, 578.0778724946719, 11179.193315394154, 17965.67607192861,
     1051.0730543534657, 5.916312075925817, 0.003778342768228011, 1.8472801679382593e-7])
WB_E = (
    [-0.011958188410851651, 119.89423098138208, -3156.9475699248055, 32732.86844374939,
     -187899.8994764422, 712537.3610845465, -1.557049803609345e6, 1.4852519861308339e6,
     532132.6079941876, -1.963099445042592e6, -4484.44579242679, 1.7984228830058286e6,
     119345.25619517374, -1.3499773937058165e6, -207838.4995663606, 654970.2138652403,
     -78643.00334616247, 40274.00078068926, 422619.58977657766, -409688.07836393174,
     -62005.75915066359, 46788.14270090656, 40784.330477857235, -12589.47744840392],
    [31630.074365558292, -127100.88940643385, 173528.1225422275, -39403.297956865215,
     -85582.57873541754, 9320.560804233442, 50882.74198960172, 20335.926473421183,
     -14897.725710713818, -23836.484117457, -13726.013896090335, 4517.908673107615,
     18056.19917986404, 14954.82860467155, 2569.623976952738, -9304.046211514986,
     -15606.429173842751, 8383.710735812094, 1591.3177623932843, -678.748230997762,
     -33.58687934953277, 3.2520554133126285, -0.19647288043440464, 0.005443394551264717])


def _half_slope(x, y, z):
    a, b, c = y - x, z - x, z - y
    m = np.minimum(np.minimum(np.abs(a), np.abs(c)), 0.25 * np.abs(b))
    return np.where((a < 0) == (c < 0), np.copysign(m, a), 0.0)


def _solve_e(eos, guess, M0, M, Pi):
    if eos.kind == "conformal":
        return np.abs(np.sqrt(np.abs(4 * M0 * M0 - 3 * M)) - M0)
    out = guess.copy()
    idx = np.arange(out.size)
    for _ in range(200):
        e, m0, m, b = out[idx], M0[idx], M[idx], Pi[idx]
        p, cs2 = eos.p_cs2(e)
        w = p / e
        A = m0 * (1 - w) + b
        B = m0 * (m0 + b) - m
        H = np.sqrt(np.abs(A * A + 4 * w * B))
        D = (A - H) / (2 * w)
        f = e + D
        fp = 1 - ((cs2 - w) * (B + D * H - ((cs2 - w) * w * D * m0) / e)) / (w * e * H)
        new = e - f / fp
        out[idx] = new
        idx = idx[~(np.abs(new - e) <= 0.001 * np.abs(new)) & ~np.isnan(new)]
        if not idx.size:
            break
    return out


def _invert(eos, t, W, guess):
    """e, p and M^mu of conserved values W[9] = (T^{tau mu}, pi^{tau mu}, Pi)."""
    M0, M1, M2, M3 = (W[k] - W[4 + k] for k in range(4))
    M = M1 * M1 + M2 * M2 + t * t * M3 * M3
    e = M0 - M / M0
    newton = ~(guess <= 0.1)
    if newton.any():
        e[newton] = _solve_e(eos, guess[newton], M0[newton], M[newton], W[8][newton])
    p = eos.p_cs2(e)[0]
    low = e < 1e-7
    return np.where(low, 1e-7, e), np.where(low, 1e-7, p), (M0, M1, M2, M3)


class _KT:
    """The state of one event: q[15], e, p, u[4] and the previous u."""

    def __init__(self, case):
        self.case, self.eos = case, _Eos(case["eos"])
        self.h = (case["h"], case["h"], 0.1)
        self.dt = case["dt"]
        self.dims = 3 if case["nz"] > 1 else 2
        self.nv = 15 if case["bulk"] else 14
        self.e_reg = self.eos.e_of_T(case["t_reg"] / HBARC)

    def start(self, e, p, u=None, pi10=None, Pi=None):
        z = np.zeros_like(e)
        u = [np.ones_like(e), z, z, z] if u is None else u
        pi10 = [z] * 10 if pi10 is None else pi10
        Pi = z if Pi is None or not self.case["bulk"] else Pi
        P = p + Pi
        T = [(e + P) * u[0] * u[m] + pi10[m] - (P if m == 0 else 0) for m in range(4)]
        self.q, self.e, self.p = np.stack(T + list(pi10) + [Pi]), e, p
        self.u, self.up = np.stack(u), np.stack(u)

    def _shift(self, padded, d, o):
        i = [slice(2, -2)] * 3
        i[d] = slice(2 + o, padded.shape[1 + d] - 2 + o)
        return padded[(slice(None), *i)]

    def _stage(self, q, qn, e, p, u, up, t, tinf):
        pad = lambda a: np.pad(a, ((0, 0), (2, 2), (2, 2), (2, 2)), mode="edge")  # noqa: E731
        Q, UP = pad(q), pad(np.concatenate([u, p[None]]))
        g = np.zeros((3, 5) + e.shape)
        for d in range(self.dims):
            g[d] = 2 * _half_slope(self._shift(UP, d, -1), self._shift(UP, d, 0),
                                   self._shift(UP, d, 1)) / self.h[d]
        acc = q + self.dt * self._sources(q, e, p, u, up, g, t)
        for d in range(self.dims):
            acc += self.dt * self._direction(Q, u, e, t, d)
        if qn is not None:
            acc = (acc + qn) / 2
        W = [acc[k].ravel() for k in (0, 1, 2, 3, 4, 5, 6, 7, 14)]
        e2, p2, M = _invert(self.eos, tinf, W, e.ravel())
        P = p2 + W[8]
        E = 1.0 / (e2 + P)
        ut = np.sqrt(np.abs((M[0] + P) * E))
        u2 = np.stack([ut, M[1] * E / ut, M[2] * E / ut, M[3] * E / ut])
        e2, p2, u2 = e2.reshape(e.shape), p2.reshape(e.shape), u2.reshape(u.shape)
        self.factor = self._regulate(acc, e2, p2, u2, tinf)
        return acc, e2, p2, u2

    def _direction(self, Q, u, e, t, d):
        """(H_b - H_f)/h and the central-difference sources of direction d."""
        v = [self._shift(Q, d, o) for o in (-2, -1, 0, 1, 2)]
        hm, h0, hp = (_half_slope(*v[k:k + 3]) for k in range(3))
        states = [v[3] - hp, v[2] + h0, v[2] - h0, v[1] + hm]
        vel = []
        for W in states:
            w = [W[k].ravel() for k in (0, 1, 2, 3, 4, 5, 6, 7, 14)]
            ee, pp, M = _invert(self.eos, t, w, e.ravel())
            P = pp + w[8]
            s = np.where(ee + P > 0, M[1 + d], -M[1 + d])
            vel.append((s / np.abs(M[0] + P)).reshape(e.shape))
        flux = lambda k: 0.5 * (vel[k] * states[k] + vel[k + 1] * states[k + 1] - np.maximum(  # noqa: E731
            np.abs(vel[k]), np.abs(vel[k + 1])) * (states[k] - states[k + 1]))
        out = (flux(2) - flux(0)) / self.h[d]
        c = (v[3] - v[1]) / (2 * self.h[d])
        vs = u[1 + d] / u[0]
        out[0] += c[4] * vs - c[5 + d] - vs * c[14]
        spatial = {0: (8, 9, 10), 1: (9, 11, 12), 2: (10, 12, 13)}[d]
        for m in range(3):
            out[1 + m] += c[5 + m] * vs - c[spatial[m]]
        out[1 + d] -= c[14] / (t * t if d == 2 else 1.0)
        return out

    def _sources(self, q, e, p, u, up, g, t):
        """Geometric and gradient sources of T^{tau mu}, relaxation equations
        of pi^{mu nu} and Pi."""
        t2 = t * t
        ut, ux, uy, un = u
        gu = g[:, :4]  # [direction][component]
        S = np.zeros_like(q)
        Pi, names = q[14], ((0, 0), (0, 1), (0, 2), (0, 3), (1, 1), (1, 2), (1, 3), (2, 2), (2, 3),
                            (3, 3))
        pi = np.empty((4, 4) + e.shape)
        for k, (a, b) in enumerate(names):
            pi[a, b] = pi[b, a] = q[4 + k]
        PP = p + Pi
        tnn = (e + PP) * un * un + PP / t2 + pi[3, 3]
        v = [u[1 + d] / ut for d in range(3)]
        dkvk = sum((gu[d][1 + d] - v[d] * gu[d][0]) / ut for d in range(3))
        S[0] = (-(q[0] / t + t * tnn) + dkvk * (pi[0, 0] - p - Pi)
                - sum(v[d] * g[d][4] for d in range(3)))
        S[1] = -q[1] / t - g[0][4] + dkvk * pi[0, 1]
        S[2] = -q[2] / t - g[1][4] + dkvk * pi[0, 2]
        S[3] = -3 * q[3] / t - g[2][4] / t2 + dkvk * pi[0, 3]

        T = self.eos.temperature(e)
        taupi_inv = float(np.float32(0.2)) * T / 0.16
        beta_pi = float(np.float32(0.2)) * (e + p)
        dtu = (u - up) / self.dt
        du = [ut * dtu[m] + sum(u[1 + d] * gu[d][m] for d in range(3)) for m in range(4)]
        D = [du[0] + t * un * un, -du[1], -du[2], -t2 * du[3] - 2 * t * ut * un]
        theta = ut / t + dtu[0] + gu[0][1] + gu[1][2] + gu[2][3]
        th3 = theta / 3
        un2, ut2 = un * un, ut * ut
        s = np.empty_like(pi)
        s[0, 0] = -t * ut * un2 + (dtu[0] - ut * du[0]) + (ut2 - 1) * th3
        for m, d in ((1, 0), (2, 1)):
            s[0, m] = (-(t * un2 * u[m]) / 2 + (dtu[m] - gu[d][0]) / 2
                       - (u[m] * du[0] + ut * du[m]) / 2 + ut * u[m] * th3)
            s[m, m] = -(gu[d][m] + u[m] * du[m]) + (1 + u[m] * u[m]) * th3
            s[m, 3] = (-ut * u[m] * un / t - (gu[d][3] + gu[2][m] / t2) / 2
                       - (un * du[m] + u[m] * du[3]) / 2 + u[m] * un * th3)
        s[0, 3] = (-un * (2 * ut2 + t2 * un2) / (2 * t) + (dtu[3] - gu[2][0] / t2) / 2
                   - (un * du[0] + ut * du[3]) / 2 + ut * un * th3)
        s[1, 2] = (-(gu[1][1] + gu[0][2]) / 2 - (uy * du[1] + ux * du[2]) / 2 + ux * uy * th3)
        s[3, 3] = (-ut * (1 + 2 * t2 * un2) / t ** 3 - gu[2][3] / t2 - un * du[3]
                   + (1 / t2 + un2) * th3)
        for a in range(4):
            for b in range(a):
                s[a, b] = s[b, a]
        # vorticity omega^mu_nu
        w = np.zeros_like(pi)
        for m, d in ((1, 0), (2, 1)):
            w[0, m] = w[m, 0] = (-dtu[m] - gu[d][0] + ut * du[m] - u[m] * du[0]
                                 - t * un2 * u[m]) / 2
            w[m, 3] = (t2 * gu[d][3] - gu[2][m] - u[m] * D[3] - t2 * un * du[m]) / 2
            w[3, m] = -w[m, 3] / t2
        w[0, 3] = (-t2 * dtu[3] - 2 * t * un - gu[2][0] - ut * D[3] - t2 * un * du[0]
                   - t ** 3 * un * un2) / 2
        w[3, 0] = w[0, 3] / t2
        w[1, 2] = (gu[0][2] - gu[1][1] + ux * du[2] - uy * du[1]) / 2
        w[2, 1] = -w[1, 2]

        metric = (1.0, -1.0, -1.0, -t2)  # lowers the index that is summed over
        a = [sum(pi[m, k] * D[k] for k in range(4)) for m in range(4)]
        ps = sum(metric[k] * metric[m] * pi[k, m] * s[k, m] for k in range(4) for m in range(4))
        delta = (1.0, 1.0, 1.0, 1.0 / t2)
        d_pp, t_pp, l_pP = 1.33333, 1.42857, 1.2
        for k, (m, n) in enumerate(names):
            I1 = u[m] * a[n] + u[n] * a[m]
            # pi^{mu lambda} omega^nu_lambda + pi^{nu lambda} omega^mu_lambda
            I3 = sum(pi[m, c] * w[n, c] + pi[n, c] * w[m, c] for c in range(4))
            I4 = sum(metric[c] * (pi[m, c] * s[n, c] + pi[n, c] * s[m, c]) / 2 for c in range(4))
            proj = u[m] * u[n] + (0 if m != n else (-1.0 if m == 0 else delta[m]))
            I4 = I4 + proj * ps / 3 if m or n else I4 - (1 - ut2) * ps / 3
            I = I1 + d_pp * theta * pi[m, n] - I3 + t_pp * I4 - l_pP * Pi * s[m, n]
            r = 2 * beta_pi * s[m, n] - pi[m, n] * taupi_inv - I
            # Christoffel terms of the Milne frame
            for x, y in ((m, n), (n, m)):
                if x == 0:
                    r = r - un * t * pi[3, y]
                if x == 3:
                    r = r - (ut * pi[3, y] + un * pi[0, y]) / t
            S[4 + k] = r / ut + pi[m, n] * dkvk
        if self.nv == 15:
            cs2 = self.eos.p_cs2(e)[1]
            b = float(np.float32(0.333333)) - cs2
            x = T / (0.16 / HBARC)
            with np.errstate(over="ignore"):
                zeta = np.where(
                    x > 1.05, 0.9 * np.exp(-(x - 1) / 0.025) + 0.25 * np.exp(-(x - 1) / 0.13)
                    + 0.001, np.where(
                        x < 0.995, 0.9 * np.exp((x - 1) / 0.0025) + 0.22 * np.exp((x - 1) / 0.022)
                        + 0.03, -13.77 * x * x + 27.55 * x - 13.45))
            tau_inv = 15 * b * b * T / zeta
            dPi = (-15 * b * b * (e + p) * theta - Pi * tau_inv - 0.666667 * Pi * theta
                   + float(np.float32(1.6)) * b * ps)
            S[14] = dPi / ut + Pi * dkvk
        return S

    def _regulate(self, q, e, p, u, t):
        """Rescales pi in cells at or below e_reg; the factor of every cell."""
        low = ~(e > self.e_reg)
        fac = np.ones_like(e)
        if low.any():
            t2 = t * t
            pi = {k: q[4 + i][low] for i, k in enumerate(
                ("tt", "tx", "ty", "tn", "xx", "xy", "xn", "yy", "yn", "nn"))}
            w = dict(tt=1, tx=-2, ty=-2, tn=-2 * t2, xx=1, xy=2, xn=2 * t2, yy=1, yn=2 * t2,
                     nn=t2 * t2)
            s = np.sqrt(np.abs(sum(w[k] * pi[k] ** 2 for k in w)))
            ut, ux, uy, un = (c[low] for c in u)
            x = [pi["tt"] - pi["xx"] - pi["yy"] - pi["nn"] * t2]
            for a in ("tt tx ty tn", "tx xx xy xn", "ty xy yy yn", "tn xn yn nn"):
                k = a.split()
                x.append(-pi[k[3]] * t2 * un + pi[k[0]] * ut - pi[k[1]] * ux - pi[k[2]] * uy)
            with np.errstate(divide="ignore", invalid="ignore"):
                rho = s / np.sqrt(e[low] ** 2 + 3 * p[low] ** 2)
                for c in x:
                    rho = np.fmax(rho, c / (0.1 * s))
                f = np.where(np.abs(rho) < 1e-7, 1.0, np.tanh(rho) / rho)
            fac[low] = f
            q[4:14] *= fac
        return fac

    def step(self, t):
        dt = self.dt
        q1, e1, p1, u1 = self._stage(self.q, None, self.e, self.p, self.u, self.up, t, t + dt)
        q2, e2, p2, u2 = self._stage(q1, self.q, e1, p1, u1, self.u, t + dt, t + dt)
        self.q, self.e, self.p, self.u, self.up = q2, e2, p2, u2, self.u

    def ring_fields(self):
        q = self.q
        return [self.u[1], self.u[2], self.u[3], self.e, q[8], q[9], q[10], q[11], q[12], q[14]]


def _square(sq, h1, h2, v0):
    """Lines (start, end, outside point) of one face in its two free axes."""
    above = sum(sq[a][b] >= v0 for a in (0, 1) for b in (0, 1))
    if above in (0, 4):
        return []
    cut = []
    for a, b, h, fix, first in ((sq[0][0], sq[1][0], h1, 0.0, True), (sq[0][0], sq[0][1], h2, 0.0, False),
                                (sq[1][0], sq[1][1], h2, h1, False), (sq[0][1], sq[1][1], h1, h2, True)):
        if (a - v0) * (b - v0) < 0:
            x = (a - v0) / (a - b) * h
        elif a == v0 and b < v0:
            x = 1e-9 * h
        elif b == v0 and a < v0:
            x = (1.0 - 1e-9) * h
        else:
            continue
        cut.append((x, fix) if first else (fix, x))
    if len(cut) == 4:
        mid = 0.25 * (sq[0][0] + sq[0][1] + sq[1][0] + sq[1][1])
        if (sq[0][0] < v0 and mid < v0) or (sq[0][0] > v0 and mid > v0):
            cut[1], cut[2] = cut[2], cut[1]
        if mid < v0:
            out = [(0.5 * h1, 0.5 * h2)] * 2
        elif sq[0][0] < v0:
            out = [(0.0, 0.0), (h1, h2)]
        else:
            out = [(h1, 0.0), (0.0, h2)]
        return [(cut[0], cut[1], out[0]), (cut[2], cut[3], out[1])]
    if len(cut) != 2:
        return []
    low = [(a * h1, b * h2) for a in (0, 1) for b in (0, 1) if sq[a][b] < v0]
    n = max(1, len(low))
    return [(cut[0], cut[1], (sum(c[0] for c in low) / n, sum(c[1] for c in low) / n))]


def _near(a, b, strict):
    d = sum(abs(x - y) for x, y in zip(a, b))
    return d < 1e-10 if strict else d <= 1e-10


def _join(items, fits):
    """Groups of items: the first free one, then each that fits, the scan
    going on from the second item after every addition."""
    free, groups = list(range(len(items))), []
    while free:
        group, i = [], 0
        while i < len(items):
            if i in free and (not group or fits(group, i)):
                group.append(i)
                free.remove(i)
                i = 0
            i += 1
        groups.append(group)
    return groups


def _cube(v, axes, held, dx, v0):
    """Polygons of one cube v[2][2][2] over `axes`, the fourth axis held:
    lists of lines in four coordinates.  Also whether it is ambiguous."""
    lines, amb = [], 0
    for f in range(3):
        for j in (0, 1):
            a1, a2 = [a for k, a in enumerate(axes) if k != f]
            sq = np.take(v, j, axis=f).tolist()
            cuts = _square(sq, dx[a1], dx[a2], v0)
            amb += len(cuts) == 2
            for ln in cuts:
                full = []
                for c in ln:
                    x = [0.0] * 4
                    x[held[0]], x[axes[f]], x[a1], x[a2] = held[1], j * dx[axes[f]], c[0], c[1]
                    full.append(x)
                lines.append(full)
    if not lines:
        return [], False
    if not amb and len(lines) != 6:
        return [lines], False

    def fits(group, i):
        end = lines[group[-1]][1]
        s, e = _near(lines[i][0], end, True), _near(lines[i][1], end, True)
        if e:
            lines[i][0], lines[i][1] = lines[i][1], lines[i][0]
        return s or e

    return [[lines[i] for i in g] for g in _join(lines, fits)], True


def _polygon(lines, axes, normal):
    s, e, o = (np.array([ln[k] for ln in lines]) for k in range(3))
    mean = (s + e).sum(0) / (2.0 * len(lines))
    x1, x2, x3 = axes
    if len(lines) == 3:
        cen = mean
    else:
        A = 0.5 * np.linalg.norm(np.cross((s - mean)[:, axes], (e - mean)[:, axes]), axis=1)
        cen = ((s + e + mean) / 3.0 * A[:, None]).sum(0) / A.sum()
    if not normal:
        return cen, None
    n = 0.5 * np.cross((s - cen)[:, axes], (e - cen)[:, axes])
    n[((o - cen)[:, axes] * n).sum(1) < 0] *= -1
    full = np.zeros(4)
    full[axes] = n.sum(0)
    return cen, full


def _tetra_normals(a, b, c):
    n = np.empty_like(a)
    for k in range(4):
        i = [m for m in range(4) if m != k]
        det = (a[:, i[0]] * (b[:, i[1]] * c[:, i[2]] - b[:, i[2]] * c[:, i[1]])
               - a[:, i[1]] * (b[:, i[0]] * c[:, i[2]] - b[:, i[2]] * c[:, i[0]])
               + a[:, i[2]] * (b[:, i[0]] * c[:, i[1]] - b[:, i[1]] * c[:, i[0]]))
        n[:, k] = (1.0 if k % 2 == 0 else -1.0) / 6.0 * det
    return n


def _elements(v, dx, v0):
    """(centroid, normal) of every element of one cell, v[2]..[2] its corners."""
    above = int((v >= v0).sum())
    if above in (0, v.size):
        return []
    if v.ndim == 3:
        d4 = [1.0] + list(dx)
        polygons, _ = _cube(v, [1, 2, 3], (0, 0.0), d4, v0)
        got = [_polygon(p, [1, 2, 3], True) for p in polygons]
        return [(c[1:], n[1:]) for c, n in got]
    polygons, ambiguous, nlines = [], False, 0
    for a in range(4):
        axes = [k for k in range(4) if k != a]
        for j in (0, 1):
            got, amb = _cube(np.take(v, j, axis=a), axes, (a, j * dx[a]), dx, v0)
            ambiguous = ambiguous or amb
            for p in got:
                nlines += len(p)
                polygons.append((p, _polygon(p, axes, False)[0]))
    if not ambiguous:
        below = int((v < v0).sum())
        ambiguous = nlines == 24 and min(below, 16 - below) == 2

    def fits(group, i):
        return any(_near(l1[0], l2[0], False) or _near(l1[1], l2[0], False)
                   for l1 in polygons[i][0] for g in group for l2 in polygons[g][0])

    groups = _join(polygons, fits) if ambiguous else [list(range(len(polygons)))]
    out = []
    for g in groups:
        s, e, o, pc = (np.array(x) for x in zip(*[(ln[0], ln[1], ln[2], polygons[i][1])
                                                 for i in g for ln in polygons[i][0]]))
        mean = (s + e).sum(0) / (2.0 * len(s))
        V = np.linalg.norm(_tetra_normals(s - mean, e - mean, pc - mean), axis=1)
        cen = ((s + e + pc + mean) / 4.0 * V[:, None]).sum(0) / V.sum()
        n = _tetra_normals(s - cen, e - cen, pc - cen)
        n[((o - cen) * n).sum(1) < 0] *= -1
        out.append((cen, n.sum(0)))
    return out


def _window_rows(case, kt, ring, n, e_fo):
    """Surface rows of the window at loop index n of a 2+1D event."""
    nx, ny, h, dt, t = case["nx"], case["ny"], case["h"], case["dt"], 0.5 + (n - 1) * case["dt"]
    E = np.stack([s[3][:, :, 0] for s in ring])
    above = sum((E[a:a + FOFREQ, b:b + nx - 1, c:c + ny - 1] >= e_fo).astype(int)
                for a in (0, 1) for b in (0, 1) for c in (0, 1))
    hit = np.argwhere((above > 0) & (above < 8))
    rows = []
    for it, ix, iy in hit:
        for cen, nrm in _elements(E[it:it + 2, ix:ix + 2, iy:iy + 2], [dt, h, h], e_fo):
            f = cen / np.array([dt, h, h])
            w = np.einsum("a,b,c->abc", *[np.array([1 - x, x]) for x in f])
            val = [float(sum((w[a] * ring[it + a][m][ix:ix + 2, iy:iy + 2, 0]).sum()
                             for a in (0, 1))) for m in range(10)]
            # windows after the first place a cell one step late
            tau = 0.5 + (n - FOFREQ + it) * dt
            ev = np.array([val[3]])
            rows.append([cen[0] + tau, cen[1] + ix * h - (nx - 1) / 2 * h,
                         cen[2] + iy * h - (ny - 1) / 2 * h, 0.0, t * nrm[0], t * nrm[1],
                         t * nrm[2], 0.0, *val[:4], kt.eos.temperature(ev)[0],
                         kt.eos.p_cs2(ev)[0][0], *val[4:]])
    return np.array(rows).reshape(-1, 20)


def _validity(case, kt, e, p, u, pi10, Pi, t):
    """Knudsen and inverse Reynolds numbers of a state at rest in time
    (u_prev = u); the two that need the second-order terms are left out."""
    F = np.pad(np.stack(u), ((0, 0), (2, 2), (2, 2), (2, 2)), mode="edge")
    cd = [(kt._shift(F, d, 1) - kt._shift(F, d, -1)) / (2 * kt.h[d]) if d < kt.dims
          else np.zeros_like(np.stack(u)) for d in range(3)]
    T = kt.eos.temperature(e)
    theta = u[0] / t + cd[0][1] + cd[1][2] + cd[2][3]
    out = {k: None for k in VALIDITY if case["bulk"] or "bulk" not in k}
    out.update(taupi=5 * 0.16 / T, dxux=cd[0][1], dyuy=cd[1][2], theta=theta,
               regulations=np.ones_like(e), kn_taupi=5 * 0.16 * theta / T)
    t2 = t * t
    w = (1, -2, -2, -2 * t2, 1, 2, 2 * t2, 1, 2 * t2, t2 * t2)
    out["re_pi"] = np.sqrt(np.abs(sum(c * v * v for c, v in zip(w, pi10)))) / p
    if case["bulk"]:
        out["re_bulk"] = np.abs(Pi) / p
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "cornelius":
        dim, n = case["dim"], case["cells"]
        if n > (EXACT_CELLS_4D if dim == 4 else EXACT_CELLS_3D):
            return None
        s = prepare(case, seed)
        counts, cen, nrm = np.zeros(n, np.int32), np.zeros((n, 10, dim)), np.zeros((n, 10, dim))
        for i, v in enumerate(s["corners"].cpu().numpy().reshape((n,) + (2,) * dim)):
            for k, (c, m) in enumerate(_elements(v, list(s["dx"]), 2.0)):
                counts[i], cen[i, k], nrm[i, k] = k + 1, c, m
        return dict(counts=counts, centroids=cen, normals=nrm)
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind in ("batch", "loop"):  # hundreds of thousands of elements
        return None
    kt, e = _KT(case), np.ascontiguousarray(_energy(case, seed))
    p = kt.eos.p_cs2(e.ravel())[0].reshape(e.shape)
    if kind in ("setup", "validity"):
        u, pi10, Pi = _flow(case, seed, e, p)
        if kind == "validity":
            return _validity(case, kt, e, p, u, pi10, Pi, 0.5)
        kt.start(e, p, u, pi10, Pi)
        return dict(zip(("ttt", "ttx", "tty", "ttn"), kt.q[:4]))
    kt.start(e, p)
    if kind == "steps":
        if cells * case["steps"] * (1 if case["nz"] == 1 else 2) > EXACT_CELL_STEPS:
            return None
        for n in range(case["steps"]):
            kt.step(0.5 + n * case["dt"])
        return {k: v for k, v in zip(SNAPSHOT, kt.ring_fields()) if case["bulk"] or k != "Pi"}
    if case["nz"] > 1 or cells * 2 * FOFREQ > EXACT_CELL_STEPS:
        return None
    ring, last = [None] * (FOFREQ + 1), None
    for n in range(1, 2 * FOFREQ):
        # after an odd number of steps the history takes u, pi and Pi of the
        # step before, as the reference's host copy does
        now = kt.ring_fields()
        keep = last if (n - 1) % 2 and last is not None else now
        k = n % FOFREQ
        if k == 0:
            ring[0] = ring[FOFREQ]
        ring[k + 1] = keep[:3] + [now[3]] + keep[4:]
        last = now
        kt.step(0.5 + (n - 1) * case["dt"])
    rows = _window_rows(case, kt, ring, 2 * FOFREQ - 1, kt.eos.e_of_T(0.15 / HBARC))
    full = np.zeros(_row_buffer(case, case["nx"], case["ny"])[0].shape)
    full[:len(rows)] = rows
    return dict(rows=full, count=len(rows))
