"""Measured workloads of the library, one call (or a driver's short loop) each.

A case is a dict of plain values; `prepare` makes what a program holds before
the call (the state, buffers and the context or network it keeps), `run` makes
the call through the public Python binding, `exact` restates the result in
64-bit torch without the library.

Kinds
  field      one effective-field evaluation, device-resident buffers
             (Zeeman + exchange + anisotropy + DMI + FFT demag)
  host       the same through the AoS float64 host entry point, the layout of
             the Rust caller, transfers included
  rk45       adaptive Dormand-Prince attempts of one film: one at a time
             (attempts = 0) or several per call with the controller on the
             device
  films      several attempts of many independent films in one call
  relax      damping-only RK23 attempts, then an energy breakdown
  mg         a field evaluation whose demag is the multigrid Poisson solve
  net        inference of the multigrid's learned initial guess
  train      one training step of it, with the gradients
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "llg-sim_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import llgmi as L  # noqa: E402

DEV = "cuda:0"
MU0 = 4.0 * math.pi * 1e-7
GAMMA = L.GAMMA_E_RAD_PER_S_T
B_EXT = (-24.6e-3, 4.3e-3, 0.0)
# perpendicular film with interfacial DMI, and a soft film
PERP = dict(ms=5.8e5, a_ex=1.5e-11, k_u=8e5, dmi=3e-3)
SOFT = dict(ms=8.0e5, a_ex=1.3e-11, k_u=0.0, dmi=0.0)
CELLS = {"2x2x1": (2e-9, 2e-9, 1e-9), "3x3x3": (3e-9, 3e-9, 3e-9), "4x4x3": (4e-9, 4e-9, 3e-9)}


def listed():
    return [
        # a macro-cell device or a unit test's film: the call is launches and latency
        {"name": "field_64", "kind": "field", "nx": 64, "ny": 64, "cell": "4x4x3", "f32": True, "perp": True,
         "holes": False},
        # the benchmark film: one evaluation of a simulation in steady use
        {"name": "field_1024", "kind": "field", "nx": 1024, "ny": 1024, "cell": "2x2x1", "f32": True, "perp": True,
         "holes": False},
        # a large patterned film of a ragged size (hole lattice, geometry mask)
        {"name": "field_1900x1100_holes", "kind": "field", "nx": 1900, "ny": 1100, "cell": "2x2x1", "f32": True,
         "perp": True, "holes": True},
        # a large film, powers of two
        {"name": "field_2048", "kind": "field", "nx": 2048, "ny": 2048, "cell": "2x2x1", "f32": True, "perp": True,
         "holes": False},
        # the drop-in call of the Rust program: double precision, host buffers
        {"name": "host_700x500_f64", "kind": "host", "nx": 700, "ny": 500, "cell": "3x3x3", "f32": False,
         "perp": True, "holes": False},
        # a standard-problem film stepped from a driver's loop, double precision
        {"name": "rk45_128x64_f64", "kind": "rk45", "nx": 128, "ny": 64, "cell": "4x4x3", "f32": False,
         "perp": False, "attempts": 0},
        # dynamics of the benchmark film
        {"name": "rk45_1024", "kind": "rk45", "nx": 1024, "ny": 1024, "cell": "2x2x1", "f32": True, "perp": True,
         "attempts": 16},
        # a parameter sweep: 64 films of mixed sizes and materials
        {"name": "films_64", "kind": "films", "count": 64, "set": 64, "f32": True, "attempts": 8},
        # relaxing a mid-sized film of a ragged size towards its ground state
        {"name": "relax_500x300", "kind": "relax", "nx": 500, "ny": 300, "cell": "3x3x3", "f32": True, "perp": False,
         "steps": 10},
        # the multigrid solve of a patterned film to a tight tolerance, cold
        {"name": "mg_512_holes", "kind": "mg", "nx": 512, "ny": 512, "cell": "3x3x3", "f32": False, "perp": False,
         "default": False},
        # inference of the initial guess for that film's box
        {"name": "net_528", "kind": "net", "batch": 1, "h": 528, "w": 528, "out": 36},
        # training it
        {"name": "train_8x528", "kind": "train", "batch": 8, "h": 528, "w": 528, "out": 36},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["field", "field", "field", "host", "rk45", "rk45", "films", "relax", "mg", "mg", "net",
                       "train"])
    if kind in ("net", "train"):
        return {"kind": kind, "batch": rng.randint(1, 3) if kind == "net" else rng.randint(1, 6),
                "h": 8 * rng.randint(12, 66), "w": 8 * rng.randint(12, 66), "out": rng.choice([20, 28, 36])}
    if kind == "films":
        return {"kind": kind, "count": rng.randint(8, 48), "set": rng.randint(0, 1 << 20), "f32": True,
                "attempts": rng.randint(2, 8)}
    hi = {"field": 2048, "host": 1024, "rk45": 1024, "relax": 700, "mg": 512}[kind]
    c = {"kind": kind, "nx": _log_int(rng, 32, hi), "ny": _log_int(rng, 32, hi), "cell": rng.choice(sorted(CELLS)),
         "f32": rng.random() < 0.7 and kind not in ("host", "mg"), "perp": rng.random() < 0.5}
    if kind in ("field", "host"):
        c["holes"] = rng.random() < 0.3
    elif kind == "rk45":
        c["attempts"] = rng.choice([0, rng.randint(2, 16)])
    elif kind == "relax":
        c["steps"] = rng.randint(4, 10)
    else:
        # the default operator (27-point, Galerkin, weighted Jacobi) or the
        # 7-point red-black one, each from a cold start
        c["cell"], c["perp"], c["default"] = "3x3x3", False, rng.random() < 0.5
        if c["default"]:
            c["nx"], c["ny"] = min(c["nx"], 256), min(c["ny"], 256)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _film(nx, ny, seed):
    """Smoothed random unit vectors, float64 [3, ny, nx] on the GPU."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    m = torch.randn((3, ny, nx), generator=g, dtype=torch.float64, device=DEV)
    for _ in range(3):
        m = 0.25 * (m.roll(1, 1) + m.roll(-1, 1) + m.roll(1, 2) + m.roll(-1, 2))
    return m / m.square().sum(0, keepdim=True).sqrt()


def _holes(nx, ny, cell, pitch=96e-9, radius=24e-9):
    """Square lattice of circular holes, uint8 [ny, nx] (1 = material)."""
    x = (torch.arange(nx, dtype=torch.float64, device=DEV) + 0.5) * cell[0]
    y = (torch.arange(ny, dtype=torch.float64, device=DEV) + 0.5) * cell[1]
    fx, fy = x % pitch - 0.5 * pitch, y % pitch - 0.5 * pitch
    return ((fx * fx)[None, :] + (fy * fy)[:, None] > radius * radius).to(torch.uint8)


def _material(case):
    return dict(PERP if case["perp"] else SOFT)


def _alpha(case):
    return 0.3 if case["perp"] else 0.02


def _case_dt(case):
    return _first_dt(_material(case), CELLS[case["cell"]], _alpha(case), case["kind"] == "relax")


def _specs(count, number):
    """Grid, material and damping of each film of a set."""
    rng = np.random.default_rng(number)
    films = []
    for _ in range(count):
        nx, ny = int(rng.choice([64, 128, 256, 512])), int(rng.choice([64, 128, 256]))
        dxy = float(rng.uniform(2e-9, 5e-9))
        films.append(dict(nx=nx, ny=ny, cell=(dxy, dxy, 3e-9), alpha=float(rng.uniform(0.01, 0.5)),
                          mat=dict(ms=float(rng.uniform(4e5, 1.2e6)), a_ex=float(rng.uniform(5e-12, 2e-11)),
                                   k_u=float(rng.uniform(0.0, 5e5)), dmi=float(rng.uniform(0.0, 4e-3)))))
    return films


def _inputs(case, seed):
    """(m, geometry mask or None) of a one-film case."""
    cell = CELLS[case["cell"]]
    m, geom = _film(case["nx"], case["ny"], seed), None
    if case["kind"] == "mg" or case.get("holes"):
        geom = _holes(case["nx"], case["ny"], cell)
        m = m * geom
    return m, geom


def _layers(base, c_pad):
    c = [base << k for k in range(4)]
    rows = []
    for k in range(4):
        rows += [(k, 16 if k == 0 else c[k - 1], c[k]), (k, c[k], c[k])]
    for k in (2, 1, 0):
        rows += [(k, c[k + 1] + c[k], c[k]), (k, c[k], c[k])]
    rows.append((0, c[0], c_pad))
    return rows   # (level, channels in, channels out)


def _net_params(case, seed):
    """He-normal weights in the library's order (per layer [tap][out][in], bias)."""
    rng = np.random.default_rng(seed)
    c_pad = (case["out"] + 15) // 16 * 16
    rows, parts = _layers(32, c_pad), []
    for i, (_, ci, co) in enumerate(rows):
        live_in, live_out = (4 if i == 0 else ci), (case["out"] if i + 1 == len(rows) else co)
        w = np.zeros((9, co, ci), dtype=np.float32)
        w[:, :live_out, :live_in] = rng.standard_normal((9, live_out, live_in)) * math.sqrt(2.0 / (9 * live_in))
        if i + 1 == len(rows):
            w *= 0.1
        parts += [w.reshape(-1), np.zeros(co, dtype=np.float32)]
    return np.concatenate(parts)


def _net_tensors(case, seed):
    """Packed inputs [batch, h, w, 16] (film with its mask inside a margin of
    six cells) and targets [batch, h, w, c_pad], bf16."""
    b, h, w, c_pad = case["batch"], case["h"], case["w"], (case["out"] + 15) // 16 * 16
    x = torch.zeros((b, h, w, 16), dtype=torch.bfloat16, device=DEV)
    t = torch.zeros((b, h, w, c_pad), dtype=torch.bfloat16, device=DEV)
    for i in range(b):
        x[i, 6:h - 6, 6:w - 6, :3] = _film(w - 12, h - 12, 1000003 * seed + i).permute(1, 2, 0).to(torch.bfloat16)
        x[i, 6:h - 6, 6:w - 6, 3] = 1.0
        z = torch.linspace(-2.0, 2.0, case["out"], device=DEV, dtype=torch.float64)
        film = _film(w, h, 1000003 * seed + 500 + i)[2]
        t[i, :, :, :case["out"]] = (0.3 * film[:, :, None] * torch.exp(-z * z)).to(torch.bfloat16)
    return x, t


# One context (or network) per grid is what a program keeps while its inputs
# change; only the last one is held here.
_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept.clear()
        _kept[key] = make()
    return _kept[key]


def _context(case):
    return L.Context(L.Grid2D(case["nx"], case["ny"], *CELLS[case["cell"]]), precision=L.F32 if case["f32"] else L.F64)


def _lib_material(mat, **kw):
    return L.Material(ms=mat["ms"], a_ex=mat["a_ex"], k_u=mat["k_u"], dmi=mat["dmi"] or None, demag=True, **kw)


def _first_dt(mat, cell, alpha, relax=False):
    """A first step size a little below the one the controller settles at: the
    exchange field of the shortest wave sets it."""
    b = 16.0 * mat["a_ex"] / (mat["ms"] * cell[0] ** 2)
    return 0.06 / (GAMMA * alpha * b) if relax else 0.4 / (GAMMA * b)


STEP = dict(mask=L.FieldMask.Full, max_err=1e-5, headroom=0.8, dt_min=1e-18, dt_max=1e-11)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("net", "train"):
        x, t = _net_tensors(case, seed)
        s = {"kind": kind, "x": x, "t": t}

        def make():
            return L.WarmStartNet(case["batch"], case["h"], case["w"], case["out"], 32, valid_width=case["w"] - 4,
                                  valid_height=case["h"] - 4)

        if kind == "net":
            # one network serves all inputs; its weights do not depend on the seed
            s["net"] = _keep(("net", case["batch"], case["h"], case["w"], case["out"]), make)
            s["net"].set_params(_net_params(case, 1))
            s["y"] = torch.empty((case["batch"], case["h"], case["w"], s["net"].c_pad), dtype=torch.float32,
                                 device=DEV)
        else:
            s["net"] = make()
            s["net"].set_params(_net_params(case, seed))
        return s
    ft = torch.float32 if case["f32"] else torch.float64
    if kind == "films":
        films = _specs(case["count"], case["set"])
        flat = torch.empty(sum(3 * f["nx"] * f["ny"] for f in films), dtype=ft, device=DEV)
        s, o = {"kind": kind, "flat": flat, "attempts": case["attempts"], "ctx": [], "m": [], "mat": [], "par": []}, 0
        for i, f in enumerate(films):
            n3 = 3 * f["nx"] * f["ny"]
            m = flat[o:o + n3].view(3, f["ny"], f["nx"])
            o += n3
            m.copy_(_film(f["nx"], f["ny"], 1000003 * seed + i))
            s["ctx"].append(L.Context(L.Grid2D(f["nx"], f["ny"], *f["cell"]),
                                      precision=L.F32 if case["f32"] else L.F64))
            s["m"].append(m)
            s["mat"].append(_lib_material(f["mat"]))
            s["par"].append(L.LLGParams(alpha=f["alpha"], b_ext=B_EXT,
                                        dt=_first_dt(f["mat"], f["cell"], f["alpha"])))
        torch.cuda.synchronize()
        out = torch.empty_like(flat)
        for c, m, mat, p in zip(s["ctx"], s["m"], s["mat"], s["par"]):   # the field of the initial states
            c.dev_build_h_eff(m, out, p, mat, L.FieldMask.Full)
            c.synchronize()
        return s
    m, geom = _inputs(case, seed)
    s = {"kind": kind, "mat": _lib_material(_material(case)),
         "par": L.LLGParams(alpha=_alpha(case), dt=_case_dt(case), b_ext=B_EXT)}
    key = (kind, case["nx"], case["ny"], case["cell"], case["f32"], case.get("default"))
    if kind == "host":
        s["ctx"] = _keep(key, lambda: _context(case))
        s["m"] = m.permute(1, 2, 0).contiguous().cpu().numpy().reshape(-1, 3)
        s["geom"] = None if geom is None else geom.cpu().numpy()
        return s
    s["m"] = m.to(ft).contiguous()
    s["geom"] = geom
    s["b"] = torch.empty_like(s["m"])
    if kind in ("field", "mg"):
        s["ctx"] = _keep(key, lambda: _context(case))
        if kind == "mg":
            s["mat"] = _lib_material(_material(case), demag_method=L.DemagMethod.PoissonMG)
            s["ctx"].set_mg_config(L.mg_config(warm_start=0) if case["default"] else
                                   L.mg_config(warm_start=0, stencil=0, prolong=0, coarse_op=0, smoother=1, bc=2,
                                               tol_rel=1e-8, v_cycles_max=300))
        return s
    # steppers: the context holds the state's slopes, so each state has its own
    s["ctx"] = _context(case)
    s["attempts"], s["steps"] = case.get("attempts"), case.get("steps")
    torch.cuda.synchronize()
    s["ctx"].dev_build_h_eff(s["m"], s["b"], s["par"], s["mat"], L.FieldMask.Full)   # the initial state's field
    s["ctx"].synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind in ("field", "mg"):
        s["ctx"].dev_build_h_eff(s["m"], s["b"], s["par"], s["mat"], L.FieldMask.Full, s["geom"])
        return s["b"]
    if kind == "host":
        return s["ctx"].build_h_eff_masked_geom(s["m"], s["par"], s["mat"], L.FieldMask.Full, s["geom"])
    # eps is left out of the steppers' outputs: in 32 bits it is a difference
    # of slopes that nearly cancel, and the next step size carries it
    if kind == "rk45":
        if s["attempts"]:
            rows = s["ctx"].dev_rk45_run(s["m"], s["par"], s["mat"], attempts=s["attempts"], **STEP)
        else:
            rows = [s["ctx"].dev_rk45_step(s["m"], s["par"], s["mat"], **STEP)]
        return {"m": s["m"], "accepted": np.array([int(a) for _, a, _ in rows]),
                "dt": np.array([u for _, _, u in rows] + [s["par"].dt])}
    if kind == "films":
        rows = L.dev_rk45_run_batch(s["ctx"], s["m"], s["par"], s["mat"], s["attempts"], **STEP)
        return {"m": s["flat"], "accepted": np.array([[int(a) for _, a, _ in r] for r in rows]),
                "dt": np.array([[u for _, _, u in r] for r in rows] + [[p.dt for p in s["par"]]])}
    if kind == "relax":
        rows = [s["ctx"].dev_rk23_relax_step(s["m"], s["par"], s["mat"], **STEP) for _ in range(s["steps"])]
        e = s["ctx"].dev_compute_energy_geom(s["m"], s["mat"], B_EXT)
        return {"m": s["m"], "accepted": np.array([int(a) for _, a, _ in rows]),
                "dt": np.array([u for _, _, u in rows] + [s["par"].dt]), "energy": np.array([e[k] for k in ENERGY])}
    if kind == "net":
        s["net"].forward(s["x"], s["y"])
        return s["y"]
    loss = s["net"].train_step(s["x"], s["t"], 5e-4)
    return {"loss": loss, "grads": s["net"].get_grads()}


ENERGY = ("exchange", "anisotropy", "zeeman", "dmi", "demag")


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def _eval_work(nx, ny, size):
    """Bytes and operations of one FFT field evaluation: m in, B out, the four
    real kernel planes; three real 2D transforms each way on 2nx x 2ny."""
    n = nx * ny
    rows = 3 * ny * 2.5 * 2 * nx * math.log2(2 * nx)
    cols = 3 * nx * 5.0 * 2 * ny * math.log2(2 * ny)
    return size * (6 * n + 4 * (nx + 1) * (ny + 1)), 2 * (rows + cols) + 20 * 2 * n + 120 * n


def work(case):
    kind = case["kind"]
    if kind in ("net", "train"):
        c_pad = (case["out"] + 15) // 16 * 16
        rows = _layers(32, c_pad)
        px = case["batch"] * case["h"] * case["w"]
        flops = sum(18.0 * ci * co * (px >> (2 * k)) for k, ci, co in rows)
        par = sum(9 * ci * co + co for _, ci, co in rows)
        if kind == "net":
            return {"bytes": px * (32 + 4 * c_pad) + 4 * par, "flops": flops}
        # weights and moments in and out, gradients out
        return {"bytes": px * (32 + 2 * c_pad) + 4 * par * 7, "flops": 3 * flops}
    size = 4 if case["f32"] else 8
    if kind == "films":
        b = f = 0.0
        for s in _specs(case["count"], case["set"]):
            eb, ef = _eval_work(s["nx"], s["ny"], size)
            n = s["nx"] * s["ny"]
            b += case["attempts"] * (6 * eb + 38 * n * size)
            f += case["attempts"] * (6 * ef + 200 * n)
        return {"bytes": b, "flops": f}
    n = case["nx"] * case["ny"]
    if kind == "mg":
        box = (case["nx"] + 12) * (case["ny"] + 12) * (36 if not case["default"] else 34)
        # the potential and its right side, each read and written once; about
        # ten V(2,2) cycles of the stencil
        return {"bytes": 6 * n * 8 + 3 * box * 8, "flops": 10 * 5 * (14 if not case["default"] else 54) * box}
    eb, ef = _eval_work(case["nx"], case["ny"], size)
    if case.get("holes"):
        eb += n
    if kind == "field":
        return {"bytes": eb, "flops": ef}
    if kind == "host":
        return {"bytes": eb + 48 * n, "flops": ef}
    if kind == "rk45":
        k = max(case["attempts"], 1)
        # six evaluations; the slopes read by the stages and the error norm
        return {"bytes": k * (6 * eb + 38 * n * size), "flops": k * (6 * ef + 200 * n)}
    k = case["steps"]
    return {"bytes": (3 * k + 1) * eb + k * 20 * n * size, "flops": (3 * k + 1) * ef + k * 100 * n}


def tolerance(case):
    """About four times what another order of the sums shows (radix-8 against
    radix-16 transforms, another tiling of the convolutions)."""
    kind = case["kind"]
    if kind == "net":
        # bf16 activations: single roundings that fall the other way travel
        # through fifteen layers
        return {"rel": 1.5e-2, "max": 0.15}
    if kind == "train":
        # as above; after a step, weights whose gradient is rounding noise
        # have moved the other way too
        return {"rel": 1e-2, "max": 0.5}
    if kind == "mg":
        # the same iteration in 64 bits
        return {"rel": 1e-10, "max": 1e-7}
    if kind in ("field", "host"):
        return {"rel": 1e-6, "max": 1e-5} if case["f32"] else {"rel": 1e-14, "max": 1e-12}
    if kind == "films" or case["f32"]:
        # the step size follows an error estimate that 32-bit slopes give to
        # about four digits
        return {"rel": 5e-4, "max": 2e-3}
    return {"rel": 1e-6, "max": 1e-5}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _kernel_quadrant(nx, ny, cell):
    """mu0 H at displacement (sx, sy) >= 0 of a unit-magnetised cell's faces,
    averaged over the target cell by the MuMax-like point rule: [4, ny, nx]
    (xx, xy, yy, zz)."""
    f64 = dict(dtype=torch.float64, device=DEV)
    sx, sy = torch.arange(nx, **f64), torch.arange(ny, **f64)
    d = torch.sqrt(((sx - 1).clamp(min=0) * cell[0])[None, :].square() +
                   ((sy - 1).clamp(min=0) * cell[1])[:, None].square())
    d = torch.where(d == 0, torch.full_like(d, min(cell)), d).reshape(-1)
    rc = torch.stack([(sx * cell[0])[None, :].expand(ny, nx).reshape(-1),
                      (sy * cell[1])[:, None].expand(ny, nx).reshape(-1), torch.zeros(nx * ny, **f64)], 1)
    count = [torch.floor((c / (d / 10.0)).clamp(min=1) + 0.5).long() for c in cell]
    key = (count[0] * 4096 + count[1]) * 4096 + count[2]
    out = torch.zeros((4, nx * ny), **f64)

    def centres(length, k):
        return (torch.arange(k, **f64) + 0.5) * (length / k) - 0.5 * length

    for value in torch.unique(key).tolist():
        at = (key == value).nonzero().reshape(-1)
        k = [value >> 24, (value >> 12) & 4095, value & 4095]
        inner = torch.stack(torch.meshgrid(*(centres(cell[q], k[q]) for q in range(3)), indexing="ij"), -1)
        inner = inner.reshape(-1, 3)
        for u in range(3):
            v, w = (u + 1) % 3, (u + 2) % 3
            pv, pw = centres(cell[v], 2 * k[v]), centres(cell[w], 2 * k[w])
            charge = cell[v] * cell[w] / (pv.numel() * pw.numel() * inner.shape[0])
            h = torch.zeros((at.numel(), 3), **f64)
            for sign in (1.0, -1.0):
                pole = torch.zeros((pv.numel(), pw.numel(), 3), **f64)
                pole[:, :, u] = sign * 0.5 * cell[u]
                pole[:, :, v], pole[:, :, w] = pv[:, None], pw[None, :]
                pole = pole.reshape(-1, 3)
                step = max(1, (1 << 23) // max(1, inner.shape[0] * min(at.numel(), 1 << 16)))
                for a0 in range(0, at.numel(), 1 << 16):
                    part = rc[at[a0:a0 + (1 << 16)]]
                    for p0 in range(0, pole.shape[0], step):
                        off = (inner[None, :, :] - pole[p0:p0 + step, None, :]).reshape(1, -1, 3)
                        r = part[:, None, :] + off
                        q = sign * charge / (4.0 * math.pi) / (r.square().sum(-1).sqrt() ** 3)
                        h[a0:a0 + (1 << 16)] += (r * q[:, :, None]).sum(1)
            if u == 0:
                out[0, at] = MU0 * h[:, 0]
            elif u == 1:
                out[1, at], out[2, at] = MU0 * h[:, 0], MU0 * h[:, 1]
            else:
                out[3, at] = MU0 * h[:, 2]
    return out.reshape(4, ny, nx)


class _Film:
    """The effective field of one film in 64 bits."""

    def __init__(self, nx, ny, cell, mat, alpha, geom=None):
        self.nx, self.ny, self.cell, self.mat, self.alpha = nx, ny, cell, mat, alpha
        self.geom = None if geom is None else geom.bool()
        quad = _kernel_quadrant(nx, ny, cell)
        full = torch.zeros((4, 2 * ny, 2 * nx), dtype=torch.float64, device=DEV)
        full[:, :ny, :nx] = quad
        full[1, 0, :], full[1, :, 0] = 0.0, 0.0
        sign = torch.tensor([1.0, -1.0, 1.0, 1.0], dtype=torch.float64, device=DEV)[:, None, None]
        if nx > 1:
            full[:, :ny, nx + 1:] = sign * full[:, :ny, 1:nx].flip(2)
        if ny > 1:
            full[:, ny + 1:, :] = sign * full[:, 1:ny, :].flip(1)
        self.k = torch.fft.rfft2(full).real

    def demag(self, m):
        f = torch.fft.rfft2(self.mat["ms"] * m, s=(2 * self.ny, 2 * self.nx))
        k = self.k
        b = torch.stack([k[0] * f[0] + k[1] * f[1], k[1] * f[0] + k[2] * f[1], k[3] * f[2]])
        return torch.fft.irfft2(b, s=(2 * self.ny, 2 * self.nx))[:, :self.ny, :self.nx]

    def _neighbour(self, m, axis, step):
        """Neighbour along x (axis 0) or y (axis 1), whether it exists and is
        material, whether it is outside the domain, and the chiral ghost."""
        dim = 2 if axis == 0 else 1
        size = m.shape[dim]
        v = m.roll(-step, dim)
        edge = torch.zeros(m.shape[1:], dtype=torch.bool, device=DEV)
        edge.select(1 - axis, size - 1 if step > 0 else 0).fill_(True)
        ok = ~edge if self.geom is None else ~edge & self.geom.roll(-step, dim - 1)
        eta = self.mat["dmi"] / (2.0 * self.mat["a_ex"])
        ghost = m.clone()
        ghost[axis] = m[axis] - step * self.cell[axis] * eta * m[2]
        ghost[2] = m[2] + step * self.cell[axis] * eta * m[axis]
        return v, ok, edge, ghost

    def field(self, m):
        mat, cell = self.mat, self.cell
        b = torch.zeros_like(m)
        lap, grad = torch.zeros_like(m), []
        for axis in (0, 1):
            pair = []
            for step in (-1, 1):
                v, ok, edge, ghost = self._neighbour(m, axis, step)
                lap += (torch.where(ok, v, ghost) - m) / cell[axis] ** 2
                pair.append(torch.where(edge, ghost, torch.where(ok, v, m)))
            grad.append((pair[1] - pair[0]) / (2.0 * cell[axis]))
        b += 2.0 * mat["a_ex"] / mat["ms"] * lap
        d = 2.0 * mat["dmi"] / mat["ms"]
        b[0] += d * grad[0][2]
        b[1] += d * grad[1][2]
        b[2] -= d * (grad[0][0] + grad[1][1])
        if self.geom is not None:
            b *= self.geom
        b[2] += 2.0 * mat["k_u"] / mat["ms"] * m[2]
        b += torch.tensor(B_EXT, dtype=torch.float64, device=DEV)[:, None, None]
        return b + self.demag(m)

    def slope(self, m, relax=False):
        c = torch.linalg.cross(m, self.field(m), dim=0)
        cc = torch.linalg.cross(m, c, dim=0)
        a = self.alpha
        return -GAMMA / (1.0 + a * a) * (a * cc if relax else c + a * cc)

    def energy(self, m):
        mat, cell = self.mat, self.cell
        vol = cell[0] * cell[1] * cell[2]
        ex = sum((m.narrow(2 - axis, 1, m.shape[2 - axis] - 1) - m.narrow(2 - axis, 0, m.shape[2 - axis] - 1))
                 .square().sum() / cell[axis] ** 2 for axis in (0, 1)) * mat["a_ex"] * vol
        an = mat["k_u"] * vol * (1.0 - m[2].square()).sum()
        ze = -mat["ms"] * vol * sum((m[q] * B_EXT[q]).sum() for q in range(3))
        grad = []
        for axis in (0, 1):
            ends = [torch.where(edge, ghost, v) for v, _, edge, ghost in
                    (self._neighbour(m, axis, step) for step in (-1, 1))]
            grad.append((ends[1] - ends[0]) / (2.0 * cell[axis]))
        d = 2.0 * mat["dmi"] / mat["ms"]
        dm = -0.5 * mat["ms"] * vol * d * (m[0] * grad[0][2] + m[1] * grad[1][2] -
                                           m[2] * (grad[0][0] + grad[1][1])).sum()
        de = -0.5 * mat["ms"] * vol * (m * self.demag(m)).sum()
        return torch.stack([torch.as_tensor(v, dtype=torch.float64, device=DEV) for v in (ex, an, ze, dm, de)])


def _unit(v):
    return v / v.square().sum(0, keepdim=True).sqrt()


_A = [[], [1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
      [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
      [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
      [35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
_BH = [5179 / 57600, 0.0, 7571 / 16695, 393 / 640, -92097 / 339200, 187 / 2100, 1 / 40]


def _next_dt(dt, eps, order):
    new = dt * STEP["headroom"] * (STEP["max_err"] / eps) ** (1.0 / order) if eps > 0 else 2.0 * dt
    return min(max(new, STEP["dt_min"]), STEP["dt_max"]), eps <= STEP["max_err"] or dt <= STEP["dt_min"]


def _dormand_prince(film, m, dt, attempts):
    used, accepted = [], []
    for _ in range(attempts):
        k = [film.slope(m)]
        for row in _A[1:]:
            v = _unit(m + dt * sum(a * kk for a, kk in zip(row, k)))
            k.append(film.slope(v))
        err = sum((b - bh) * kk for b, bh, kk in zip(_A[6] + [0.0], _BH, k))
        new, ok = _next_dt(dt, float(err.abs().max()) * dt, 5)
        used.append(dt)
        accepted.append(int(ok))
        m, dt = (v if ok else m), new
    return m, accepted, used, dt


def _bogacki_shampine(film, m, dt, attempts):
    used, accepted = [], []
    for _ in range(attempts):
        k1 = film.slope(m, True)
        k2 = film.slope(_unit(m + dt * 0.5 * k1), True)
        k3 = film.slope(_unit(m + dt * 0.75 * k2), True)
        new_m = _unit(m + dt * (2 / 9 * k1 + 1 / 3 * k2 + 4 / 9 * k3))
        k4 = film.slope(new_m, True)
        low = _unit(m + dt * (7 / 24 * k1 + 1 / 4 * k2 + 1 / 3 * k3 + 1 / 8 * k4))
        new, ok = _next_dt(dt, float((new_m - low).abs().max()), 3)
        used.append(dt)
        accepted.append(int(ok))
        m, dt = (new_m if ok else m), new
    return m, accepted, used, dt


class _Conv3(torch.autograd.Function):
    """3x3 convolution, channels last, weights [tap][out][in], zero border."""

    @staticmethod
    def _shift(x, tap):
        dy, dx = tap // 3 - 1, tap % 3 - 1
        p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
        h, w = x.shape[1:3]
        return p[:, 1 + dy:1 + dy + h, 1 + dx:1 + dx + w].reshape(-1, x.shape[3])

    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        y = b.expand(x.shape[0] * x.shape[1] * x.shape[2], -1).clone()
        for tap in range(9):
            y += _Conv3._shift(x, tap) @ w[tap].t().contiguous()
        return y.reshape(*x.shape[:3], -1)

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        flat = g.reshape(-1, g.shape[3])
        gx = torch.zeros(flat.shape[0], x.shape[3], dtype=g.dtype, device=g.device)
        gw = torch.empty_like(w)
        for tap in range(9):
            gx += _Conv3._shift(g, 8 - tap) @ w[tap]
            gw[tap] = flat.t().contiguous() @ _Conv3._shift(x, tap)
        return gx.reshape(x.shape), gw, flat.sum(0)


def _unet(case, flat, x):
    c_pad = (case["out"] + 15) // 16 * 16
    rows, o, par = _layers(32, c_pad), 0, []
    for _, ci, co in rows:
        w = flat[o:o + 9 * ci * co].view(9, co, ci)
        o += 9 * ci * co
        par.append((w, flat[o:o + co]))
        o += co

    def conv(i, v, relu=True):
        y = _Conv3.apply(v, *par[i])
        return torch.relu(y) if relu else y

    skips = []
    for k in range(4):
        if k:
            b, h, w, c = x.shape
            x = x.reshape(b, h // 2, 2, w // 2, 2, c).mean((2, 4))
        x = conv(2 * k + 1, conv(2 * k, x))
        skips.append(x)
    for i, k in enumerate((2, 1, 0)):
        up = x.repeat_interleave(2, 1).repeat_interleave(2, 2)
        x = conv(9 + 2 * i, conv(8 + 2 * i, torch.cat([up, skips[k]], 3)))
    return conv(14, x, False)


def exact(case, seed):
    kind = case["kind"]
    if kind == "mg":
        # the result is the iterate that meets the tolerance, with boundary
        # values of a tree code: the value is defined by the iteration itself
        return None
    if kind in ("net", "train"):
        x, t = _net_tensors(case, seed)
        flat = torch.tensor(_net_params(case, 1 if kind == "net" else seed), device=DEV).double()
        if kind == "net":
            with torch.no_grad():
                return _unet(case, flat, x.double())
        flat.requires_grad_(True)
        d = (_unet(case, flat, x.double()) - t.double())[:, :case["h"] - 4, :case["w"] - 4, :case["out"]]
        loss = d.square().mean()
        loss.backward()
        return {"loss": float(loss), "grads": flat.grad.cpu().numpy()}
    if kind == "films":
        flat, acc, used, last = [], [], [], []
        for i, f in enumerate(_specs(case["count"], case["set"])):
            film = _Film(f["nx"], f["ny"], f["cell"], f["mat"], f["alpha"])
            m = _film(f["nx"], f["ny"], 1000003 * seed + i)
            m, a, u, dt = _dormand_prince(film, m, _first_dt(f["mat"], f["cell"], f["alpha"]), case["attempts"])
            flat.append(m.reshape(-1))
            acc.append(a)
            used.append(u)
            last.append(dt)
        return {"m": torch.cat(flat), "accepted": np.array(acc).T.copy(),
                "dt": np.concatenate([np.array(used).T, np.array(last)[None, :]])}
    m, geom = _inputs(case, seed)
    film = _Film(case["nx"], case["ny"], CELLS[case["cell"]], _material(case), _alpha(case), geom)
    if kind in ("field", "host"):
        b = film.field(m)
        return b if kind == "field" else b.permute(1, 2, 0).reshape(-1, 3).cpu().numpy()
    dt = _case_dt(case)
    if kind == "rk45":
        m, a, u, dt = _dormand_prince(film, m, dt, max(case["attempts"], 1))
        return {"m": m, "accepted": np.array(a), "dt": np.array(u + [dt])}
    m, a, u, dt = _bogacki_shampine(film, m, dt, case["steps"])
    return {"m": m, "accepted": np.array(a), "dt": np.array(u + [dt]), "energy": film.energy(m).cpu().numpy()}
