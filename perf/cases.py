"""Workloads of the epi5_MT hot path through its Python entry points.

Every case is a call (or a few) that a program using ``epi_amd`` makes, over
tissues of the seeded generator (``epi_amd.configs``) with the library's own
launch shapes:

  step          a stretch of the driver's loop (``TissueSet.step``) and the
                output record that the reference writes after it
                (``snapshot_begin`` / ``snapshot_wait``); with ``ca_every`` the
                stretch ends on a forced calc_ca2p
  solve         one calc_ca2p of frozen tissues and the output record
  rd_forward    a frozen reaction-diffusion window, forward
  rd_adjoint    its loss and gradients, checkpointed
  mech_forward  a frozen mechanics window, forward
  mech_adjoint  its loss and gradients, checkpointed
  b_sweep       calc_ext_stim over grids the caller holds on the device

``listed()`` are the cases that stand for the range, ``draw()`` gives others
of the same ranges, ``exact()`` what a case computes, in plain 64-bit torch.
"""
import ctypes as C
import math

import numpy as np
import torch

from epi_amd import configs, native
from epi_amd.configs import ALIVE, DEAD, FIX, MEMB, MUSUME

STEPS_KEPT = 14000   # steps that a tissue's random stream lasts
MARGIN = 12.0   # free height above the top layer: a tissue drifts upward over thousands of steps


def listed():
    return [
        # a unit-test tissue (about 420 cells): nothing but launches and their latency
        dict(name="step_tiny", kind="step", tissues=1, side=16, free=160, layers=2, grid=16, nz=32, dz=0.875,
             fix=4, dead=False, steps=100, ca_every=0),
        # ragged sizes: an odd grid with dz != dx, layers that are not full, a DEAD top layer that is shed
        dict(name="step_odd", kind="step", tissues=1, side=50, free=1777, layers=5, grid=37, nz=41, dz=0.93,
             fix=16, dead=True, steps=100, ca_every=100),
        # the small parity tissue (64x64 sheet, 2,000 free cells, about 6,100 in all), as one researcher runs it
        dict(name="step_small", kind="step", tissues=1, side=64, free=2000, layers=4, grid=64, nz=64, dz=0.8125,
             fix=16, dead=False, steps=100, ca_every=0),
        # the large parity tissue (128x128 sheet, 20,000 free cells, grid 128x128x256), a solve every 50 steps
        # (about what its own cornifications trigger)
        dict(name="step_large", kind="step", tissues=1, side=128, free=20000, layers=8, grid=128, nz=256, dz=0.8125,
             fix=64, dead=True, steps=50, ca_every=50),
        # a parameter study: 32 independent tissues of uneven sheets, cell counts and grids in one context
        dict(name="step_batch", kind="step", tissues=32, side=0, free=0, layers=2, grid=0, nz=0, dz=0.0,
             fix=16, dead=False, steps=50, ca_every=50),
        # one calc_ca2p of a small ragged tissue (what a gated solve of one tissue costs) ...
        dict(name="solve_odd", kind="solve", tissues=1, side=30, free=701, layers=5, grid=33, nz=45, dz=0.71,
             fix=16, dead=True),
        # ... and of the large one
        dict(name="solve_large", kind="solve", tissues=1, side=128, free=20000, layers=8, grid=128, nz=256, dz=0.8125,
             fix=64, dead=True),
        # fitting Ca2+ parameters: 5,000 free cells on a 64x64x128 grid, 200 sub-steps, and its gradient
        dict(name="rd_forward", kind="rd_forward", tissues=1, side=64, free=5000, layers=8, grid=64, nz=128, dz=0.8125,
             fix=16, dead=False, n_sub=200),
        dict(name="rd_adjoint", kind="rd_adjoint", tissues=1, side=64, free=5000, layers=8, grid=64, nz=128, dz=0.8125,
             fix=16, dead=False, n_sub=200, every=20),
        # fitting mechanics parameters: tissues of 2,000 to 6,000 cells in one context, 100 steps, and the gradient
        dict(name="mech_forward", kind="mech_forward", tissues=1, side=40, free=2300, layers=2, grid=48, nz=48, dz=1.4,
             fix=16, dead=False, n_steps=100),
        dict(name="mech_adjoint", kind="mech_adjoint", tissues=24, side=40, free=0, layers=2, grid=48, nz=48, dz=1.4,
             fix=16, dead=False, n_steps=100, every=10),
        # the B stencil alone over a caller's grids, uneven and up to the largest the tissues use
        dict(name="b_sweep", kind="b_sweep", grids=12, edge=96, depth=192),
    ]


def draw(rng):
    kind = rng.choice(["step", "step", "step", "solve", "rd_forward", "rd_adjoint", "mech_forward", "mech_adjoint",
                       "b_sweep"])
    log_int = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
    if kind == "b_sweep":
        return dict(kind=kind, grids=log_int(1, 12), edge=log_int(17, 96), depth=log_int(24, 192))
    side = 2 * log_int(8, 48 if kind in ("step", "solve") else 32)
    box = _box(side)
    sites = int(box / 2.0) ** 2
    fix = 4 if side < 24 else 16
    dead = rng.random() < 0.5 and kind in ("step", "solve")
    layers = rng.randint(3 if dead else 2, 6)
    free = int(sites * layers * rng.uniform(0.55, 0.95)) - fix
    grid = max(13, int(box / rng.uniform(0.6, 1.1)))
    dz = round(rng.uniform(0.6, 1.1), 3)
    nz = int((_top(layers, dead) + MARGIN) / dz) + rng.randint(1, 9)
    c = dict(kind=kind, tissues=1, side=side, free=free, layers=layers, grid=grid, nz=nz, dz=dz, fix=fix, dead=dead)
    if kind == "step":
        c["steps"] = rng.randint(20, 100)
        c["ca_every"] = rng.choice([0, 0, c["steps"]])
    elif kind.startswith("rd_"):
        c["n_sub"] = log_int(20, 200)
    elif kind.startswith("mech_"):
        c["n_steps"] = log_int(10, 100)
    if kind.endswith("_adjoint"):
        c["every"] = rng.randint(4, 20)
    return c


# ---- tissues ---------------------------------------------------------------
def _box(side):
    """the sheet's extent: every x stays below the last bucket (configs.batched_configs)"""
    return 2.0 * math.ceil(0.4 * side)


def _top(layers, dead):
    """height of the top layer's centres (configs.make_tissue), and what iz_bound adds"""
    return 2 * configs.R_MEMB + configs.R_MAX + 2.2 * (layers - 1) + (0.7 if dead else 0.0) + 2.8


def _sizes(case):
    """per tissue: side, free cells, layers, grid edge, nz, dz"""
    if case["tissues"] == 1:
        return [(case["side"], case["free"], case["layers"], case["grid"], case["nz"], case["dz"])]
    out = []
    for t in range(case["tissues"]):
        r = np.random.default_rng(3000 + t)
        if case["kind"] == "step":      # sheets of 32 to 96, 500 to 8,000 free cells, grid edges of 32 to 96
            side = int(r.integers(16, 49)) * 2
            box, edge = _box(side), int(r.integers(32, 97))
            free = int(r.integers(500, 8001))
            nz, dz = 2 * edge, box / edge
            cap = configs.batched_capacity(int(box / 2.0), nz * dz, dz, case["fix"])
            out.append((side, max(64, min(free, cap)), case["layers"], edge, nz, dz))
        else:                           # 2,000 to 6,000 cells on a 40x40 sheet
            free = int(r.integers(2000, 6001)) - 40 * 40 - case["fix"]
            out.append((case["side"], free, case["layers"], case["grid"], case["nz"], case["dz"]))
    return out


def _specs(case, seed):
    out = []
    for t, (side, free, layers, grid, nz, dz) in enumerate(_sizes(case)):
        box = _box(side)
        hot = 30 if case["kind"] == "step" and case["tissues"] == 1 else 8
        out.append(configs.make_tissue(seed * 64 + t, nmx=side, nmy=side, lx=box, ly=box, nx=grid, ny=grid, nz=nz,
                                       n_fix=case["fix"], n_free=free, n_layers=layers, dead_top=case["dead"],
                                       n_hot_alive=hot, lz=nz * dz))
    return out


def _draws(spec, seed, t, tissues):
    """a replay stream for thousands of steps: a division-ready cell takes one draw a step"""
    st = spec["cells"]["state"]
    ready = int(np.count_nonzero((st == FIX) | (st == MUSUME)))
    return native.mt19937_64_uniform(seed * 64 + t, min(STEPS_KEPT * (ready + 32), 16_000_000 // tissues))


def _kpa(spec):
    """per-cell IP3 production (calc_Kpa, ca2p.cpp:101-110)"""
    c = spec["cells"]
    return np.where(c["state"] == ALIVE, 4.0 + (6.0 - 4.0) * 0.5 * (1.0 + np.tanh(3.0 - c["agek"])), 6.0)


def _rd_params(spec, seed):
    """the window's parameters, and those of its target: perturbed by 5 %"""
    kpa = _kpa(spec)
    sign = np.random.default_rng(seed).choice([-1.0, 1.0], kpa.size)
    return (dict(du=0.01, dp=0.1, gj0=0.99, kpa=kpa),
            dict(du=0.01 * 1.05, dp=0.1 * 0.95, gj0=0.99 * 0.95, kpa=kpa * (1 + 0.05 * sign)))


MECH = dict(eps=0.01, k_adh=3.0, k_spring=25.0, k_bend=0.5)
MECH_TARGET = dict(eps=0.0105, k_adh=2.85, k_spring=26.25, k_bend=0.475)


def _crumple(specs, seed):
    """a curved sheet, so that bending takes part"""
    for t, s in enumerate(specs):
        c, m = s["cells"], s["nmemb"]
        c["z"][:m] += np.random.default_rng(seed * 64 + t).uniform(-0.05, 0.05, m)
    return specs


# ---- the cases' entry points -----------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "b_sweep":
        return _prepare_b(case, seed)
    specs = _specs(case, seed)
    if kind.startswith("mech_"):
        specs = _crumple(specs, seed)
    ts = native.TissueSet([s["geometry"] for s in specs])
    for t, s in enumerate(specs):
        ts.load(t, s)
    state = {"case": case, "ts": ts}
    if kind == "step":
        for t, s in enumerate(specs):
            ts.set_rng(t, _draws(s, seed, t, case["tissues"] // 4 + 1))
        state["drivers"] = [native.Driver(0, 0, 0, case["ca_every"], 0) for _ in specs]
        return state
    if kind.startswith("mech_"):
        ts.mech_begin()
        state["params"] = [MECH] * len(specs)
        if kind == "mech_adjoint":
            ts.mech_forward([MECH_TARGET] * len(specs), case["n_steps"])
            state["targets"] = [ts.mech_get_positions(t) for t in range(len(specs))]
        return state
    ts.setup_map_lat()
    state["zz"] = ts.calc_zzmax()
    if kind.startswith("rd_"):
        pairs = [_rd_params(s, seed + t) for t, s in enumerate(specs)]
        state["params"] = [p for p, _ in pairs]
        ts.rd_begin(state["zz"])
        if kind == "rd_adjoint":
            ts.rd_forward([q for _, q in pairs], case["n_sub"])
            state["targets"] = [ts.rd_get_ca2p(t) for t in range(len(specs))]
    return state


def _record(ts):
    """the output record of every tissue, one download beside the next one's packing, in columns of the tissues'
    capacities (cells come and go)"""
    ts.snapshot_begin(0, 0)
    parts = []
    for t in range(ts.T):
        if t + 1 < ts.T:
            ts.snapshot_begin(t + 1, (t + 1) % 2)
        parts.append(ts.snapshot_wait(t % 2))
    out = {"n": np.array([p["n"] for p in parts])}
    for k in parts[0]:
        if k not in ("tissue", "n"):
            out[k] = np.zeros(sum(g.max_cells for g in ts.geos), parts[0][k].dtype)
            at = 0
            for p, g in zip(parts, ts.geos):
                out[k][at:at + p["n"]] = p[k]
                at += g.max_cells
    return out


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "b_sweep":
        rc = state["lib"].epi_calc_ext_stim_noalloc(C.c_void_p(state["views"].data_ptr()), case["grids"],
                                                    C.c_void_p(state["err"].data_ptr()),
                                                    C.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(f"epi_calc_ext_stim_noalloc: {rc}")
        return {"b": state["b_out"], "err": state["err"]}
    ts = state["ts"]
    if kind == "step":
        ts.step(state["drivers"], case["steps"])
        return _record(ts)
    if kind == "solve":
        ts.calc_ca2p(state["zz"])
        return _record(ts)
    if kind == "rd_forward":
        ts.rd_forward(state["params"], case["n_sub"])
        return [ts.rd_get_ca2p(t) for t in range(ts.T)]
    if kind == "rd_adjoint":
        loss, g = ts.rd_adjoint(state["params"], case["n_sub"], case["every"], state["targets"])
        return {"loss": loss, "grads": g}
    if kind == "mech_forward":
        ts.mech_forward(state["params"], case["n_steps"])
        return [ts.mech_get_positions(t) for t in range(ts.T)]
    loss, g = ts.mech_adjoint(state["params"], case["n_steps"], case["every"], state["targets"])
    return {"loss": loss, "grads": np.array([[q[k] for k in MECH] for q in g])}


# ---- the B stencil's grids ---------------------------------------------------
class _View(C.Structure):   # epi_bfield_view (include/epi_amd.h)
    _fields_ = [("nx", C.c_int32), ("ny", C.c_int32), ("nz", C.c_int32), ("xp", C.c_int32), ("pl", C.c_int64),
                ("lz", C.c_double), ("zzmax", C.c_double), ("b_in", C.c_void_p), ("b_out", C.c_void_p),
                ("cmap1", C.c_void_p), ("cmap2", C.c_void_p), ("state", C.c_void_p), ("agek", C.c_void_p)]


def _b_shapes(case):
    """(nx, ny, nz, xp, iz_bound) per grid, dx = dz = 0.8; the first is the largest"""
    r = np.random.default_rng(case["edge"] * 1000 + case["depth"])
    out = []
    for i in range(case["grids"]):
        e = case["edge"] if i == 0 else int(r.integers(16, case["edge"] + 1))
        d = case["depth"] if i == 0 else int(r.integers(20, case["depth"] + 1))
        nx, ny = e, max(8, e - int(r.integers(0, 4)))
        out.append((nx, ny, d, (nx + 16) // 16 * 16, int(d * 0.72)))
    return out


def _b_inputs(case, seed):
    """per grid, on the host: B, the cell of each voxel (blobs of a few voxels, half the tissue's volume), the
    AFM mask (1 inside the tissue but for a few holes) and the cells' states and ages"""
    out = []
    for i, (nx, ny, nz, xp, izb) in enumerate(_b_shapes(case)):
        g = torch.Generator().manual_seed(seed * 64 + i)
        shape = (nz + 1, ny + 1, xp)   # z, y, x
        b = torch.rand(shape, generator=g, dtype=torch.float64) * 0.02 + 0.09
        cz, cy, cx = (nz + 4) // 4, (ny + 4) // 4, (xp + 3) // 4
        n = cz * cy * cx
        blob = torch.arange(n, dtype=torch.int32)
        blob[torch.rand(n, generator=g) < 0.5] = -1
        cmap1 = blob.view(cz, cy, cx).repeat_interleave(4, 0).repeat_interleave(4, 1).repeat_interleave(4, 2)
        cmap1 = cmap1[:nz + 1, :ny + 1, :xp].clone()
        hole = torch.rand((cz, cy, cx), generator=g) < 0.1
        cmap2 = (~hole).to(torch.uint8).repeat_interleave(4, 0).repeat_interleave(4, 1).repeat_interleave(4, 2)
        cmap2 = cmap2[:nz + 1, :ny + 1, :xp].clone()
        top = izb - 3
        cmap1[top:], cmap2[top:] = -1, 0
        for a in (b, cmap1, cmap2):   # planes x = nx and y = ny are the periodic copies
            a[:, ny, :] = a[:, 0, :]
            a[:, :, nx] = a[:, :, 0]
        kinds = torch.tensor([ALIVE, ALIVE, ALIVE, DEAD, MUSUME, FIX, MEMB], dtype=torch.uint8)
        state = kinds[torch.randint(0, len(kinds), (n,), generator=g)]
        agek = torch.rand(n, generator=g, dtype=torch.float64) * 6.0 + 19.0
        out.append((b, cmap1, cmap2, state, agek))
    return out


def _prepare_b(case, seed):
    lib = native.load_library()
    shapes, views, keep, b_out = _b_shapes(case), (_View * case["grids"])(), [], []
    for v, (nx, ny, nz, xp, izb), host in zip(views, shapes, _b_inputs(case, seed)):
        dev = [a.cuda() for a in host]
        out = torch.zeros_like(dev[0])
        v.nx, v.ny, v.nz, v.xp, v.pl = nx, ny, nz, xp, xp * (ny + 1)
        v.lz, v.zzmax = nz * 0.8, (izb + 0.5) * 0.8 - 2.8
        v.b_in, v.b_out = dev[0].data_ptr(), out.data_ptr()
        v.cmap1, v.cmap2, v.state, v.agek = (a.data_ptr() for a in dev[1:])
        keep.append(dev)
        b_out.append(out)
    d_views = torch.frombuffer(bytearray(bytes(views)), dtype=torch.uint8).cuda()
    err = torch.full((case["grids"],), -1, dtype=torch.int32, device="cuda")
    return {"case": case, "lib": lib, "views": d_views, "err": err, "b_out": b_out, "keep": keep}


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    """Bytes: each cell's words, its list and the active grid points read and written once per step or sub-step
    (a step: 120 + 8 k per cell with k list entries, maps 5 and B 21 per point; a sub-step: 96 + 28 k per AFM cell
    with k coupled entries, ATP 22 per point; a reverse step twice a forward one).  Operations: about 60 per list
    entry and law, 30 per grid point."""
    if case["kind"] == "b_sweep":
        pts = sum(nx * ny * izb for nx, ny, nz, xp, izb in _b_shapes(case))
        return {"bytes": 21.0 * pts, "flops": 30.0 * pts}
    by = fl = 0.0
    for side, free, layers, grid, nz, dz in _sizes(case):
        n = side * side + case["fix"] + free
        need = max(layers, math.ceil((free + case["fix"]) / int(_box(side) / 2.0) ** 2))
        pts = grid * grid * min(nz, int(_top(need, case["dead"]) / dz))
        k, kc = 12.6, 13.0
        step = (120.0 + 8 * k) * n
        sub = (96.0 + 28 * kc) * free + 22.0 * pts
        f_step, f_sub = 60.0 * k * n, (40.0 * kc + 100) * free + 30.0 * pts
        if case["kind"] == "step":
            s, c = case["steps"], (1000 if case["ca_every"] else 0)
            by += s * (step + 26.0 * pts) + c * sub + 102.0 * n
            fl += s * (f_step + 30.0 * pts) + c * f_sub
        elif case["kind"] == "solve":
            by += 1000 * sub
            fl += 1000 * f_sub
        elif case["kind"].startswith("rd_"):
            m = case["n_sub"] * (3 if case["kind"] == "rd_adjoint" else 1)
            by += m * sub
            fl += m * f_sub
        else:
            m = case["n_steps"] * (3 if case["kind"] == "mech_adjoint" else 1)
            by += m * (88.0 + 4 * k) * n
            fl += m * f_step
    return {"bytes": by, "flops": fl}


# ---- the same results in plain 64-bit torch ------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "b_sweep":
        return {"b": [_exact_b(s, i) for s, i in zip(_b_shapes(case), _b_inputs(case, seed))], "err": None}
    if kind == "step":
        return None   # divisions, removals and list order: not an arithmetic result
    cost = sum(free * 13 + grid * grid * nz // 2 for side, free, layers, grid, nz, dz in _sizes(case))
    specs = _specs(case, seed)
    if kind == "solve":
        if cost * 1000 > 1.5e8:
            return None
        m = _CaModel(specs[0])
        u, avg, _ = m.window(1000, *m.default_params(), averages=True)
        avg = torch.where(m.afm, avg / 1000, 0.0)
        u = torch.where(m.afm | ~m.inner, u, 0.0)   # the end of a solve clears the other cells past the sheet
        rec = dict.fromkeys(("n", "state", "touch", "rest_div_times", "pair", "fix_origin") + native.SNAPSHOT_F64)
        avg = torch.where(m.inner, avg, torch.tensor(specs[0]["values"]["ca2p_avg"]))
        empty = specs[0]["geometry"].max_cells - m.n
        rec["ca2p"], rec["ca2p_avg"] = np.pad(u.numpy(), (0, empty)), np.pad(avg.numpy(), (0, empty))
        return rec
    if kind.startswith("rd_"):
        if cost * case["n_sub"] * (5 if kind == "rd_adjoint" else 1) > 4e8:
            return None
        m = _CaModel(specs[0])
        base, target = _rd_params(specs[0], seed)
        if kind == "rd_forward":
            return [m.window(case["n_sub"], *m.params(base))[0].numpy()]
        with torch.no_grad():
            want = m.window(case["n_sub"], *m.params(target))[0]
        p = [q.clone().requires_grad_() for q in m.params(base)]
        u = m.window(case["n_sub"], *p)[0]
        loss = ((u - want)[m.afm] ** 2).mean()
        g = torch.autograd.grad(loss, p)
        kpa = torch.where(m.afm, g[3], 0.0)
        return {"loss": loss.detach().numpy().reshape(1),
                "grads": [{"du": float(g[0]), "dp": float(g[1]), "gj0": float(g[2]), "kpa": kpa.numpy()}]}
    cells = sum(side * side + free for side, free, layers, grid, nz, dz in _sizes(case))
    if cells * case["n_steps"] * (6 if kind == "mech_adjoint" else 1) > 4e6:
        return None
    losses, grads, out = [], [], []
    for s in _crumple(specs, seed):
        m = _MechModel(s)
        p = [torch.tensor(MECH[k], dtype=torch.float64) for k in MECH]
        if kind == "mech_forward":
            out.append(m.window(case["n_steps"], *p).numpy())
            continue
        with torch.no_grad():
            want = m.window(case["n_steps"], *(torch.tensor(MECH_TARGET[k], dtype=torch.float64) for k in MECH))
        p = [q.requires_grad_() for q in p]
        loss = (m.delta(m.window(case["n_steps"], *p) - want) ** 2).sum() / want.shape[1]
        losses.append(float(loss.detach()))
        grads.append([float(g) for g in torch.autograd.grad(loss, p)])
    return out if kind == "mech_forward" else {"loss": np.array(losses), "grads": np.array(grads)}


def _exact_b(shape, host):
    """calc_ext_stim (ext_stim.cpp:18-69): z ends mirror and repeat, x and y are periodic"""
    nx, ny, nz, xp, izb = shape
    b, cmap1, cmap2, state, agek = host
    u, m, cell = b[:nz, :ny, :nx], cmap2[:nz, :ny, :nx].double(), cmap1[:nz, :ny, :nx].long()
    at = torch.arange(nz)
    down, up = torch.cat([at[1:2], at[:-1]]), torch.cat([at[1:], at[-1:]])
    lap = sum(torch.roll(m, s, d) * (torch.roll(u, s, d) - u) for d in (1, 2) for s in (1, -1))
    lap = lap + m[down] * (u[down] - u) + m[up] * (u[up] - u)
    s = torch.where(cell >= 0, state[cell.clamp(min=0)].long(), MEMB)
    on = (s == DEAD) | (s == ALIVE)
    age = torch.where(on, agek[cell.clamp(min=0)], 0.0)
    f = (on & (age > 22.0 - 0.5) & (age <= 22.0 + 2.0)).double() - 0.025 * u
    new = u + 0.01 * (0.0009 * lap * (1 / 0.8) ** 2 + f)
    out = torch.zeros_like(b)
    out[:izb, :ny, :nx] = new[:izb]
    out[:izb, ny, :nx], out[:izb, :ny, nx], out[:izb, ny, nx] = new[:izb, 0], new[:izb, :, 0], new[:izb, 0, 0]
    return out


def _near(a, b, box, reach):
    """index pairs (i, j) of points with |a_i - b_j| <= reach_ij, periodic in x and y; reach(i, j) on broadcast axes"""
    got = []
    for i0 in range(0, a[0].numel(), 2048):
        i1 = min(i0 + 2048, a[0].numel())
        d2 = 0
        for k in range(3):
            d = a[k][i0:i1, None] - b[k][None, :]
            if k < 2:
                d = d - box * torch.round(d / box)
            d2 = d2 + d * d
        i, j = torch.nonzero(d2 <= reach(i0, i1) ** 2, as_tuple=True)
        got.append(torch.stack([i + i0, j]))
    return torch.cat(got, 1)


def _cells(spec):
    c, n = spec["cells"], spec["nmemb"]
    pos = [torch.tensor(c[k]) for k in "xyz"]
    return c, n, pos, torch.tensor(c["radius"]), torch.tensor(c["state"]).long()


class _CaModel:
    """calc_ca2p's sub-step (ca2p.cpp:14-402) of a generated tissue (no AIR, no DER cells)"""

    def __init__(self, spec):
        g, (c, nm, pos, rad, st) = spec["geometry"], _cells(spec)
        self.g, self.n = g, st.numel()
        self.inner = torch.arange(self.n) >= nm
        self.afm = self.inner & ((st == ALIVE) | (st == FIX) | (st == MUSUME))
        self.dead = st == DEAD
        self.alive = st == ALIVE
        self.agek = torch.tensor(c["agek"])
        self.u0, self.p0, self.h0 = (torch.tensor(spec["values"][k]) for k in ("ca2p", "ip3", "ex_inert"))
        p = [q[nm:] for q in pos]
        e = _near(p, p, g.lx, lambda i0, i1: 1.2 * (rad[nm:][i0:i1, None] + rad[nm:][None, :])) + nm
        self.src, self.dst = e[:, e[0] != e[1]]     # every free cell is ALIVE, DEAD, FIX or MUSUME
        # setup_map_lat (map.cpp:18-167): the highest cell index within a radius, the mask within twice an AFM radius
        dims, d = (g.nx, g.ny, g.nz), (g.lx / g.nx, g.ly / g.ny, g.lz / g.nz)
        lat = [(pos[k] * (dims[k] / (g.lx, g.ly, g.lz)[k])).long() for k in range(3)]
        lat = [lat[k] % dims[k] for k in range(3)]
        half = [int(1.4 * dims[k] / (g.lx, g.ly, g.lz)[k]) for k in range(3)]
        owner = torch.full((g.nx * g.ny * g.nz,), -1, dtype=torch.long)
        mask = torch.zeros(g.nx * g.ny * g.nz, dtype=torch.float64)
        idx = torch.arange(self.n)
        for i in range(-2 * half[0], 2 * half[0] + 1):
            for j in range(-2 * half[1], 2 * half[1] + 1):
                for k in range(-2 * half[2], 2 * half[2] + 1):
                    wide = abs(i) > half[0] or abs(j) > half[1] or abs(k) > half[2]
                    q = [lat[0] + i, lat[1] + j, lat[2] + k]
                    dx = [q[a] * d[a] - pos[a] for a in range(3)]
                    dx = [dx[0] - g.lx * torch.round(dx[0] / g.lx), dx[1] - g.ly * torch.round(dx[1] / g.ly), dx[2]]
                    d2 = dx[0] ** 2 + dx[1] ** 2 + dx[2] ** 2
                    ok = (q[2] >= 1) & (q[2] < g.nz) & (self.afm if wide else torch.ones_like(self.afm))
                    v = ((q[0] % g.nx) * g.ny + q[1] % g.ny) * g.nz + q[2].clamp(0, g.nz - 1)
                    hit = ok & (d2 < rad ** 2)
                    owner.scatter_reduce_(0, v[hit], idx[hit], "amax")
                    mask[v[ok & self.afm & (d2 < (2 * rad) ** 2)]] = 1.0
        own = owner.view(g.nx, g.ny, g.nz)
        own_afm = torch.where(own >= 0, self.afm[own.clamp(min=0)], False)
        self.owner = torch.where(own_afm, own, -1)
        self.mask = mask.view(g.nx, g.ny, g.nz)
        z = pos[2][nm:]
        self.izb = int((float(z.max()) + 2.8) / d[2])
        self.A0 = torch.tensor(spec["fields"]["atp"])[:g.nx, :g.ny, :g.nz + 1]
        B = torch.tensor(spec["fields"]["b"])
        a = [lat[k][self.afm] for k in range(3)]
        self.corner = [((a[0] + i) % g.nx, (a[1] + j) % g.ny, a[2] + k)
                       for i in (0, 1) for j in (0, 1) for k in (0, 1)]
        self.Bavg = sum(B[q] for q in self.corner) / 8
        self.inv2 = (g.nx / g.lx) ** 2
        a = self.agek[self.afm]
        al = self.alive[self.afm]
        self.th = torch.where(al, 0.2 + 0.4 * (1 + torch.tanh(3.0 - a)), 1.0)
        self.iag = torch.where(al, 0.5 * (1 + torch.tanh((a - 3.0) / 1.5)), 0.0)

    def params(self, p):
        return [torch.as_tensor(p[k], dtype=torch.float64) for k in ("du", "dp", "gj0", "kpa")]

    def default_params(self):
        kpa = torch.where(self.alive, 4.0 + (1 + torch.tanh(3.0 - self.agek)), 6.0)
        return self.params(dict(du=0.01, dp=0.1, gj0=0.99, kpa=kpa))

    def window(self, n_sub, du, dp, gj0, kpa, averages=False):
        dt, izb, n = 0.01, self.izb, self.n
        afm, kpa = self.afm, kpa[self.afm]
        ea = afm[self.src]                          # edges seen from AFM cells, and from DEAD ones (ALIVE partners)
        s, d = self.src[ea], self.dst[ea]
        toward = self.alive[d]
        ed = self.dead[self.src] & self.alive[self.dst]
        s2, d2 = self.src[ed], self.dst[ed]
        u, p, h, A = self.u0, self.p0, self.h0[afm], self.A0[:, :, :izb + 1]
        w = gj0 * torch.ones(s.numel(), dtype=torch.float64)
        own, has = self.owner[:, :, :izb].clamp(min=0), self.owner[:, :, :izb] >= 0
        m = self.mask
        zm = torch.cat([torch.tensor([1]), torch.arange(izb - 1)])
        zp = torch.arange(1, izb + 1).clamp(max=self.g.nz - 1)
        m0 = m[:, :, :izb]
        avg = torch.zeros(n, dtype=torch.float64)
        add = lambda i, v: torch.zeros(n, dtype=torch.float64).index_add(0, i, v)
        for _ in range(n_sub):
            su, sp = add(s, w * (u[d] - u[s]))[afm], add(s, w * (p[d] - p[s]))[afm]
            fw = (1 - w) + 0.5 * (torch.tanh((0.1 - (u[d] - u[s]).abs()) / 0.1) - 1)
            w = torch.where(toward, w + dt * fw, w)
            ua, pa = u[afm], p[afm]
            Aavg = sum(A[q] for q in self.corner) / 8
            er = 8.1 * (0.567 + 0.1 * pa / (pa + 0.05)) * (0.11 + 0.89 * ua / (0.7 + ua)) * h
            diff = er - 2.0 * ua / (0.1 + ua) + 0.02 + 0.48 * self.Bavg ** 2 / (0.01 + self.Bavg ** 2) + du * self.iag * su
            pn = pa + dt * (kpa * Aavg / (0.5 + Aavg) - 0.3 * pa + dp * self.iag * sp)
            dead = add(s2, p[d2] - p[s2])
            p = torch.where(self.dead, p + dt * (dp * dead - 0.3 * p), p).masked_scatter(afm, pn)
            h = h + dt * (0.49 / (0.49 + ua * ua) - h) / self.th
            u = u.masked_scatter(afm, ua + dt * diff)
            src = torch.where(has, torch.zeros(n, dtype=torch.float64).masked_scatter(afm, diff)[own], 0.0)
            a = A[:, :, :izb]
            lap = sum(torch.roll(m0, k, x) * (torch.roll(a, k, x) - a) for x in (0, 1) for k in (1, -1))
            lap = lap + m[:, :, zm] * (A[:, :, zm] - a) + m[:, :, zp] * (A[:, :, zp.clamp(max=izb)] - a)
            A = torch.cat([a + dt * (lap * self.inv2 + 0.002 * src.clamp(min=0) - 0.5 * a), A[:, :, izb:]], 2)
            if averages:
                avg = avg + u
        return u, avg, p


class _MechModel:
    """cell_interaction + pos_copy (cell_interaction.cpp:48-685) of a generated tissue with frozen lists"""

    def __init__(self, spec):
        g, (c, nm, pos, rad, st) = spec["geometry"], _cells(spec)
        self.box = torch.tensor([g.lx, g.ly, float("inf")], dtype=torch.float64)[:, None]
        self.x0, self.r, self.nm = torch.stack(pos), rad, nm
        self.agek = torch.tensor(c["agek"])
        free = [q[nm:] for q in pos]
        i, j = _near(free, pos, g.lx, lambda a, b: 1.2 * (rad[nm:][a:b, None] + rad[None, :]))
        i = i + nm
        keep = i != j
        i, j = i[keep], j[keep]
        si, sj = st[i], st[j]
        # find_dermis: the nearest membrane particle of a FIX or MUSUME cell
        d = ((self.delta(self.x0[:, i] - self.x0[:, j])) ** 2).sum(0)
        near = torch.full((st.numel(),), float("inf"), dtype=torch.float64)
        memb = sj == MEMB
        near.scatter_reduce_(0, i[memb], d[memb], "amin")
        derm = memb & (d == near[i])
        upper = (si == ALIVE) | (si == DEAD)
        upper_j = (sj == ALIVE) | (sj == DEAD)
        basal = (si == FIX) | (si == MUSUME)
        law = {"lj": basal & memb & ~derm, "fix": (si == FIX) & derm, "mus": (si == MUSUME) & derm,
               "adh": upper & (~upper_j | (i > j)),
               "pro": ((si == FIX) & ((sj == MUSUME) | ((sj == FIX) & (i > j)))) | ((si == MUSUME) & (sj == MUSUME) & (i > j))}
        self.law = {k: (i[v], j[v]) for k, v in law.items()}
        a, b = self.law["adh"]
        self.strong = (self.agek[a] > 3.0) & (self.agek[b] > 3.0)
        self.mus_k = torch.where(torch.tensor(c["rest_div_times"])[self.law["mus"][0]] > 0, 5.0, 0.0).double()
        # the triangular sheet (cellmanager.cpp:66-113), neighbours in a ring
        nx, k = g.nmx, torch.arange(nm)
        row, col = k // nx, k % nx
        rows = nm // nx
        at = lambda y, x: (y % rows) * nx + x % nx
        odd = row % 2
        self.ring = torch.stack([at(row, col + 1), at(row - 1, col + odd), at(row - 1, col + odd - 1), at(row, col - 1),
                                 at(row + 1, col + odd - 1), at(row + 1, col + odd)])

    def delta(self, d):
        return torch.cat([d[:2] - self.box[:2] * torch.round(d[:2] / self.box[:2]), d[2:]])

    def window(self, n_steps, eps, k_adh, k_spring, k_bend):
        x, dt, nm, r = self.x0, 0.01, self.nm, self.r
        ring = self.ring
        far = torch.stack([ring[i][ring[(i + 1) % 6]] for i in range(6)])

        def lj(s, R):
            q = R ** 6 / s ** 3
            return 4 * eps * q * (q - 1) / s

        def adhesion(s, R, K):
            d = s.sqrt()
            e = d / R - 1
            return torch.where(e + 1 > 1.2, 0.0, -(K / d) * e * (1 - e * e / 0.2 ** 2))

        for _ in range(n_steps):
            move = torch.zeros_like(x)
            terms = []
            for k, (i, j) in self.law.items():
                v = self.delta(x[:, i] - x[:, j])
                s, R = (v * v).sum(0), r[i] + r[j]
                touch = s < R * R
                if k == "lj":
                    coef = lj(s, R)
                elif k == "fix":
                    coef = torch.where(touch, lj(s, R), -(k_spring / s.sqrt()) * (s.sqrt() / R - 1))
                else:
                    K = self.mus_k if k == "mus" else torch.where(self.strong, k_adh, k_adh * 0.01) if k == "adh" else k_adh * 0.01
                    coef = torch.where(touch, lj(s, R), adhesion(s, R, K))
                terms.append((i, j, dt * coef * v))
            for a in range(3):   # each sheet edge once
                i, j = torch.arange(nm), ring[a]
                v = self.delta(x[:, i] - x[:, j])
                s, R = (v * v).sum(0), 2.0
                d, cr, lam = s.sqrt(), 2.0 * 0.25, 1.25 * 2.0
                q, q3 = cr ** 6 / s ** 3, cr ** 6 / (lam - d) ** 6
                coef = torch.where(s < cr * cr, 4 * eps * q * (q - 1) / s,
                                   torch.where(s < R * R, -(0.2 / d) * (d / cr - 1),
                                               -(0.2 / R) * (0.75 / 0.25) - 4 * eps * q3 * (q3 - 1) / ((lam - d) * d)))
                terms.append((i, j, dt * coef * v))
            for i, j, t in terms:
                move = move.index_add(1, i, t).index_add(1, j, -t)
            z = x[2, :nm]
            q = r[:nm] ** 6 / z ** 6
            wall = torch.where(z < r[:nm], dt * 4 * eps * q * (q - 1) / (2 * z), 0.0)
            X = x[:, :nm]
            bend = torch.zeros_like(X)
            sub = lambda p, q: self.delta(p - q)
            cross = lambda p, q: torch.linalg.cross(p, q, dim=0)
            unit = lambda p: p / (p * p).sum(0).sqrt()
            fac = lambda c: torch.where(c >= 0, 1 - c, 1 / (1 + c) ** 2)
            for i in range(6):
                A, B, D, E = x[:, ring[i]], x[:, ring[(i + 1) % 6]], x[:, ring[(i + 2) % 6]], x[:, far[i]]
                n1, n2 = unit(cross(sub(X, B), sub(A, B))), unit(cross(sub(A, B), sub(E, B)))
                c = (n1 * n2).sum(0)
                bend = bend + fac(c) * cross(sub(A, B), n2 - c * n1)
                n1, n2 = unit(cross(sub(X, D), sub(B, D))), unit(cross(sub(X, B), sub(A, B)))
                c = (n1 * n2).sum(0)
                bend = bend + fac(c) * (cross(sub(B, D), n2 - c * n1) + cross(sub(A, B), n1 - c * n2))
            sheet = dt * k_bend * bend + torch.stack([torch.zeros_like(wall), torch.zeros_like(wall), wall])
            x = x + move + torch.cat([sheet, torch.zeros(3, x.shape[1] - nm, dtype=torch.float64)], 1)
        return x
