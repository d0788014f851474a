"""Performance cases of the batched patch update, each through an entry point
that an application calls.

A case is one of these kinds:

  block     nsteps of hipclaw_advance from a saved state, then the frame: the
            stretch of a run between two output frames
  graph     the same stretch replayed from a captured graph
  subcycle  coarse steps with a time step per level, then the frame
  loop      the run loop without regridding: the state is kept before every
            step and its Courant number is read after it
  regrid    the run loop with gradient tags, forest adapt, transfer and new
            programs every few steps, from a checkpoint
  ensemble  independent runs in one forest of isolated blocks, each at its own
            dt, replayed from a captured graph
  batch     one batched update of caller-owned device buffers
  halo      ghost-patch messages packed, unpacked and forwarded (several ranks)
  monitor   the diagnostics of a run: conservation totals and refinement tags

The frame of an FP64 run is the whole state (hipclaw_get_q); that of an
FP32-bulk run is the float cell values its VTK file holds
(hipclaw_vtk_values).  Both go to a pinned host buffer that the program keeps.

Forests depend on the case alone, the data on the seed: a bore with a
rarefaction behind it on a ring (shallow water), a shock and a light bubble
(Euler), a disk (advection), each with a smooth perturbation.
"""
import ctypes as C
import math

import numpy as np
import torch

import forestclaw_amd as fa

MBC = 2
SOLVERS = {"advection": fa.RP_ADVECTION, "swe": fa.RP_SHALLOW, "euler": fa.RP_EULER}
PRECISIONS = {"fp64": fa.FP64, "fp32": fa.FP32_BULK}
GAMMA, GRAV = 1.4, 1.0
# floating-point operations of one cell update: a Riemann solve, limiter and
# two transverse solves per interface in both directions
FLOPS = {"advection": 60, "swe": 480, "euler": 800}


def listed():
    return [
        # a small uniform run, each step a call of its own: latency and launches
        {"name": "advection_loop_fp64", "kind": "loop", "problem": "advection", "mx": 16,
         "minlevel": 4, "maxlevel": 4, "precision": "fp64", "sync": False, "steps": 20},
        # a production run of the FP32-bulk form between two frames: ~10^4
        # patches of 32 x 32 on levels 3 to 8, with conservation fix-up
        {"name": "dambreak_block_fp32", "kind": "block", "problem": "swe", "mx": 32,
         "minlevel": 3, "maxlevel": 8, "precision": "fp32", "sync": True, "steps": 200},
        # the FP64 parity form on a mid-size forest
        {"name": "dambreak_block_fp64", "kind": "block", "problem": "swe", "mx": 32,
         "minlevel": 3, "maxlevel": 7, "precision": "fp64", "sync": True, "steps": 100},
        # the application's own loop with a regrid every four steps
        {"name": "dambreak_regrid_fp64", "kind": "regrid", "problem": "swe", "mx": 32,
         "minlevel": 3, "maxlevel": 6, "precision": "fp64", "sync": True, "steps": 24},
        # four equations, walls, a brick of blocks, small patches
        {"name": "shockbubble_block_fp64", "kind": "block", "problem": "euler", "mx": 16,
         "minlevel": 2, "maxlevel": 7, "precision": "fp64", "sync": True, "steps": 100},
        {"name": "shockbubble_loop_fp32", "kind": "loop", "problem": "euler", "mx": 16,
         "minlevel": 2, "maxlevel": 7, "precision": "fp32", "sync": True, "steps": 50},
        # a parameter study: 32 dam breaks in one forest
        {"name": "ensemble_graph_fp32", "kind": "ensemble", "problem": "swe", "mx": 16,
         "minlevel": 2, "maxlevel": 7, "runs": 32, "precision": "fp32", "sync": True, "steps": 100},
        # a time step per level
        {"name": "dambreak_subcycle_fp64", "kind": "subcycle", "problem": "swe", "mx": 16,
         "minlevel": 3, "maxlevel": 7, "precision": "fp64", "sync": True, "steps": 4},
        # patches whose size no tile divides, in the order a partition left them
        {"name": "batch_swe_24x20_fp64", "kind": "batch", "problem": "swe", "mx": 24, "my": 20,
         "patches": 3000, "precision": "fp64", "limiter": 4, "order": 2},
        # a limiter per wave family other than MC, small patches
        {"name": "batch_euler_8x8_fp64", "kind": "batch", "problem": "euler", "mx": 8, "my": 8,
         "patches": 700, "precision": "fp64", "limiter": 3, "order": 2},
        # one exchange of a rank with 300 boundary patches
        {"name": "halo_exchange", "kind": "halo", "problem": "swe", "mx": 32, "minlevel": 3,
         "maxlevel": 6, "precision": "fp64", "sync": True, "patches": 300},
        # conservation check and tags of a large forest
        {"name": "monitor", "kind": "monitor", "problem": "swe", "mx": 32, "minlevel": 3,
         "maxlevel": 8, "precision": "fp64", "sync": False},
    ]


def draw(rng):
    kind = rng.choice(["block", "block", "block", "graph", "subcycle", "loop", "loop", "regrid",
                       "ensemble", "batch", "batch", "batch", "halo", "monitor"])
    precision = rng.choice(["fp64", "fp32"])
    problem = rng.choice(["swe", "swe", "euler", "advection"])
    if kind == "batch":
        # (the FP32-bulk form's results are looked at through frames)
        mx, my = rng.choice([(16, 16), (32, 32), (8, 8), (rng.randint(8, 48), rng.randint(8, 48)),
                             (rng.randint(8, 24), rng.randint(8, 24))])
        cells = int(math.exp(rng.uniform(math.log(2e3), math.log(4e6))))
        return {"kind": kind, "problem": problem, "mx": mx, "my": my,
                "patches": max(3, min(60000, cells // (mx * my))), "precision": "fp64",
                "limiter": rng.choice([4, 4, 4, 1, 2, 3]), "order": rng.choice([2, 2, 2, 1])}
    mx = rng.choice([8, 12, 16, 16, 18, 20, 24, 32, 32, 40])
    minlevel = rng.randint(2, 4)
    maxlevel = rng.randint(max(3, minlevel), 7 if mx <= 24 else 6)
    sync = rng.random() < 0.7
    case = {"kind": kind, "problem": problem, "mx": mx, "minlevel": minlevel, "maxlevel": maxlevel,
            "precision": precision, "sync": sync, "steps": 2 * rng.randint(5, 50)}
    if kind in ("regrid", "monitor", "halo"):
        # the tags, and so the leaves of the regridded forest, follow the FP64 data
        case.update(problem="swe", precision="fp64")
    if kind == "regrid":
        case["steps"] = 4 * rng.randint(2, 6)
    elif kind == "subcycle":
        case.update(problem=rng.choice(["swe", "euler"]), steps=rng.randint(1, 3),
                    maxlevel=max(minlevel + 1, min(maxlevel, minlevel + 4)))
    elif kind == "ensemble":
        case.update(problem="swe", mx=rng.choice([8, 16, 20]), minlevel=2, maxlevel=rng.randint(4, 6),
                    runs=rng.randint(3, 48))
    elif kind == "halo":
        del case["steps"]
        case.update(sync=True, patches=rng.randint(5, 60) if maxlevel < 5 else rng.randint(20, 400))
    elif kind == "monitor":
        del case["steps"]
    return case


# ------------------------------------------------------------------ forests

def _refine(forest, maxlevel, touches, nbx, limit=None):
    """Refine every leaf that touches(x0, x1, y0, y1, block) up to maxlevel
    (or limit[block] of its block); boxes in block units, so that a block is
    one unit wide."""
    for _ in range(maxlevel):
        lv, gx, gy = forest.leaves()
        w = np.ldexp(1.0, -lv.astype(np.int64))
        block = np.minimum(gx >> lv, nbx - 1)
        flags = touches(gx * w, (gx + 1) * w, gy * w, (gy + 1) * w, block)
        if limit is not None:
            flags = flags & (lv < limit[block])
        flags = flags & (lv < maxlevel)
        if not flags.any():
            return
        forest.refine(flags.astype(np.int32), maxlevel)


def _ring(x0, x1, y0, y1, cx, cy, rin, rout):
    """Boxes that meet the ring rin <= r <= rout about (cx, cy)."""
    near = np.hypot(np.maximum(np.maximum(x0 - cx, cx - x1), 0.0),
                    np.maximum(np.maximum(y0 - cy, cy - y1), 0.0))
    far = np.hypot(np.maximum(np.abs(x0 - cx), np.abs(x1 - cx)),
                   np.maximum(np.abs(y0 - cy), np.abs(y1 - cy)))
    return (near <= rout) & (far >= rin)


def _make_forest(case):
    """The forest of a case and the extent it covers."""
    problem, lo, hi = case["problem"], case["minlevel"], case["maxlevel"]
    if case["kind"] == "ensemble":
        n = case["runs"]
        forest = fa.Forest(n, 1, (False, False), lo, isolated=True)
        limit = np.array([max(lo, hi - (3 * b) % 4) for b in range(n)])
        _refine(forest, hi, lambda x0, x1, y0, y1, b: _ring(
            x0, x1, y0, y1, b + 0.5, 0.5, 0.17 + 0.1 * ((5 * b) % 7) / 7, 0.2 + 0.1 * ((5 * b) % 7) / 7),
            n, limit)
        return forest, (0.0, float(n), 0.0, 1.0)
    if problem == "swe":
        forest = fa.Forest(1, 1, (False, False), lo)
        _refine(forest, hi, lambda x0, x1, y0, y1, b: _ring(x0, x1, y0, y1, 0.5, 0.5, 0.17, 0.27), 1)
        return forest, (0.0, 1.0, 0.0, 1.0)
    if problem == "euler":
        # blocks half a unit wide: the shock at x = 0.2 and the bubble's edge
        # r = 0.1 about (0.5, 0.25) in block units
        forest = fa.Forest(4, 1, (False, False), lo)
        _refine(forest, hi, lambda x0, x1, y0, y1, b: ((x0 <= 0.42) & (x1 >= 0.39)) |
                _ring(x0, x1, y0, y1, 1.0, 0.5, 0.185, 0.215), 4)
        return forest, (0.0, 2.0, 0.0, 0.5)
    forest = fa.Forest(1, 1, (True, True), lo)
    if hi > lo:
        _refine(forest, hi, lambda x0, x1, y0, y1, b: _ring(x0, x1, y0, y1, 0.5, 0.5, 0.17, 0.23), 1)
    return forest, (0.0, 1.0, 0.0, 1.0)


# ------------------------------------------------------------------ data

def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _centres(forest, extent, mx, my):
    """Cell centres with ghost cells on the GPU, (npatch, ny, nx)."""
    xl, yl, dx, dy = (_dev(a)[:, None, None] for a in forest.geometry(extent, mx, my))
    i = torch.arange(1 - MBC, mx + MBC + 1, device="cuda", dtype=torch.float64) - 0.5
    j = torch.arange(1 - MBC, my + MBC + 1, device="cuda", dtype=torch.float64) - 0.5
    return torch.broadcast_tensors(xl + i[None, None, :] * dx, yl + j[None, :, None] * dy)


def _euler_state(rho, u, v, p):
    return torch.stack([rho, rho * u, rho * v, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v)], 1)


def _field(case, x, y, seed):
    """The solution at cell centres (x, y): (npatch, meqn, ny, nx)."""
    g = np.random.default_rng(seed)
    sx, sy, phase = g.uniform(-0.004, 0.004), g.uniform(-0.004, 0.004), g.uniform(0, 2 * math.pi)
    amp = g.uniform(0.5, 0.8)
    problem = case["problem"]
    if problem == "advection":
        r = torch.hypot(x - 0.5 - sx, y - 0.5 - sy)
        return ((r < 0.2) * (1.0 + 0.1 * torch.sin(9 * x + phase) * torch.cos(7 * y)))[:, None].contiguous()
    if problem == "euler":
        mach = g.uniform(1.4, 1.6)
        p2 = 1.0 + 2.0 * GAMMA / (GAMMA + 1.0) * (mach ** 2 - 1.0)
        rho2 = (GAMMA + 1.0) * mach ** 2 / ((GAMMA - 1.0) * mach ** 2 + 2.0)
        u2 = mach * math.sqrt(GAMMA) * (1.0 - 1.0 / rho2)
        behind = x < 0.2 + sx
        bubble = torch.hypot(x - 0.5 - sx, y - 0.25 - sy) < 0.1
        wave = 1.0 + 0.02 * torch.sin(11 * x + phase) * torch.cos(13 * y - phase)
        one = torch.ones_like(wave)
        rho = torch.where(behind, rho2 * one, torch.where(bubble, (0.1 + 0.1 * amp) * one, one))
        return _euler_state(rho * wave, torch.where(behind, u2 * one, 0.02 * wave),
                            0.03 * torch.sin(9 * x + phase), torch.where(behind, p2 * one, one) * wave)
    if case["kind"] == "ensemble":
        b = torch.clamp(torch.floor(x), 0, case["runs"] - 1)
        x = x - b
        front = 0.19 + 0.1 * torch.remainder(5 * b, 7) / 7
    else:
        front = 0.25
    dx, dy = x - 0.5 - sx, y - 0.5 - sy
    r = torch.hypot(dx, dy)
    # still water ahead of the front
    ripple = 1.0 + 0.05 * torch.sin(5 * torch.atan2(dy, dx) + 12 * r + phase)
    h = 1.0 + amp * ripple * torch.exp(-((r - front) / 0.08) ** 2) * 0.5 * (1.0 - torch.tanh((r - front) * 400.0))
    # outgoing simple wave: u = 2 (c - c0)
    u = 2.0 * (torch.sqrt(GRAV * h) - math.sqrt(GRAV))
    rr = torch.clamp(r, min=1e-6)
    return torch.stack([h, h * u * dx / rr, h * u * dy / rr], 1)


def _speeds(problem, q):
    """Largest wave speed per patch."""
    if problem == "advection":
        return torch.full((q.shape[0],), 1.0, device=q.device, dtype=q.dtype)
    u, v = torch.abs(q[:, 1] / q[:, 0]), torch.abs(q[:, 2] / q[:, 0])
    if problem == "euler":
        p = (GAMMA - 1) * (q[:, 3] - 0.5 * (q[:, 1] ** 2 + q[:, 2] ** 2) / q[:, 0])
        c = torch.sqrt(GAMMA * p / q[:, 0])
    else:
        c = torch.sqrt(GRAV * q[:, 0])
    return (torch.maximum(u, v) + c).amax(dim=(1, 2))


def _pinned(shape, dtype):
    return torch.zeros(shape, dtype=dtype, pin_memory=True)


def _to_host(t):
    return _pinned(t.shape, t.dtype).copy_(t).numpy()


# ------------------------------------------------------------------ states

def _solver(case, forest, max_patches):
    problem = case["problem"]
    mthbc = {"advection": (2, 2, 2, 2), "swe": (1, 1, 1, 1), "euler": (1, 1, 3, 3)}[problem]
    return fa.Solver(SOLVERS[problem], case["mx"], case["mx"], precision=PRECISIONS[case["precision"]],
                     mthbc=mthbc, grav=GRAV, gamma=GAMMA, max_patches=max_patches,
                     time_sync=bool(case["sync"]), subcycle=case["kind"] == "subcycle")


def _load(st):
    """The forest and data of a state onto its solver (a start or a restart)."""
    sv = st["solver"]
    sv.set_forest(st["forest"], st["extent"])
    sv.set_q(st["q0"])
    if st["aux"] is not None:
        sv.set_aux(st["aux"])
    sv.ghost_fill()


def _frame(st):
    """The solution as the program writes it out."""
    sv = st["solver"]
    n = sv.npatch
    L = fa.lib()
    if n > len(st["frame"]):
        raise RuntimeError("the forest outgrew the frame buffer")
    out = st["frame"][:n]
    if st["case"]["precision"] == "fp32":
        L.hipclaw_vtk_values.argtypes = [C.c_void_p, C.c_int, C.c_int, C.c_void_p]
        fa._check(L.hipclaw_vtk_values(sv._h, 0, n, out.ctypes.data), "hipclaw_vtk_values")
    else:
        fa._check(L.hipclaw_get_q(sv._h, out.reshape(-1), 0, n), "hipclaw_get_q")
    return out


def _frame_buffer(case, sv, n):
    if case["precision"] == "fp32":
        return _pinned((n, sv.my, sv.mx, sv.meqn), torch.float32).numpy()
    return _pinned((n,) + sv.patch_shape, torch.float64).numpy()


def prepare(case, seed):
    fa.initialize_device(0)
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    kind, mx = case["kind"], case["mx"]
    forest, extent = _make_forest(case)
    n = forest.npatch
    x, y = _centres(forest, extent, mx, mx)
    q = _field(case, x, y, seed)
    aux = None
    if case["problem"] == "advection":
        aux = np.empty((n, 2) + tuple(x.shape[1:]))
        aux[:, 0], aux[:, 1] = 1.0, 0.5
    speed = _speeds(case["problem"], q)
    dx = _dev(forest.geometry(extent, mx, mx)[2])
    sv = _solver(case, forest, 2 * n if kind == "regrid" else n)
    st = {"case": case, "solver": sv, "forest": forest, "extent": extent, "aux": aux,
          "q0": _to_host(q), "frame": None, "dt": 0.85 * float((dx / speed.max()).min())}
    del q, x, y
    _load(st)
    if kind == "ensemble":
        lv, gx, _ = forest.leaves()
        block = torch.as_tensor(np.minimum(gx >> lv, case["runs"] - 1).astype(np.int64), device="cuda")
        big = torch.full((case["runs"],), 1e30, device="cuda", dtype=torch.float64)
        per_run = big.scatter_reduce(0, block, dx / speed.max(), "amin")
        sv.set_dt_scale(0.85 * per_run[block].cpu().numpy())
        st["dt"] = 1.0
    if kind in ("graph", "ensemble"):
        sv.capture_graph(st["dt"], case["steps"])
    if kind in ("block", "graph", "ensemble", "subcycle"):
        sv.save_step()
    if kind == "subcycle":
        st["dt"] *= 2 ** (forest.maxlevel - forest.minlevel)
    if kind == "halo":
        sv.advance(st["dt"], 2)   # the messages carry the step's edge fluxes
        # the messages of the rank's boundary patches, and the patches that
        # stand for the neighbour's
        k = min(case["patches"], n // 2)
        order = np.random.default_rng(n).permutation(n)
        st["slots"] = np.sort(order[:k]).astype(np.int32)
        st["remote"] = np.sort(order[k:2 * k]).astype(np.int32)
        st["sent"], st["forwarded"] = (torch.zeros((k, sv.ghost_pack_elems()), device="cuda",
                                                   dtype=torch.float64) for _ in range(2))
    if kind not in ("halo", "monitor"):
        st["frame"] = _frame_buffer(case, sv, 4 * n if kind == "regrid" else n)
    torch.cuda.synchronize()
    return st


def _prepare_batch(case, seed):
    mx, my, n = case["mx"], case["my"], case["patches"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def rand(lo, hi):
        return lo + (hi - lo) * torch.rand((n, 1, 1), device="cuda", dtype=torch.float64, generator=g)

    x = torch.arange(mx + 2 * MBC, device="cuda", dtype=torch.float64)[None, None, :]
    y = torch.arange(my + 2 * MBC, device="cuda", dtype=torch.float64)[None, :, None]

    def wave(amp):   # a smooth wave across the patch
        return amp * torch.sin(rand(0.02, 0.25) * x + rand(0.0, 6.0)) * torch.cos(rand(0.02, 0.25) * y + rand(0.0, 6.0))

    # half of the patches hold a front
    front = (x * torch.cos(rand(0.0, 6.0)) + y * torch.sin(rand(0.0, 6.0)) > rand(-10.0, 20.0)) * (rand(0.0, 1.0) > 0.5)
    problem = case["problem"]
    aux = None
    if problem == "advection":
        q = (front + wave(0.2))[:, None].contiguous()
        aux = torch.stack([1.0 + wave(0.5), 0.5 + wave(0.4)], 1)
    elif problem == "swe":
        h = 1.0 + 0.6 * front + wave(0.2)
        q = torch.stack([h, h * (0.3 * front + wave(0.3)), h * wave(0.3)], 1)
    else:
        q = _euler_state(1.0 + 0.8 * front + wave(0.15), 0.4 * front + wave(0.2), wave(0.2), 1.0 + front + wave(0.2))
    level = torch.randint(0, 3, (n,), device="cuda", generator=g)
    dx = torch.ldexp(torch.full((n,), 1.0 / 1024, device="cuda", dtype=torch.float64), level)
    speed = 2.0 if problem == "advection" else float(_speeds(problem, q).max())
    sv = fa.Solver(SOLVERS[problem], mx, my, precision=PRECISIONS[case["precision"]],
                   order=(case["order"], 2 if case["order"] == 2 else 1),
                   mthlim=[case["limiter"]] * fa.SOLVER_SHAPES[SOLVERS[problem]][1],
                   grav=GRAV, gamma=GAMMA, max_patches=1)
    slots = np.random.default_rng(n).permutation(n).astype(np.int32)
    st = {"case": case, "solver": sv, "q": q, "out": q.clone(), "aux": aux, "dx": dx, "dy": dx.clone(),
          "slots": slots, "dt": 0.8 / 1024 / speed, "cfl": C.c_double(0.0)}
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------ passes

def run(st):
    return globals()["_run_" + st["case"]["kind"]](st)


def _run_block(st):
    sv = st["solver"]
    sv.restore_step()
    cfl = sv.advance(st["dt"], st["case"]["steps"])
    return {"frame": _frame(st), "cfl": cfl}


def _run_graph(st):
    sv = st["solver"]
    sv.restore_step()
    sv.replay_graph()
    return {"frame": _frame(st)}


_run_ensemble = _run_graph


def _run_subcycle(st):
    sv = st["solver"]
    sv.restore_step()
    cfl = sv.advance_subcycle(st["dt"], st["case"]["steps"])
    return {"frame": _frame(st), "cfl": cfl}


def _run_loop(st):
    sv, dt = st["solver"], st["dt"]
    sv.set_q(st["q0"])
    sv.ghost_fill()
    most = 0.0
    for _ in range(st["case"]["steps"]):
        sv.save_step()
        cfl = sv.advance(dt, 1)
        if cfl > 1.0:   # retaken with a smaller step
            sv.restore_step()
            cfl = sv.advance(0.5 * dt, 1)
        most = max(most, cfl)
    return {"frame": _frame(st), "cfl": most}


def _run_regrid(st):
    sv, case, dt = st["solver"], st["case"], st["dt"]
    start = st["forest"]
    forest = fa.Forest(start.nbx, start.nby, start.periodic, leaves=start.leaves())
    st = dict(st, forest=forest)
    _load(st)
    for k in range(case["steps"]):
        sv.save_step()
        cfl = sv.advance(dt, 1)
        if cfl > 1.0:
            sv.restore_step()
            sv.advance(0.5 * dt, 1)
        if (k + 1) % 4 == 0:
            refine, coarsen = sv.tag(0, 2.0, 1.0)
            kind, src = forest.adapt(refine, 1 - coarsen, case["minlevel"], case["maxlevel"])
            sv.regrid(forest, kind, src, st["extent"])
            sv.ghost_fill()
    # the frame file's record has room for every patch the run may reach
    _frame(st)
    leaves = np.full((3, len(st["frame"])), -1, np.int32)
    leaves[:, :forest.npatch] = forest.leaves()
    return {"frame": st["frame"], "leaves": leaves}


def _run_batch(st):
    sv, p = st["solver"], lambda t: None if t is None else t.data_ptr()
    fa._check(fa.lib().hipclaw_step_batch_noalloc(
        C.byref(sv.cfg), st["q"].shape[0], p(st["q"]), p(st["out"]), p(st["aux"]), p(st["dx"]), p(st["dy"]),
        st["slots"], len(st["slots"]), st["dt"], torch.cuda.current_stream().cuda_stream,
        C.byref(st["cfl"])), "hipclaw_step_batch_noalloc")
    return {"q": st["out"], "cfl": st["cfl"].value}


def _run_halo(st):
    sv = st["solver"]
    sv.ghost_pack(st["slots"], st["sent"].data_ptr())
    sv.ghost_unpack(st["remote"], st["sent"].data_ptr())
    sv.ghost_pack(st["remote"], st["forwarded"].data_ptr())
    return {"sent": st["sent"], "forwarded": st["forwarded"]}


def _run_monitor(st):
    sv = st["solver"]
    hi, lo = sv.mass()
    refine, coarsen = sv.tag(0, 2.0, 1.0)
    return {"mass": hi, "refine": refine, "coarsen": coarsen}


# ------------------------------------------------------------------ work

def _bytes_per_cell(meqn, maux, mx, my):
    """One update: q read with its halo and written, aux read with its halo."""
    halo = (mx + 2 * MBC) * (my + 2 * MBC) / (mx * my)
    return 8.0 * (meqn * (halo + 1.0) + maux * halo)


def work(case):
    problem, mx = case["problem"], case["mx"]
    meqn, _, maux = fa.SOLVER_SHAPES[SOLVERS[problem]]
    if case["kind"] == "batch":
        cells = case["patches"] * mx * case["my"]
        return {"bytes": cells * _bytes_per_cell(meqn, maux, mx, case["my"]), "flops": cells * FLOPS[problem]}
    forest, _ = _make_forest(case)
    n = forest.npatch
    cells = n * mx * mx
    slab = 8.0 * n * meqn * (mx + 2 * MBC) ** 2
    if case["kind"] == "monitor":
        return {"bytes": 8.0 * cells * (meqn + 1), "flops": cells * (8 * meqn + 12)}
    if case["kind"] == "halo":
        k = min(case["patches"], n // 2)
        band = meqn * ((mx + 2 * MBC) ** 2 - (mx - 4 * MBC) ** 2) + 4 * (4 * meqn + 2) * mx
        return {"bytes": 8.0 * k * band * 6, "flops": 0}
    updates = cells * case["steps"]
    if case["kind"] == "subcycle":
        lv = forest.leaves()[0].astype(np.int64)
        updates = int((2 ** (lv - forest.minlevel)).sum()) * mx * mx * case["steps"]
    frame = 4.0 * cells * meqn + 8.0 * cells * meqn if case["precision"] == "fp32" else 2.0 * slab
    return {"bytes": updates * _bytes_per_cell(meqn, maux, mx, mx) + frame, "flops": updates * FLOPS[problem]}


# ------------------------------------------------------------------ exact values

def exact(case, seed):
    """The batched update, and the uniform advection run, in plain torch in 64
    bits (the wave-propagation step of Clawpack 4.6 on padded arrays); the
    messages and totals from the data.  A run on an adapted forest has no
    such value here."""
    if case["kind"] == "batch":
        st = _prepare_batch(case, seed)
        a = None if st["aux"] is None else st["aux"]
        r = (st["dt"] / st["dx"])[:, None, None]
        q, speed = _step(case["problem"], st["q"], a, r, case["limiter"], case["order"], 2 if case["order"] == 2 else 1)
        return {"q": q.cpu().numpy(), "cfl": float(speed)}
    if case["kind"] == "loop" and case["problem"] == "advection" and case["minlevel"] == case["maxlevel"]:
        return _exact_advection(case, seed)
    if case["kind"] == "monitor":
        forest, extent = _make_forest(case)
        x, y = _centres(forest, extent, case["mx"], case["mx"])
        q = _field(case, x, y, seed)[:, :, MBC:-MBC, MBC:-MBC]
        _, _, dx, dy = forest.geometry(extent, case["mx"], case["mx"])
        area = _dev(dx * dy)[:, None, None, None]
        return {"mass": (q * area).sum(dim=(2, 3)).sum(dim=0).cpu().numpy(), "refine": None, "coarsen": None}
    return None


def _exact_advection(case, seed):
    forest, extent = _make_forest(case)
    mx = case["mx"]
    x, y = _centres(forest, extent, mx, mx)
    q0 = _field(case, x, y, seed)
    _, gx, gy = forest.leaves()
    n = (1 << case["minlevel"]) * mx
    whole = torch.empty((1, 1, n, n), device="cuda", dtype=torch.float64)
    for p in range(forest.npatch):
        whole[0, 0, gy[p] * mx:(gy[p] + 1) * mx, gx[p] * mx:(gx[p] + 1) * mx] = q0[p, 0, MBC:-MBC, MBC:-MBC]
    r = torch.full((1, 1, 1), 0.85, device="cuda", dtype=torch.float64)   # dt / dx at speed 1
    pad = lambda t: torch.nn.functional.pad(t, (MBC,) * 4, mode="circular")  # noqa: E731
    aux = pad(torch.cat([torch.full_like(whole, 1.0), torch.full_like(whole, 0.5)], 1))
    speed = 0.0
    for _ in range(case["steps"]):
        out, speed = _step("advection", pad(whole), aux, r, 4, 2, 2)
        whole = out[:, :, MBC:-MBC, MBC:-MBC]
    whole = pad(whole)
    frame = torch.stack([whole[0, :, gy[p] * mx:(gy[p] + 1) * mx + 2 * MBC, gx[p] * mx:(gx[p] + 1) * mx + 2 * MBC]
                         for p in range(forest.npatch)])
    if case["precision"] == "fp32":
        frame = frame[:, 0, MBC:-MBC, MBC:-MBC, None]
    return {"frame": frame.cpu().numpy(), "cfl": float(speed)}


def _normal(problem, ql, qr, ar, n):
    """Riemann solves between cells ql and qr; n = 1 (x) or 2 (y).  Returns
    waves, speeds, the two fluctuations and what the transverse solve needs."""
    d = qr - ql
    if problem == "advection":
        s = ar[:, n - 1]
        w = d
        return [w], [s], torch.clamp(s, max=0)[:, None] * w, torch.clamp(s, min=0)[:, None] * w, None
    t = 3 - n
    rl, rr = torch.sqrt(ql[:, 0]), torch.sqrt(qr[:, 0])
    u = (ql[:, n] / rl + qr[:, n] / rr) / (rl + rr)
    v = (ql[:, t] / rl + qr[:, t] / rr) / (rl + rr)

    def vec(*parts):   # mass, normal and transverse momentum (and energy)
        out = [parts[0], None, None] + list(parts[3:])
        out[n], out[t] = parts[1], parts[2]
        return torch.stack(out, 1)

    zero = torch.zeros_like(u)
    if problem == "swe":
        a = torch.sqrt(GRAV * 0.5 * (ql[:, 0] + qr[:, 0]))
        a1 = ((u + a) * d[:, 0] - d[:, n]) / (2 * a)
        a2 = d[:, t] - v * d[:, 0]
        a3 = (d[:, n] - (u - a) * d[:, 0]) / (2 * a)
        waves = [vec(a1, a1 * (u - a), a1 * v), vec(zero, zero, a2), vec(a3, a3 * (u + a), a3 * v)]
        speeds = [u - a, u, u + a]

        def lam(q, sign):
            return q[:, n] / q[:, 0] + sign * torch.sqrt(GRAV * q[:, 0])
        roe = (u, v, a)
    else:
        g1 = GAMMA - 1.0

        def pressure(q):
            return g1 * (q[:, 3] - 0.5 * (q[:, 1] ** 2 + q[:, 2] ** 2) / q[:, 0])
        enth = ((ql[:, 3] + pressure(ql)) / rl + (qr[:, 3] + pressure(qr)) / rr) / (rl + rr)
        uv = u * u + v * v
        a2s = g1 * (enth - 0.5 * uv)
        a = torch.sqrt(a2s)
        a3 = g1 / a2s * ((enth - uv) * d[:, 0] + u * d[:, n] + v * d[:, t] - d[:, 3])
        a2 = d[:, t] - v * d[:, 0]
        a4 = (d[:, n] + (a - u) * d[:, 0] - a * a3) / (2 * a)
        a1 = d[:, 0] - a3 - a4
        waves = [vec(a1, a1 * (u - a), a1 * v, a1 * (enth - u * a)), vec(zero, zero, a2, a2 * v),
                 vec(a3, a3 * u, a3 * v, a3 * 0.5 * uv), vec(a4, a4 * (u + a), a4 * v, a4 * (enth + u * a))]
        speeds = [u - a, u, u, u + a]

        def lam(q, sign):
            return q[:, n] / q[:, 0] + sign * torch.sqrt(GAMMA * pressure(q) / q[:, 0])
        roe = (u, v, a, enth, uv, g1 / a2s)
    # left-going parts with the transonic rarefactions split (entropy fix)
    s0, s1 = lam(ql, -1), lam(ql + waves[0], -1)
    first = torch.where((s0 < 0) & (s1 > 0), s0 * (s1 - speeds[0]) / (s1 - s0), torch.clamp(speeds[0], max=0))
    none = (s0 >= 0) & (speeds[0] > 0)
    s2, s3 = lam(qr - waves[-1], 1), lam(qr, 1)
    last = torch.where((s2 < 0) & (s3 > 0), s2 * (s3 - speeds[-1]) / (s3 - s2), torch.clamp(speeds[-1], max=0))
    amdq = first[:, None] * waves[0]
    inner = sum(speeds[k][:, None] * waves[k] for k in range(1, len(waves) - 1)) + last[:, None] * waves[-1]
    amdq = torch.where(none[:, None], torch.zeros_like(amdq), amdq + torch.where((speeds[1] < 0)[:, None], inner, torch.zeros_like(amdq)))
    apdq = sum(s[:, None] * w for s, w in zip(speeds, waves)) - amdq
    return waves, speeds, amdq, apdq, roe


def _transverse(problem, roe, asdq, am, ap, n):
    """asdq split into its down-going and up-going parts; am, ap: aux of the
    cell it acts on and of the next cell up."""
    t = 3 - n
    if problem == "advection":
        return torch.clamp(am[:, t - 1:t], max=0) * asdq, torch.clamp(ap[:, t - 1:t], min=0) * asdq
    u, v, a = roe[:3]

    def vec(*parts):
        out = [parts[0], None, None] + list(parts[3:])
        out[n], out[t] = parts[1], parts[2]
        return torch.stack(out, 1)

    zero = torch.zeros_like(u)
    m, mn, mt = asdq[:, 0], asdq[:, n], asdq[:, t]
    if problem == "swe":
        a1, a3 = ((v + a) * m - mt) / (2 * a), (mt - (v - a) * m) / (2 * a)
        waves = [vec(a1, a1 * u, a1 * (v - a)), vec(zero, mn - u * m, zero), vec(a3, a3 * u, a3 * (v + a))]
    else:
        enth, uv, g1a2 = roe[3:]
        a3 = g1a2 * ((enth - uv) * m + u * mn + v * mt - asdq[:, 3])
        a2 = mn - u * m
        a4 = (mt + (a - v) * m - a * a3) / (2 * a)
        a1 = m - a3 - a4
        waves = [vec(a1, a1 * u, a1 * (v - a), a1 * (enth - v * a)),
                 vec(a3, a3 * u + a2, a3 * v, a3 * 0.5 * uv + a2 * u),
                 vec(a4, a4 * u, a4 * (v + a), a4 * (enth + v * a))]
    speeds = [v - a, v, v + a]
    return (sum(torch.clamp(s, max=0)[:, None] * w for s, w in zip(speeds, waves)),
            sum(torch.clamp(s, min=0)[:, None] * w for s, w in zip(speeds, waves)))


def _philim(limiter, r):
    if limiter == 1:
        return torch.clamp(torch.clamp(r, max=1), min=0)
    if limiter == 2:
        return torch.clamp(torch.maximum(torch.clamp(2 * r, max=1), torch.clamp(r, max=2)), min=0)
    if limiter == 3:
        return (r + r.abs()) / (1 + r.abs())
    return torch.clamp(torch.minimum(torch.clamp((1 + r) / 2, max=2), 2 * r), min=0)


def _sweep(problem, q, aux, r, n, limiter, order, trans):
    """One sweep along the last axis over all rows but the outermost.
    Returns the normal flux parts (m, p) at every interface, the four
    transverse parts and the largest Courant number."""
    row = q[:, :, 1:-1]
    ar = None if aux is None else aux[:, :, 1:-1, 1:]
    waves, speeds, amdq, apdq, roe = _normal(problem, row[..., :-1], row[..., 1:], ar, n)
    cfl = max(float((r * s[..., 1:-1].abs()).max()) for s in speeds)
    corr = torch.zeros_like(amdq)
    if order == 2:
        for w, s in zip(waves, speeds):
            norm = (w * w).sum(1)
            dot = torch.zeros_like(norm)
            dot[..., 1:] = (w[..., 1:] * w[..., :-1]).sum(1)
            right = torch.zeros_like(norm)
            right[..., :-1] = dot[..., 1:]
            phi = _philim(limiter, torch.where(s > 0, dot, right) / torch.where(norm == 0, 1.0, norm))
            phi = torch.where(norm == 0, 1.0, phi)
            phi[..., 0] = phi[..., -1] = 1.0
            corr = corr + (s.abs() * (1 - s.abs() * r))[:, None] * (phi[:, None] * w)
    fm, fp = amdq + 0.5 * corr, -apdq + 0.5 * corr
    if order == 2 and trans == 2:
        amdq, apdq = amdq + corr, apdq - corr
    none = [None, None, None, None]
    if aux is not None:   # aux of the cells left and right of each interface, and one row up
        none = [aux[:, :, 1:-1, :-1], aux[:, :, 2:, :-1], aux[:, :, 1:-1, 1:], aux[:, :, 2:, 1:]]
    left = _transverse(problem, roe, amdq, none[0], none[1], n)
    right = _transverse(problem, roe, apdq, none[2], none[3], n)
    return fm, fp, left, right, cfl


def _step(problem, q, aux, r, limiter, order, trans):
    """q after one step (ghost cells as they were) and the Courant number."""
    turn = lambda t: None if t is None else t.transpose(2, 3)  # noqa: E731
    fm, fp, xl, xr, cx = _sweep(problem, q, aux, r, 1, limiter, order, trans)
    gm, gp, yl, yr, cy = _sweep(problem, turn(q), turn(aux), r, 2, limiter, order, trans)
    half = -0.5 * r[:, None]

    def cross(left, right):
        """Transverse parts at the two faces (below, above) of every cell of a
        sweep's rows that is not outermost along it."""
        return [half * (a[..., 1:] + b[..., :-1]) for a, b in zip(left, right)]

    below, above = cross(xl, xr)     # rows 0..my+1, columns 0..mx+1 less the halo's ends
    gx = above[:, :, :-1] + below[:, :, 1:]          # y-faces 1/2 .. my+1/2
    before, after = cross(yl, yr)
    fy = turn(after[:, :, :-1] + before[:, :, 1:])   # x-faces
    fx_m, fx_p = (t[:, :, 1:-1, 1:-1] + fy[:, :, 1:-1] for t in (fm, fp))
    gy_m, gy_p = (turn(t[:, :, 1:-1, 1:-1]) + gx[..., 1:-1] for t in (gm, gp))
    out = q.clone()
    out[:, :, MBC:-MBC, MBC:-MBC] -= r[:, None] * (fx_m[..., 1:] - fx_p[..., :-1]) + \
        r[:, None] * (gy_m[:, :, 1:] - gy_p[:, :, :-1])
    return out, max(cx, cy)
