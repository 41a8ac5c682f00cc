"""The workloads whose speed this repository answers for.

Each case is one pass through the solver's public entry points
(ssf_pbf_cuda_amd.pbfx) on a scene of this repository's own kind: a dam break
from the lattice (scenes.config0/1/2 and the tests' small dams), the reference
simulators' scenes (scenes.reference_dam, scenes.reference_sphere_jet), a
batch of dam breaks (scenes.batch_config3) and the differentiable rollout
(scenes.config4).  A pass starts from the same resident input every time: it
copies the input over the state arrays, which the step then advances in place.

"wild" flows use the dam-break workload's tensile correction (k = 0.1), which
throws the fluid out of its lattice within a step and collapses it into piles
over a run; "calm" ones use k = 0.001, which keeps the lattice's density over
many steps, as a settled simulation does.
"""
from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from ssf_pbf_cuda_amd import pbfx, scenes

FLOWS = {"wild": 0.1, "calm": 0.001}


def listed():
    return [
        # the tests' 960-particle dam, one synchronous step: what an interactive
        # caller waits for when the scene is tiny (launches and latency only)
        {"name": "dam_960_sync", "kind": "step", "entry": "sync", "nx": 12, "ny": 10, "nz": 8, "h": 0.1, "iters": 4,
         "flow": "calm", "final": "both", "planes": True, "spheres": 0, "blocks": 1},
        # one frame of the reference application (the sphere jet): emission of a
        # batch, then the step as shipped, with the live count read back
        {"name": "jet_frame_12k", "kind": "jet", "n": 12000},
        # the reference's dam simulator: its lattice, its fixed sphere, no final passes
        {"name": "reference_dam_10k", "kind": "refdam", "space": 0.16},
        # the 32,768-particle dam through the allocation-free step that serving
        # loops and captured graphs use
        {"name": "static_dam_32k", "kind": "static", "nx": 32, "ny": 32, "nz": 32, "h": 0.1, "iters": 4,
         "flow": "calm", "final": "both", "planes": True, "spheres": 0, "blocks": 1},
        # the 32,768-particle dam chained over its collapse into piles
        {"name": "rollout_dam_32k", "kind": "rollout", "steps": 40, "nx": 32, "ny": 32, "nz": 32, "h": 0.1, "iters": 4,
         "flow": "wild", "final": "both", "planes": True, "spheres": 0, "blocks": 1},
        # a ragged, settled scene in motion with a sphere among the planes and
        # XSPH only, plus the density and original-order read-outs of a frame
        {"name": "readout_calm_290k", "kind": "readout", "nx": 101, "ny": 67, "nz": 43, "h": 0.05, "iters": 3,
         "flow": "calm", "final": "xsph", "planes": True, "spheres": 1, "blocks": 1},
        # the headline workload: 1,048,576 particles, one step from the lattice
        {"name": "dam_1m", "kind": "step", "entry": "async", "nx": 128, "ny": 128, "nz": 64, "h": 0.05, "iters": 4,
         "flow": "wild", "final": "both", "planes": True, "spheres": 0, "blocks": 1},
        # the same dam chained: the state after the first steps is piles and spray
        {"name": "rollout_dam_1m", "kind": "rollout", "steps": 10, "nx": 128, "ny": 128, "nz": 64, "h": 0.05,
         "iters": 4, "flow": "wild", "final": "both", "planes": True, "spheres": 0, "blocks": 1},
        # the largest single scene: 8,388,608 particles in two blocks, 3 iterations
        {"name": "double_dam_8m", "kind": "step", "entry": "async", "nx": 128, "ny": 256, "nz": 128, "h": 0.025,
         "iters": 3, "flow": "wild", "final": "both", "planes": True, "spheres": 0, "blocks": 2},
        # parameter sweeps: many independent dams by one recorded graph per step
        {"name": "batch_256_graph", "kind": "batch", "entry": "graph", "scenes": 256, "n_min": 4096, "n_max": 200000,
         "iters": 4, "flow": "wild"},
        # a small batch stepped without a graph
        {"name": "batch_24_async", "kind": "batch", "entry": "async", "scenes": 24, "n_min": 1000, "n_max": 12000,
         "iters": 4, "flow": "calm"},
        # gradient-based fitting: 65,536 particles, forward and backward over 10
        # steps with checkpoints every 5
        {"name": "adjoint_65k", "kind": "adjoint", "steps": 10, "every": 5, "nx": 64, "ny": 32, "nz": 32, "h": 0.1,
         "iters": 4, "flow": "wild", "final": "both", "planes": True, "spheres": 0, "blocks": 1},
    ]


def _log_between(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _lattice(rng, lo, hi):
    """A ragged lattice of about lo..hi points (log-uniform)."""
    a = _log_between(rng, lo, hi) ** (1.0 / 3.0)
    nx, ny = (max(4, int(round(a * rng.uniform(0.6, 1.6)))) for _ in range(2))
    return {"nx": nx, "ny": ny, "nz": max(4, int(round(a ** 3 / (nx * ny))))}


def draw(rng):
    kind = rng.choice(["step", "step", "step", "static", "rollout", "readout", "jet", "refdam", "batch", "adjoint"])
    if kind == "jet":
        return {"kind": kind, "n": int(_log_between(rng, 121, 48000))}
    if kind == "refdam":
        return {"kind": kind, "space": round(rng.uniform(0.08, 0.3), 4)}
    if kind == "batch":
        n_min = int(_log_between(rng, 800, 8000))
        return {"kind": kind, "entry": rng.choice(["graph", "async"]), "scenes": rng.randint(3, 64), "n_min": n_min,
                "n_max": int(n_min * rng.uniform(2, 12)), "iters": rng.choice([3, 4]), "flow": rng.choice(["wild", "calm"])}
    lo, hi = {"step": (800, 2.0e6), "static": (800, 3.2e4), "rollout": (4000, 1.0e5), "readout": (4000, 1.0e6),
              "adjoint": (800, 4.0e4)}[kind]
    c = {"kind": kind, **_lattice(rng, lo, hi), "h": rng.choice([0.1, 0.05, 0.025]), "iters": rng.choice([2, 3, 4, 4, 5]),
         "flow": rng.choice(["wild", "calm"]), "final": rng.choice(["both", "both", "xsph", "none"]),
         "planes": True, "spheres": rng.choice([0, 0, 1]), "blocks": rng.choice([1, 1, 2])}
    if kind == "step":
        c["entry"] = rng.choice(["sync", "async"])
    if kind == "rollout":
        c["steps"] = rng.randint(4, 16)
    if kind == "adjoint":
        c.update(steps=rng.randint(3, 8), every=rng.randint(2, 5), blocks=1, iters=rng.choice([3, 4]))
    return c


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _jittered(points, amount, g):
    u = torch.rand(points.shape, generator=g, device="cuda", dtype=torch.float32)
    return points + (2.0 * u - 1.0) * amount


def _grid_points(nx, ny, nz, origin, space):
    """The lattice in the order of scenes.cartesian_volume (x fastest)."""
    ax = [torch.arange(n, device="cuda", dtype=torch.float32) * space + o for n, o in zip((nx, ny, nz), origin)]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return torch.stack([x, y, z], dim=-1).reshape(-1, 3)


def _no_points(n):
    """The particle arrays of a Scene that is used for its geometry only."""
    return np.broadcast_to(np.zeros((1, 3), np.float32), (n, 3))


def _dam(case):
    """(scene geometry, lattice blocks) of a dam-break case: one block in the
    corner, or two at the x-ends, in a box of the benchmark's proportions."""
    h, nx, ny, nz = case["h"], case["nx"], case["ny"], case["nz"]
    s = 0.5 * h
    n = nx * ny * nz * case["blocks"]
    box = (8.0 * nx * s, ny * s, 2.0 * nz * s) if case["blocks"] == 2 else (2.0 * nx * s, 2.0 * ny * s, nz * s + s)
    if n == 1048576:  # the benchmark's box: the lattice fills an eighth of its floor
        box = (4.0 * nx * s, 2.0 * ny * s, 4.0 * nz * s)
    over = {"scorr_k": FLOWS[case["flow"]], "xsph_on": int(case["final"] != "none"),
            "vort_on": int(case["final"] == "both")}
    hi = np.asarray(box, np.float32)
    pts, nrm = scenes.box_planes(np.zeros(3, np.float32), hi)
    none = np.zeros((0, 4), np.float32)
    outer = np.array([[0.75 * box[0], 0.2 * box[1], 0.5 * box[2], 0.15 * min(box)]], np.float32)
    sc = scenes.Scene(name=case.get("name", "dam"), x=_no_points(n), v=_no_points(n),
                      params=scenes.dam_params(h, **over), iters=case["iters"], box_lo=np.zeros(3, np.float32),
                      box_hi=hi, area_lo=np.full(3, -scenes.NO_DELETION, np.float32),
                      area_hi=np.full(3, scenes.NO_DELETION, np.float32),
                      grid=scenes.calc_grid_size(2.0 * float(np.float32(h)), hi), plane_points=pts,
                      plane_normals=nrm, inner_spheres=none, outer_spheres=outer if case["spheres"] else none)
    o = (0.5 * s, 0.5 * s, 0.5 * s)
    blocks = [(o, (nx, ny, nz))]
    if case["blocks"] == 2:
        blocks.append(((box[0] - nx * s + 0.5 * s, o[1], o[2]), (nx, ny, nz)))
    return sc, blocks


def _dam_input(case, sc, blocks, seed):
    g = _generator(seed)
    s = sc.params.stable_distance
    x = torch.cat([_grid_points(*n, o, s) for o, n in blocks])
    x = _jittered(x, 0.01 * case["h"], g)
    sigma = 0.1 if case["flow"] == "calm" or case["kind"] == "adjoint" else 0.01
    v = sigma * torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float32)
    return x, v


def _jet_input(case, sc, jx, jv, seed):
    """The jet's fluid collected in the bottom of its sphere, in slow motion."""
    g = _generator(seed)
    space = sc.params.stable_distance
    p = _grid_points(60, 60, 60, (0.05, 0.05, 0.05), space)
    inside = p[((p - 3.0) ** 2).sum(1) < 2.9 ** 2]
    order = torch.sort(inside[:, 1], stable=True).indices[: case["n"]]
    x = _jittered(inside[order], 0.05 * space, g)
    v = 0.3 * torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float32)
    return x, v


def _refdam_input(case, sc, seed):
    g = _generator(seed)
    x = _jittered(torch.from_numpy(np.ascontiguousarray(sc.x)).cuda(), 0.05 * case["space"], g)
    return x, 0.1 * torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float32)


def _batch_scenes(case):
    """Dam breaks of log-uniform size with their own parameters
    (scenes.batch_config3's geometry and ranges)."""
    h, s = 0.1, 0.05
    u = scenes.uniform01_f32(3, np.arange(4 * case["scenes"], dtype=np.uint64)).astype(np.float64).reshape(-1, 4)
    out = []
    for k in range(case["scenes"]):
        n = math.exp(math.log(case["n_min"]) + u[k, 0] * (math.log(case["n_max"]) - math.log(case["n_min"])))
        a = max(2, int(round(n ** (1.0 / 3.0))))
        dims = {"nx": a, "ny": a, "nz": max(1, int(round(n / (a * a))))}
        sc, blocks = _dam({"h": h, **dims, "blocks": 1, "iters": case["iters"], "flow": case["flow"],
                           "final": "both", "spheres": 0, "kind": "batch"})
        p = dataclasses.replace(sc.params, stable_density=float(np.float32(sc.params.stable_density * (0.9 + 0.2 * u[k, 1]))),
                                xsph_parameter=float(np.float32(0.005 + 0.045 * u[k, 2])),
                                vc_parameter=float(np.float32(0.001 * u[k, 3])))
        out.append((dataclasses.replace(sc, params=p), blocks))
    return out


def _batch_input(scs, seed):
    g = _generator(seed)
    x = torch.cat([_grid_points(*blocks[0][1], blocks[0][0], sc.params.stable_distance) for sc, blocks in scs])
    x = _jittered(x, 0.001, g)
    return x, 0.01 * torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float32)


def _adjoint_seeds(n, seed):
    """dL/d(final x, v) of a linear loss."""
    g = _generator(seed + 77)
    return [torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64) for _ in range(2)]


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "jet":
        sc, jx, jv = scenes.reference_sphere_jet()
        x0, v0 = _jet_input(case, sc, jx, jv, seed)
        st["jet"] = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (jx, jv)]
        cap = scenes.JET_CAPACITY
    elif kind == "refdam":
        sc = scenes.reference_dam(case["space"])
        x0, v0 = _refdam_input(case, sc, seed)
        cap = sc.n
    elif kind == "batch":
        scs = _batch_scenes(case)
        x0, v0 = _batch_input(scs, seed)
        sc = [s for s, _ in scs]
        cap = x0.shape[0]
    else:
        sc, blocks = _dam(case)
        x0, v0 = _dam_input(case, sc, blocks, seed)
        cap = sc.n
    n = x0.shape[0]
    st["sc"], st["n"] = sc, n
    st["xv0"] = torch.stack([x0, v0])
    if kind == "jet":
        st["x"], st["v"] = (torch.zeros((cap, 3), device="cuda") for _ in range(2))
    else:
        st["xv"] = st["xv0"].clone()  # the state the step advances: one array, one copy restores it
        st["x"], st["v"] = st["xv"][0], st["xv"][1]
    if kind == "static":
        dev = lambda a, w: torch.from_numpy(np.ascontiguousarray(a, np.float32).reshape(-1, w)).cuda() if len(a) else None  # noqa: E731
        st["bound"] = dict(inner=dev(sc.inner_spheres, 4), outer=dev(sc.outer_spheres, 4),
                           plane_points=dev(sc.plane_points, 3), plane_normals=dev(sc.plane_normals, 3))
    elif kind == "batch":
        st["solver"] = pbfx.BatchSolver(sc)
        off = np.concatenate([[0], np.cumsum([s.n for s in sc])]).astype(np.int32)
        st["off0"] = torch.from_numpy(off).cuda()
        st["off"] = st["off0"].clone()
        if case["entry"] == "graph":
            st["stream"] = torch.cuda.Stream()
            torch.cuda.synchronize()
            st["solver"].graph_capture(st["x"], st["v"], st["off"], case["iters"], 1, st["stream"])
    else:
        st["solver"] = pbfx.Solver.for_scene(sc, capacity=cap)
    if kind == "readout":
        st["rho"] = torch.zeros(n, device="cuda")
        st["xr"], st["vr"] = (torch.zeros((n, 3), device="cuda") for _ in range(2))
    if kind == "adjoint":
        st["solver"].adj_enable(case["steps"], case["every"])
        st["gx"], st["gv"] = _adjoint_seeds(n, seed)
        st["gx0"], st["gv0"] = (torch.zeros((n, 3), dtype=torch.float64, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    case, sc, n = st["case"], st["sc"], st["n"]
    kind = case["kind"]
    x, v = st["x"], st["v"]
    cur = torch.cuda.current_stream()
    if kind == "jet":
        x[:n].copy_(st["xv0"][0])
        v[:n].copy_(st["xv0"][1])
        m = st["solver"].add_particles(x, v, n, st["jet"][0], st["jet"][1], st["jet"][0].shape[0], cur)
        live = st["solver"].step(x, v, m, sc.area_lo, sc.area_hi, sc.iters, cur)
        return {"x": x[:live], "v": v[:live], "n": live}
    if kind == "batch" and case["entry"] == "graph":
        s = st["stream"]
        s.wait_stream(cur)
        with torch.cuda.stream(s):
            st["xv"].copy_(st["xv0"])
            st["off"].copy_(st["off0"])
            st["solver"].graph_launch(1, s)
        cur.wait_stream(s)
        return {"x": x, "v": v, "offsets": st["off"]}
    st["xv"].copy_(st["xv0"])
    if kind == "batch":
        st["solver"].batch_step_async(x, v, st["off0"], n, case["iters"], cur)
        st["solver"].batch_offsets(st["off"], cur)
        return {"x": x, "v": v, "offsets": st["off"]}
    if kind == "static":
        pbfx.step_static(sc.params, sc.box_hi, x, v, n, sc.area_lo, sc.area_hi, sc.iters, stream=cur, **st["bound"])
        return {"x": x, "v": v}
    if kind == "refdam":
        live = st["solver"].step(x, v, n, sc.area_lo, sc.area_hi, sc.iters, cur, boundary=False)
        return {"x": x[:live], "v": v[:live], "n": live}
    if kind == "adjoint":
        live = st["solver"].adj_forward(x, v, n, sc.area_lo, sc.area_hi, sc.iters, case["steps"], cur)
        gc, ge, e = st["solver"].adj_backward(st["gx"], st["gv"], st["gx0"], st["gv0"], cur)
        return {"x": x[:live], "v": v[:live], "gx0": st["gx0"], "gv0": st["gv0"], "gc": gc, "ge": ge, "exponent": e}
    if kind == "rollout":
        for _ in range(case["steps"]):
            st["solver"].step_async(x, v, n, sc.area_lo, sc.area_hi, sc.iters, cur)
        return {"x": x, "v": v}
    if kind == "readout":
        st["solver"].step_async(x, v, n, sc.area_lo, sc.area_hi, sc.iters, cur)
        st["solver"].density(x, st["rho"], cur)
        st["solver"].restore_order(x, v, st["xr"], st["vr"], cur)
        return {"x": st["xr"], "v": st["vr"], "rho": st["rho"]}
    if case["entry"] == "sync":
        live = st["solver"].step(x, v, n, sc.area_lo, sc.area_hi, sc.iters, cur)
        return {"x": x[:live], "v": v[:live], "n": live}
    st["solver"].step_async(x, v, n, sc.area_lo, sc.area_hi, sc.iters, cur)
    return {"x": x, "v": v}


def work(case):
    """The state read and written once per step (x and v, 24 bytes each way;
    FP64 gradients likewise in the backward pass), and the arithmetic of the
    pair sums: about 29 listed pairs per particle in every Jacobi iteration
    (35 operations for lambda, 45 for delta-p) and about 30 pairs in each
    final pass (40 operations)."""
    kind = case["kind"]
    if kind == "jet":
        n, iters, passes, pairs = case["n"] + 121, 3, 0, 20
    elif kind == "refdam":
        k = int(3.4 / case["space"]) + 1
        n, iters, passes, pairs = k ** 3, 3, 0, 20
    elif kind == "batch":
        n, iters, passes, pairs = sum(s.n for s, _ in _batch_scenes(case)), case["iters"], 3, 29
    else:
        n, iters, pairs = case["nx"] * case["ny"] * case["nz"] * case["blocks"], case["iters"], 29
        passes = {"both": 3, "xsph": 1, "none": 0}[case["final"]]
    steps = case.get("steps", 1)
    nbytes, flops = 48.0 * n, n * pairs * (80.0 * iters + 40.0 * passes)
    if kind == "readout":
        nbytes += 28.0 * n
    if kind == "adjoint":  # forward once, recomputed once, and about three times its arithmetic backwards
        return {"bytes": steps * nbytes + 96.0 * n, "flops": 5.0 * steps * flops}
    return {"bytes": steps * nbytes, "flops": steps * flops}


# ---------------------------------------------------------------- 64 bits
def _f32(t):
    """Rounded to float32, kept in 64 bits."""
    return t.to(torch.float32).to(torch.float64)


def _cells(p, cw):
    """floor(p / cell width) with the float32 division the grid is defined by."""
    return torch.floor(_f32(p / cw)).to(torch.int64)


def _keys(cell, grid):
    gx, gy, gz = grid
    return ((cell[:, 2] & (gz - 1)) * gy + (cell[:, 1] & (gy - 1))) * gx + (cell[:, 0] & (gx - 1))


def _around():
    return [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]


def _visit(cell, grid, off, body):
    """body(j, valid) for the 27 cells around `cell` in z, y, x order, one
    member of each cell at a time."""
    for d in _around():
        k = _keys(cell + torch.tensor(d, device=cell.device), grid)
        lo, hi = off[k], off[k + 1]
        for t in range(int((hi - lo).max())):
            body(torch.clamp(lo + t, max=cell.shape[0] - 1), lo + t < hi)


def _w(r2, ih):
    t = torch.clamp(1.0 - r2 * ih * ih, min=0.0)
    return 1.56668147065 * ih ** 3 * t ** 3


def _collide(p, dp, sc, sphere_only):
    """The boundary responses, sweep by sweep until none fires."""
    planes = [] if sphere_only else list(zip(sc.plane_points, sc.plane_normals))
    inner = [np.array([3.0, 3.0, 3.0, 3.0])] if sphere_only else list(sc.inner_spheres)
    t = lambda a: torch.tensor(np.asarray(a, np.float64), device=p.device)  # noqa: E731
    live = torch.ones(p.shape[0], dtype=torch.bool, device=p.device)
    for _ in range(sc.params.max_sweeps):
        hit = torch.zeros_like(live)
        for s, is_in in [(s, True) for s in inner] + [(s, bool(sc.params.outer_as_inner)) for s in sc.outer_spheres]:
            c = t(s[:3]) - (p + dp)
            d = c.norm(dim=1)
            fire = live & ((d > float(s[3])) if is_in else (d < float(s[3])))
            moved = dp + c * (1.0001 if is_in else 0.9999) - float(s[3]) * c / d[:, None]
            dp = torch.where(fire[:, None], moved, dp)
            hit |= fire
        for q, m in planes:
            nrm = t(m)
            b = (p + dp - t(q)) @ nrm
            fire = live & (b < 0.0)
            dp = torch.where(fire[:, None], dp - b[:, None] * nrm, dp)
            hit |= fire
        live = live & hit
        if not bool(live.any()):
            break
    return dp


def _exact_step(x, v, sc, sphere_only=False):
    """One step in 64 bits, in the solver's sorted order: (x, v, density over
    the lists, the input index of each row).  The sort and the neighbour lists
    are decided as the step defines them, on float32 predicted positions."""
    P, grid = sc.params, sc.grid
    h, cw = float(P.smoothing_length), float(np.float32(P.smoothing_length))
    ih, m, rho = 1.0 / h, float(P.particle_mass), float(P.stable_density)
    dt, beta = float(P.time_step), m / rho
    grav = torch.tensor([float(np.float32(c)) for c in P.body_force], dtype=torch.float64, device=x.device)
    x, v = x.double(), v.double()
    p = x + dt * (v + dt * grav)
    pf = _f32(x + dt * _f32(v + dt * grav))  # the float32 prediction: decides cells and lists
    key = _keys(_cells(pf, cw), grid)
    lo, hi = (torch.tensor(np.asarray(a, np.float64), device=x.device) for a in (sc.area_lo, sc.area_hi))
    ncell = grid[0] * grid[1] * grid[2]
    key = torch.where(((pf < lo) | (pf > hi)).any(1), torch.full_like(key, ncell), key)
    key, idx = torch.sort(key, stable=True)
    live = int((key < ncell).sum())
    key, idx = key[:live], idx[:live]
    off = torch.searchsorted(key, torch.arange(ncell + 2, device=x.device))
    x, p, pf = x[idx], p[idx], pf[idx]
    cap = int(P.max_pair) - 1
    lst = torch.zeros((live, cap), dtype=torch.int64, device=x.device)
    cnt = torch.zeros(live, dtype=torch.int64, device=x.device)
    rows = torch.arange(live, device=x.device)
    h2 = float(np.float32(P.smoothing_length) * np.float32(P.smoothing_length))

    def collect(j, valid):
        d = _f32(pf - pf[j])
        r2 = _f32(d[:, 2] ** 2 + _f32(d[:, 1] ** 2 + _f32(d[:, 0] ** 2)))
        take = valid & (r2 < h2) & (cnt < cap)
        lst[rows[take], cnt[take]] = j[take]
        cnt.add_(take.long())

    _visit(_cells(pf, cw), grid, off, collect)

    def pairs(k):  # W and grad W of every particle's k-th listed pair
        j = lst[:, k]
        on = k < cnt
        d = p - p[j]
        r2 = (d * d).sum(1)
        r = torch.sqrt(torch.where(r2 > 0, r2, torch.ones_like(r2)))
        kd = -14.3239448745 * ih ** 4 * torch.clamp(1.0 - r * ih, min=0.0) ** 2
        g = d * (kd / r * (on & (r2 > 0)))[:, None]
        return j, on, _w(r2, ih) * on, g

    wdq = float(_w(torch.tensor((P.scorr_dq_over_h * h) ** 2, dtype=torch.float64), ih))
    w04 = float(_w(torch.tensor((0.4 * h) ** 2, dtype=torch.float64), ih))
    for _ in range(sc.iters):
        sw, sg2, sg = torch.zeros_like(p[:, 0]), torch.zeros_like(p[:, 0]), torch.zeros_like(p)
        for k in range(cap):
            _, _, w, g = pairs(k)
            sw, sg, sg2 = sw + w, sg + g, sg2 + (g * g).sum(1)
        s = (sw * beta - 1.0) / (beta * beta * (sg2 + (sg * sg).sum(1)) + float(P.relaxation))
        dp = torch.zeros_like(p)
        for k in range(cap):
            j, on, w, g = pairs(k)
            if P.scorr_mode == scenes.SCORR_PAPER:
                corr = float(P.scorr_k) * (w / wdq) ** int(P.scorr_n)
            else:
                corr = (torch.clamp(-s, min=0.0) + torch.clamp(-s[j], min=0.0)) * 10.0 * w ** 4 / w04 ** 4
            dp = dp - ((s + s[j] + corr) * on)[:, None] * g
        p = p + _collide(p, dp * beta, sc, sphere_only)
    vel = (p - x) / dt
    cell = _cells(_f32(p), cw)

    def final(term):
        tot = [torch.zeros_like(p)]

        def add(j, valid):
            d = p[j] - p
            tot[0] = tot[0] + term(j, d, (d * d).sum(1)) * valid[:, None]

        _visit(cell, grid, off, add)
        return tot[0]

    def spiky(d, r2):  # grad of the spiky kernel along d
        r = torch.sqrt(torch.where(r2 > 0, r2, torch.ones_like(r2)))
        return d * ((-14.3239448745 * ih ** 4 * torch.clamp(1.0 - r * ih, min=0.0) ** 2) / r * (r2 > 0))[:, None]

    if P.vort_on:
        om = beta * final(lambda j, d, r2: torch.linalg.cross(vel[j] - vel, spiky(d, r2)))
        mag = om.norm(dim=1)
        eta = final(lambda j, d, r2: mag[j][:, None] * spiky(d, r2))
        size = eta.norm(dim=1, keepdim=True)
        unit = torch.where(size > 0, eta / torch.where(size > 0, size, torch.ones_like(size)), torch.zeros_like(eta))
        vel = vel + float(P.vc_parameter) * torch.linalg.cross(unit, om) * rho * dt
    if P.xsph_on:
        vel = vel + float(P.xsph_parameter) * beta * final(lambda j, d, r2: (vel[j] - vel) * _w(r2, ih)[:, None])
    dens = torch.zeros_like(p[:, 0])
    for k in range(cap):
        dens = dens + pairs(k)[2] * m
    return p, vel, dens, idx


def exact(case, seed):
    """The pass in 64 bits, for single steps of settled flows.  The wild flow
    has no such value: its particles meet the walls at exactly the wall's
    coordinate, where a rounding decides which response fires, so that a step
    in 64 bits and the same step in 32 lie 10% apart (1e-4 without walls).
    Chained runs and gradients of millions of pairs take too long in plain
    torch."""
    kind = case["kind"]
    if kind in ("rollout", "adjoint") or case.get("flow") == "wild":
        return None
    if kind == "jet":
        sc, jx, jv = scenes.reference_sphere_jet()
        x, v = _jet_input(case, sc, jx, jv, seed)
        x, v = (torch.cat([a, torch.from_numpy(b).cuda()]) for a, b in ((x, jx), (v, jv)))
        p, vel, _, _ = _exact_step(x, v, sc)
        return {"x": p, "v": vel, "n": None}
    if kind == "refdam":
        sc = scenes.reference_dam(case["space"])
        p, vel, _, _ = _exact_step(*_refdam_input(case, sc, seed), sc, sphere_only=True)
        return {"x": p, "v": vel, "n": None}
    if kind == "batch":
        if case["scenes"] > 32:
            return None
        scs = _batch_scenes(case)
        x, v = _batch_input(scs, seed)
        out, at = [], 0
        for sc, _ in scs:
            out.append(_exact_step(x[at:at + sc.n], v[at:at + sc.n], sc)[:2])
            at += sc.n
        return {"x": torch.cat([a for a, _ in out]), "v": torch.cat([b for _, b in out]), "offsets": None}
    sc, blocks = _dam(case)
    if sc.n > 2_500_000:
        return None
    x, v = _dam_input(case, sc, blocks, seed)
    p, vel, dens, idx = _exact_step(x, v, sc)
    if kind == "readout":
        back, vback = torch.empty_like(p), torch.empty_like(p)
        back[idx], vback[idx] = p, vel
        return {"x": back, "v": vback, "rho": dens}
    if kind == "step" and case["entry"] == "sync":
        return {"x": p, "v": vel, "n": None}
    return {"x": p, "v": vel}
