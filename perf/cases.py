"""Timed cases of the MPM substep library, each through the entry points a program calls.

Kinds of case
  frame   one frame of a resident simulation as the fused node runs it (import the particles,
          k substeps, export them): elastic, fluid, sand and FLIP scenes from a few thousand
          particles, where launches and latency count, to the 4,194,304 of the dam break
  nodes   one pass of the node chain on two AoSoA32 TileVectors (a J-fluid and a fixed-corotated
          object), call by call, with MaxVelSqr read back, as the graph of seven nodes does it
  batch   many independent scenes in one context: a saved state loaded, one replay of a captured
          10-substep HIP graph, the states exported
  grad    a differentiable rollout, forward and backward, through the autograd function
  morton  the Morton reordering of a particle TileVector

Positions, velocities and deformations come from the seed: material cells filled with jittered
(or uniformly random) positions, a smooth flow with its gradient as C, deformations of a few per
cent, as in the middle of a simulation.
"""
import math

import torch
from torch.utils.checkpoint import checkpoint

from zeno_amd.diff import Rollout, rollout
from zeno_amd.zmpm import (ANISO_ARAP, BOUNDARY_STICKY_BOX, COLLIDER_SLIP, COLLIDER_STICKY, LAYOUT_AOSOA32,
                           MODEL_FCR, MODEL_JFLUID, MODEL_NEO_HOOKEAN, MODEL_STABLE_NEO_HOOKEAN, MODEL_STVK_HENCKY,
                           PLASTIC_DRUCKER_PRAGER, SHAPE_HALFSPACE, SHAPE_SPHERE, TRANSFER_AFLIP, TRANSFER_APIC,
                           TRANSFER_FLIP, Context, StepParams, collider, particle_view)

DEV = "cuda:0"
PAD = 3
GRAVITY = (0.0, -9.8, 0.0)
RHO = 1000.0
PPC = 8
SOLIDS = {"fcr": MODEL_FCR, "sand": MODEL_STVK_HENCKY, "nhk": MODEL_NEO_HOOKEAN, "snhk": MODEL_STABLE_NEO_HOOKEAN}
TRANSFERS = {"apic": TRANSFER_APIC, "aflip": TRANSFER_AFLIP, "flip": TRANSFER_FLIP}
BULK = 1e4


def listed():
    return [
        # the smallest ordinary scene: both models on a 32^3 grid (launch latency)
        dict(name="frame_mixed_3k", kind="frame", n=3264, cells=32, solid="fcr", fluid=0.735, transfer="apic",
             layout="jitter", colliders=False, steps=8),
        # the plain elastic cube: 65,536 particles at dx 1/128
        dict(name="frame_cube_65k", kind="frame", n=65536, cells=128, solid="fcr", fluid=0.0, transfer="apic",
             layout="jitter", colliders=False, steps=20),
        # a fluid tank in mid-simulation: random cell counts, particles in no spatial order, an odd size
        dict(name="frame_tank_613k", kind="frame", n=613057, cells=128, solid="fcr", fluid=0.9, transfer="apic",
             layout="shuffled", colliders=False, steps=20),
        # the dam break, the throughput workload
        dict(name="frame_dam_4M", kind="frame", n=4194304, cells=256, solid="fcr", fluid=0.9314, transfer="apic",
             layout="jitter", colliders=False, steps=20),
        # Drucker-Prager sand under ASFLIP over a slope and a sphere (plasticity, colliders)
        dict(name="frame_sand_asflip_200k", kind="frame", n=200003, cells=96, solid="sand", fluid=0.0,
             transfer="aflip", layout="random", colliders=True, steps=10),
        # stable Neo-Hookean jelly in fluid under FLIP
        dict(name="frame_jelly_flip_98k", kind="frame", n=98317, cells=64, solid="snhk", fluid=0.5, transfer="flip",
             layout="random", colliders=False, steps=10),
        # the node chain on two TileVectors: a small graph and an ordinary one
        dict(name="nodes_20k", kind="nodes", n=20011, cells=48, fluid=0.6),
        dict(name="nodes_500k", kind="nodes", n=500009, cells=128, fluid=0.6),
        # 256 independent elastic boxes, 2k to 64k particles each, as one batch
        dict(name="batch_256", kind="batch", scenes=256, lo=2048, hi=65536, steps=10),
        # the differentiable block of 131,072 particles, and a few small scenes identified together
        dict(name="grad_block_131k", kind="grad", scenes=1, n=131072, cells=128, steps=16, every=8),
        dict(name="grad_scenes_8x5k", kind="grad", scenes=8, n=5003, cells=64, steps=12, every=4),
        # Morton reordering of a 28-channel TileVector
        dict(name="morton_1M", kind="morton", n=1048583, nch=28),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "nodes", "batch", "grad", "morton"])
    if kind == "frame":
        n = _log(rng, 2000, 3500000) | 1
        need = (n / PPC / 0.12) ** (1.0 / 3.0) + 8
        cells = next(c for c in (32, 48, 64, 96, 128, 192, 256) if c >= need or c == 256)
        solid = rng.choice(["fcr", "fcr", "sand", "nhk", "snhk", "arap"])
        transfer = rng.choice(["apic", "apic", "apic", "aflip", "flip"])
        big = n > 600000
        return dict(kind="frame", n=n, cells=cells, solid="fcr" if big else solid,
                    fluid=round(rng.choice([0.0, rng.uniform(0.2, 0.9)]) if not big else rng.uniform(0.7, 0.95), 3),
                    transfer="apic" if big else transfer, layout=rng.choice(["jitter", "random", "shuffled"]),
                    colliders=rng.random() < 0.3, steps=rng.choice([4, 8, 10, 20]))
    if kind == "nodes":
        n = _log(rng, 4000, 2000000) | 1
        need = (n / PPC / 0.12) ** (1.0 / 3.0) + 8
        cells = next(c for c in (32, 48, 64, 96, 128, 192, 256) if c >= need or c == 256)
        return dict(kind="nodes", n=n, cells=cells, fluid=round(rng.uniform(0.2, 0.8), 3))
    if kind == "batch":
        lo = _log(rng, 500, 8000)
        return dict(kind="batch", scenes=_log(rng, 3, 160), lo=lo, hi=lo * rng.choice([2, 4, 8]), steps=10)
    if kind == "grad":
        n = _log(rng, 2000, 110000) | 1
        return dict(kind="grad", scenes=rng.choice([1, 1, 3, 8]) if n < 30000 else 1, n=n,
                    cells=64 if n < 30000 else 128, steps=rng.choice([6, 10, 16]), every=rng.choice([4, 8]))
    return dict(kind="morton", n=_log(rng, 3000, 4000000), nch=rng.choice([20, 28]))


# ------------------------------------------------------------------ inputs
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1009 + salt)
    return g


def _fill(n, lo, size, dx, layout, g):
    """n positions (3, n) in the box of cells [lo, lo + size): PPC jittered per cell, cells in x-major
    order (the last cell part full), or uniform in the cells' boxes."""
    need = -(-n // PPC)
    side = max(1, math.ceil(need ** (1.0 / 3.0)))
    d = [min(side, size[0]), min(side, size[1]), 1]
    d[2] = -(-need // (d[0] * d[1]))
    while d[2] > size[2]:
        k = 0 if d[0] < size[0] else 1
        d[k] += 1
        d[2] = -(-need // (d[0] * d[1]))
    ext = torch.tensor(d, device=DEV, dtype=torch.float64)[:, None]
    off = torch.tensor(lo, device=DEV, dtype=torch.float64)[:, None]
    if layout == "jitter":
        c = torch.arange(need, device=DEV)
        cell = torch.stack([c // (d[1] * d[2]), (c // d[2]) % d[1], c % d[2]]).double()
        x = cell.repeat_interleave(PPC, dim=1)[:, :n] + torch.rand(3, n, generator=g, device=DEV, dtype=torch.float64)
    else:
        x = torch.rand(3, n, generator=g, device=DEV, dtype=torch.float64) * ext
    return (off + x) * dx


def _flow(x, g, speed):
    """A smooth velocity field (3, n) and its gradient (9, n) at the positions, with a little noise."""
    n = x.shape[1]
    v = torch.zeros_like(x)
    C = torch.zeros(9, n, device=DEV, dtype=torch.float64)
    r = torch.rand(6, 7, generator=g, device=DEV, dtype=torch.float64).cpu()
    for m in range(6):
        k = [2.0 * math.pi * (3.0 + 5.0 * float(r[m, a])) * (1 if float(r[m, 3]) < 0.5 else -1) ** a for a in range(3)]
        p = k[0] * x[0] + k[1] * x[1] + k[2] * x[2] + 6.28 * float(r[m, 4])
        a, comp = speed * (0.4 + 0.6 * float(r[m, 5])), m % 3
        v[comp] += a * torch.sin(p)
        for c in range(3):
            C[3 * comp + c] += a * k[c] * torch.cos(p)
    v += 0.02 * speed * torch.randn(3, n, generator=g, device=DEV, dtype=torch.float64)
    v += speed * torch.tensor([[0.3], [-0.5], [0.2]], device=DEV, dtype=torch.float64)
    return v, C


def _deformation(n, x, g, amount):
    p = 2.0 * math.pi * 6.0 * (x[0] + 0.7 * x[1] + 0.4 * x[2])
    F = torch.zeros(9, n, device=DEV, dtype=torch.float64)
    ph = torch.rand(9, generator=g, device=DEV, dtype=torch.float64).cpu() * 6.28
    for q in range(9):
        F[q] = (1.0 if q % 4 == 0 else 0.0) + amount * torch.sin(p + float(ph[q]))
    return F + 0.1 * amount * torch.randn(9, n, generator=g, device=DEV, dtype=torch.float64)


def _particles(x, fluid, g, speed, amount=0.04):
    """SoA float32 state: fluid (n,) bool marks the J-fluid particles (J in F[0], material 0), the rest material 1."""
    n = x.shape[1]
    v, C = _flow(x, g, speed)
    F = _deformation(n, x, g, amount)
    J = 1.0 + 0.5 * amount * torch.sin(2.0 * math.pi * 5.0 * (x[0] - x[2]))
    F = torch.where(fluid[None, :], torch.zeros_like(F), F)
    F[0] = torch.where(fluid, J, F[0])
    f = lambda t: t.float().contiguous()  # noqa: E731
    return {"x": f(x), "v": f(v), "C": f(C), "F": f(F), "mat": (~fluid).int().contiguous()}


def _dt(cells):
    return 0.0128 / cells


def _materials(solid, dx):
    s = dict(model=SOLIDS.get(solid, MODEL_FCR), E=1e5, nu=0.3, rho=RHO, vol=dx ** 3 / PPC, flip_beta=0.5)
    if solid == "sand":
        s.update(plasticity=PLASTIC_DRUCKER_PRAGER, friction_angle=35.0)
    if solid == "arap":
        s.update(aniso=ANISO_ARAP, aniso_strength=5.0)
    return [dict(model=MODEL_JFLUID, rho=RHO, vol=dx ** 3 / PPC, bulk=BULK), s]


def _frame_inputs(case, seed):
    cells, n = case["cells"], case["n"]
    dx = 1.0 / cells
    g = _gen(seed)
    nf = int(round(case["fluid"] * n))
    room = cells - 2 * (PAD + 1)
    # the fluid stands at the low wall, the solid beside it; each takes the room it needs
    w = max(2, int(room * (0.55 if nf else 0.0)))
    parts, flags = [], []
    if nf:
        parts.append(_fill(nf, (PAD, PAD, PAD), (w, room, room), dx, case["layout"], g))
        flags.append(torch.ones(nf, dtype=torch.bool, device=DEV))
    if n - nf:
        lo = (PAD + w + 2, PAD + 2, PAD + 2)
        parts.append(_fill(n - nf, lo, (room - w - 2, room - 2, room - 2), dx, case["layout"], g))
        flags.append(torch.zeros(n - nf, dtype=torch.bool, device=DEV))
    x, fluid = torch.cat(parts, dim=1), torch.cat(flags)
    if case["layout"] == "shuffled":
        p = torch.randperm(n, generator=g, device=DEV)
        x, fluid = x[:, p].contiguous(), fluid[p].contiguous()
    st = _particles(x, fluid, g, speed=0.6)
    if case["transfer"] == "aflip":
        st["beta"] = (0.5 * torch.rand(n, generator=g, device=DEV)).contiguous()
    if case["solid"] == "arap":
        a = torch.randn(3, n, generator=g, device=DEV)
        st["a"] = (a / a.norm(dim=0, keepdim=True)).contiguous()
    return st, dx, _materials(case["solid"], dx)


SLOPE = (0.6, 0.8, 0.0, 0.18)     # a slip plane n . x = d
BALL = (0.45, 0.15, 0.45, 0.12)   # a sticky sphere


# Channel maps of the two TileVectors (Generation.cpp:868-884): x 1, v 4, vol 7, C 8, J or F at 19.
CHN = {"m": 0, "x": 1, "v": 4, "vol": 7, "C": 8, "J": 19, "F": 19}


def _tiles(planes, nch):
    """(nch, n) channel planes -> the TileVector's flat AoSoA32 buffer."""
    n = planes.shape[1]
    t = -(-n // 32)
    buf = torch.zeros(nch, t * 32, device=planes.device, dtype=planes.dtype)
    buf[:, :n] = planes
    return buf.view(nch, t, 32).permute(1, 0, 2).contiguous().view(-1)


def _nodes_inputs(case, seed):
    st, dx, mats = _frame_inputs(dict(case, layout="random", transfer="apic", solid="fcr", colliders=False), seed)
    g = _gen(seed, 5)
    objs = []
    for fluid in (True, False):
        sel = (st["mat"] == 0) == fluid
        n = int(sel.sum())
        planes = torch.zeros(20 if fluid else 28, n, device=DEV)
        planes[1:4], planes[4:7], planes[8:17] = st["x"][:, sel], st["v"][:, sel], st["C"][:, sel]
        planes[7] = mats[0]["vol"] * (0.8 + 0.4 * torch.rand(n, generator=g, device=DEV))
        planes[0] = RHO * planes[7]
        if fluid:
            planes[19] = st["F"][0, sel]
        else:
            planes[19:28] = st["F"][:, sel]
        objs.append(planes)
    return objs, dx, mats


def _batch_inputs(case, seed):
    """Scene descriptions fixed by their index, particles from the seed."""
    import random
    descs, mats, xs, scene, speeds = [], [], [], [], []
    g = _gen(seed)
    for i in range(case["scenes"]):
        r = random.Random(977 * i + 13)
        n = int(round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"])))))
        cells = r.choice([64, 128])
        side = r.uniform(0.1, 0.3)
        E = math.exp(r.uniform(math.log(1e4), math.log(1e6)))
        mats.append(dict(model=MODEL_FCR, E=E, nu=r.uniform(0.1, 0.4), rho=RHO, vol=side ** 3 / n, scene=i))
        descs.append(dict(dx=1.0 / cells, n_cells=cells, dt=1e-4, gravity=GRAVITY, boundary=BOUNDARY_STICKY_BOX, pad=PAD))
        xs.append(0.5 - 0.5 * side + side * torch.rand(3, n, generator=g, device=DEV, dtype=torch.float64))
        scene.append(torch.full((n,), i, dtype=torch.int32, device=DEV))
    x, scene = torch.cat(xs, dim=1), torch.cat(scene)
    st = _particles(x, torch.zeros(x.shape[1], dtype=torch.bool, device=DEV), g, speed=0.5, amount=0.02)
    st["mat"] = scene.contiguous()
    return st, descs, mats


def _grad_inputs(case, seed):
    g = _gen(seed)
    cells, n, S = case["cells"], case["n"], case["scenes"]
    dx = 1.0 / cells
    descs, mats, xs, scene = [], [], [], []
    side = math.ceil((n / PPC) ** (1.0 / 3.0))
    lo = (cells - side) // 2
    for i in range(S):
        xs.append(_fill(n, (lo, lo, lo), (side + 1,) * 3, dx, "jitter", g))
        scene.append(torch.full((n,), i, dtype=torch.int32, device=DEV))
        mats.append(dict(model=MODEL_FCR, rho=RHO, vol=dx ** 3 / PPC, scene=i))
        descs.append(dict(dx=dx, n_cells=cells, dt=_dt(cells), gravity=GRAVITY, boundary=BOUNDARY_STICKY_BOX, pad=PAD))
    x = torch.cat(xs, dim=1)
    st = _particles(x, torch.zeros(x.shape[1], dtype=torch.bool, device=DEV), g, speed=0.5)
    st["mat"] = torch.cat(scene).contiguous()
    E = (5e4 * (1.0 + 0.2 * torch.rand(S, generator=g, device=DEV))).float().cpu()
    nu = (0.25 + 0.1 * torch.rand(S, generator=g, device=DEV)).float().cpu()
    # dL/dx of a loss that pulls the body apart along x, squeezes it along y and shakes it a little
    c = x.mean(dim=1, keepdim=True)
    w = torch.tensor([[1.0], [-0.7], [0.4]], device=DEV, dtype=torch.float64)
    xbar = (2.0 * w * (x - c) + 0.02 * torch.randn(x.shape, generator=g, device=DEV, dtype=torch.float64)) / n
    return st, descs, mats, E, nu, xbar.float().contiguous()


# ------------------------------------------------------------------ prepare / run
def _step(cells):
    return StepParams(_dt(cells), GRAVITY, BOUNDARY_STICKY_BOX, PAD)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "frame":
        st, dx, mats = _frame_inputs(case, seed)
        ctx = Context(dx, case["cells"], case["n"])
        ctx.set_materials(mats)
        ctx.set_transfer(TRANSFERS[case["transfer"]])
        if case["colliders"]:
            ctx.set_colliders([collider(COLLIDER_SLIP, SHAPE_HALFSPACE, SLOPE),
                               collider(COLLIDER_STICKY, SHAPE_SPHERE, BALL)])
        return dict(kind=kind, ctx=ctx, st=st, p=_step(case["cells"]), steps=case["steps"])
    if kind == "nodes":
        objs, dx, mats = _nodes_inputs(case, seed)
        ctx = Context(dx, case["cells"], case["n"])
        ctx.set_materials(mats)
        tin = [_tiles(o, o.shape[0]) for o in objs]
        tout = [torch.zeros_like(t) for t in tin]

        def views(tiles):
            out = []
            for k, (o, t) in enumerate(zip(objs, tiles)):
                F = dict(J=t) if k == 0 else dict(F=t)
                out.append(particle_view(o.shape[1], t, t, t, layout=LAYOUT_AOSOA32, tile_channels=o.shape[0], chn=CHN,
                                         m=t, vol=t, default_material=k, **F))
            return out

        return dict(kind=kind, ctx=ctx, tin=tin, tout=tout, vin=views(tin), vout=views(tout), dt=_dt(case["cells"]))
    if kind == "batch":
        st, descs, mats = _batch_inputs(case, seed)
        ctx = Context.scenes(descs, st["x"].shape[1])
        ctx.set_materials(mats)
        ctx.import_state(st)
        ctx.autotune(None, 4)
        ctx.graph_capture(None, case["steps"])
        saved = ctx.new_state_buffer()
        ctx.state_save(saved)
        return dict(kind=kind, ctx=ctx, saved=saved)
    if kind == "grad":
        st, descs, mats, E, nu, xbar = _grad_inputs(case, seed)
        ctx = Context.scenes(descs, st["x"].shape[1])
        sim = Rollout(ctx, st, mats, None, case["steps"], checkpoint_every=case["every"])
        v0 = st["v"].clone().requires_grad_(True)
        return dict(kind=kind, sim=sim, v0=v0, E=E.requires_grad_(True), nu=nu.requires_grad_(True), xbar=xbar)
    g = _gen(seed)
    n, nch = case["n"], case["nch"]
    planes = torch.rand(nch, n, generator=g, device=DEV)
    ctx = Context(1.0 / 64, 64, n)
    i32 = dict(dtype=torch.int32, device=DEV)
    src = _tiles(planes, nch)
    return dict(kind=kind, ctx=ctx, n=n, nch=nch, src=src, dst=torch.zeros_like(src), codes=torch.zeros(n, **i32),
                o2o=torch.zeros(n, **i32), inv=torch.zeros(n, **i32))


def run(s):
    kind = s["kind"]
    if kind == "frame":
        ctx = s["ctx"]
        ctx.import_state(s["st"])
        ctx.substeps(s["p"], s["steps"])
        return ctx.export_state(DEV)
    if kind == "nodes":
        ctx, dt = s["ctx"], s["dt"]
        ctx.import_objects(s["vin"])
        ctx.grid_clear()
        ctx.p2g(dt)
        ctx.grid_update(dt, GRAVITY)
        vmax = ctx.max_vel_sqr()
        ctx.boundary(BOUNDARY_STICKY_BOX, PAD)
        ctx.g2p(dt)
        ctx.export_objects(s["vout"])
        return dict(fluid=s["tout"][0], solid=s["tout"][1], vmax=vmax)
    if kind == "batch":
        ctx = s["ctx"]
        ctx.state_load(s["saved"])
        ctx.graph_launch()
        return ctx.export_state(DEV)
    if kind == "grad":
        x = rollout(s["v0"], s["E"], s["nu"], s["sim"])
        g = torch.autograd.grad(x, (s["v0"], s["E"], s["nu"]), s["xbar"])
        return dict(x=x.detach(), v0=g[0], E=g[1], nu=g[2])
    s["ctx"].order_by_morton_code(LAYOUT_AOSOA32, s["nch"], s["n"], s["src"], s["dst"], 1, (0.0, 0.0, 0.0),
                                  (1.0, 1.0, 1.0), s["codes"], s["o2o"], s["inv"])
    return dict(dst=s["dst"], codes=s["codes"], order=s["o2o"], inverse=s["inv"])


# ------------------------------------------------------------------ work
def work(case):
    """Bytes and operations one pass cannot do without: per substep a solid particle's x, v, C, F and
    material word read and written once (196 B) or a fluid particle's x, v, C, J (132 B) and 32 B per
    active node (n / PPC of them, plus a rim); the import and the export read and write the caller's
    buffers once.  Operations: 27 nodes x 4 channels scattered with a multiply and an add per affine
    term, 27 x 3 gathered for v and C."""
    kind = case["kind"]
    if kind == "morton":
        return {"bytes": case["n"] * (8.0 * case["nch"] + 12.0), "flops": 20.0 * case["n"]}
    if kind == "frame":
        n, steps, nf = case["n"], case["steps"], case["fluid"] * case["n"]
        passes = 2.0 if case["transfer"] != "apic" else 1.0
    elif kind == "nodes":
        n, steps, nf, passes = case["n"], 1, case["fluid"] * case["n"], 1.0
    elif kind == "batch":
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        n, steps, nf, passes = case["scenes"] * mean, case["steps"], 0.0, 1.0
    else:  # forward, recomputation and the adjoint of every substep
        n, steps, nf, passes = case["scenes"] * case["n"], 4 * case["steps"], 0.0, 1.0
    sub = 196.0 * (n - nf) + 132.0 * nf + 32.0 * n / PPC
    flops = n * (27 * 4 * 2 + 297 * 2) * passes
    return {"bytes": sub * steps + 2 * 100.0 * n, "flops": flops * steps}


# ------------------------------------------------------------------ reference in 64 bits
def _polar(F):
    """Rotation of F (..., 3, 3), det F > 0, by Newton's iteration (differentiable)."""
    X = F
    for _ in range(9):
        r0, r1, r2 = X[:, 0], X[:, 1], X[:, 2]
        cof = torch.stack([torch.linalg.cross(r1, r2), torch.linalg.cross(r2, r0), torch.linalg.cross(r0, r1)], dim=1)
        det = (r0 * cof[:, 0]).sum(dim=1)
        X = 0.5 * (X + cof / det[:, None, None])
    return X


def _cof(F):
    r0, r1, r2 = F[:, 0], F[:, 1], F[:, 2]
    return torch.stack([torch.linalg.cross(r1, r2), torch.linalg.cross(r2, r0), torch.linalg.cross(r0, r1)], dim=1)


def _eig(B):
    """Eigenvalues (n, 3) and vectors (n, 3, 3) of symmetric B by cyclic Jacobi rotations."""
    A, V = B.clone(), torch.eye(3, device=B.device, dtype=B.dtype).expand_as(B).clone()
    for _ in range(7):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            apq = A[:, p, q]
            zero = apq == 0
            tau = (A[:, q, q] - A[:, p, p]) / torch.where(zero, torch.ones_like(apq), 2.0 * apq)
            t = torch.where(tau >= 0, 1.0, -1.0) / (tau.abs() + torch.sqrt(1.0 + tau * tau))
            t = torch.where(zero, torch.zeros_like(t), t)
            c = 1.0 / torch.sqrt(1.0 + t * t)
            s = t * c
            for M, axis in ((A, 1), (A, 2), (V, 2)):
                mp, mq = M.select(axis, p).clone(), M.select(axis, q).clone()
                M.select(axis, p).copy_(c[:, None] * mp - s[:, None] * mq)
                M.select(axis, q).copy_(s[:, None] * mp + c[:, None] * mq)
    return torch.stack([A[:, 0, 0], A[:, 1, 1], A[:, 2, 2]], dim=1), V


def _hencky(F):
    w, U = _eig(F @ F.transpose(1, 2))
    s = torch.sqrt(w)
    return s, torch.log(s), U


def _tau(F, mu, lam, solid, fiber):
    """Kirchhoff stress P F^T of the solid models; mu, lam (n,) or numbers."""
    mu, lam = (t[:, None, None] if isinstance(t, torch.Tensor) else t for t in (mu, lam))
    if solid == "sand":
        s, e, U = _hencky(F)
        d = 2.0 * mu * e + lam * e.sum(dim=1, keepdim=True)
        return (U * d[:, None, :]) @ U.transpose(1, 2)
    cof = _cof(F)
    J = (F[:, 0] * cof[:, 0]).sum(dim=1)[:, None, None]
    if solid == "nhk":
        P = mu * F + (lam * torch.log(J) - mu) / J * cof
    elif solid == "snhk":
        P = mu * F + (lam * (J - 1.0) - mu) * cof
    else:
        P = 2.0 * mu * (F - _polar(F)) + lam * (J - 1.0) * cof
    if fiber is not None:
        Fa = F @ fiber[:, :, None]
        P = P + 5.0 * mu * (1.0 - 1.0 / Fa.norm(dim=1, keepdim=True)) * (Fa @ fiber[:, None, :])
    return P @ F.transpose(1, 2)


def _drucker_prager(F, mu, lam):
    s, e, U = _hencky(F)
    sphi = math.sin(math.radians(35.0))
    alpha = math.sqrt(2.0 / 3.0) * 2.0 * sphi / (3.0 - sphi)
    tr = e.sum(dim=1, keepdim=True)
    eh = e - tr / 3.0
    nh = eh.norm(dim=1, keepdim=True)
    dg = nh + (3.0 * lam + 2.0 * mu) / (2.0 * mu) * tr * alpha
    ep = torch.where(tr >= 0, torch.zeros_like(e), e - dg / nh.clamp_min(1e-300) * eh)
    move = (tr >= 0) | (dg > 0)
    Fn = (U * (torch.exp(ep) / s)[:, None, :]) @ U.transpose(1, 2) @ F
    return torch.where(move[:, :, None], Fn, F)


class _Scene:
    """What the reference substep keeps besides the state: per-particle dx, dt, node offsets and widths."""

    def __init__(self, dx, dt, cells, base, m, vol, nodes, transfer="apic", solid="fcr", fiber=None, colliders=False,
                 beta=None, single=None):
        self.dx, self.dt, self.cells, self.base, self.m, self.vol, self.nodes = dx, dt, cells, base, m, vol, nodes
        self.transfer, self.solid, self.fiber, self.colliders, self.beta = transfer, solid, fiber, colliders, beta
        self.single = single  # (dx, cells) of a one-scene context, for colliders


def _collide(v, pos):
    d = pos @ torch.tensor(SLOPE[:3], device=v.device, dtype=v.dtype) - SLOPE[3]
    nrm = torch.tensor(SLOPE[:3], device=v.device, dtype=v.dtype)
    v = torch.where((d < 0)[:, None], v - (v @ nrm)[:, None] * nrm, v)
    r = (pos - torch.tensor(BALL[:3], device=v.device, dtype=v.dtype)).norm(dim=1) - BALL[3]
    return torch.where((r < 0)[:, None], torch.zeros_like(v), v)


def _substep(sc, x, v, C, F, J, mu, lam, sol, vmax=None):
    """One substep of all particles: x, v (n, 3), C (n, 3, 3), F (ns, 3, 3) of the solid ones (indices
    sol), J (nf,) of the others."""
    n, dev = x.shape[0], x.device
    one = lambda t: t[:, None] if isinstance(t, torch.Tensor) else t  # noqa: E731
    two = lambda t: t[:, None, None] if isinstance(t, torch.Tensor) else t  # noqa: E731
    dx, dt = one(sc.dx), one(sc.dt)
    X = x / dx
    low = torch.floor(X.detach() - 0.5)
    f = X - low
    w = [0.5 * (1.5 - f) ** 2, 0.75 - (f - 1.0) ** 2, 0.5 * (f - 0.5) ** 2]
    dw = [f - 1.5, -2.0 * (f - 1.0), f - 0.5]
    width = sc.cells + 8
    i0 = low.long() + 2
    flu = torch.ones(n, dtype=torch.bool, device=dev)
    flu[sol] = False
    flu = flu.nonzero()[:, 0]
    tau = torch.zeros(n, 3, 3, device=dev, dtype=x.dtype)
    if sol.numel():
        tau = tau.index_copy(0, sol, _tau(F, mu, lam, sc.solid, sc.fiber))
    if flu.numel():
        tau = tau.index_copy(0, flu, (BULK * J * (J - 1.0))[:, None, None] * torch.eye(3, device=dev, dtype=x.dtype))
    m, vol = one(sc.m), two(sc.vol)
    flip = sc.transfer != "apic"
    force = -two(sc.dt) * vol * tau
    stress = force * 4.0 / two(sc.dx) ** 2
    B = two(sc.m) * C

    def node(o):
        k = i0 + torch.tensor(o, device=dev)
        return sc.base + (k[:, 0] * width + k[:, 1]) * width + k[:, 2]

    offs = [(a, b, c) for a in range(3) for b in range(3) for c in range(3)]
    grid = torch.zeros(sc.nodes, 7 if flip else 4, device=dev, dtype=x.dtype)
    mass = (m * torch.ones_like(x[:, :1]))
    for o in offs:
        W = (w[o[0]][:, 0] * w[o[1]][:, 1] * w[o[2]][:, 2])[:, None]
        d = ((torch.tensor(o, device=dev, dtype=x.dtype) - f) * dx)[:, :, None]
        if sc.transfer == "flip":
            gw = torch.stack([dw[o[0]][:, 0] * w[o[1]][:, 1] * w[o[2]][:, 2], w[o[0]][:, 0] * dw[o[1]][:, 1] * w[o[2]][:, 2],
                              w[o[0]][:, 0] * w[o[1]][:, 1] * dw[o[2]][:, 2]], dim=1) / dx
            val = torch.cat([mass, m * v, (force @ gw[:, :, None])[:, :, 0]], dim=1)
        elif flip:
            val = torch.cat([mass, m * v + (B @ d)[:, :, 0], (stress @ d)[:, :, 0]], dim=1)
        else:
            val = torch.cat([mass, m * v + ((B + stress) @ d)[:, :, 0]], dim=1)
        grid = grid.index_add(0, node(o), W * val) if grid.requires_grad or x.requires_grad else grid.index_add_(0, node(o), W * val)
    gm = grid[:, :1]
    has = gm != 0
    inv = torch.where(has, 1.0 / torch.where(has, gm, torch.ones_like(gm)), torch.zeros_like(gm))
    gv = grid[:, 1:4] * inv
    # gravity and walls by scene: every particle's scene offsets name its nodes' scene
    gdt, ncell, off, wid = sc.node_dt, sc.node_cells, sc.node_base, sc.node_width
    acc = torch.tensor(GRAVITY, device=dev, dtype=x.dtype)[None, :] * gdt
    gs = grid[:, 4:7] * inv + gv + torch.where(has, acc, torch.zeros_like(acc)) if flip else None
    if not flip:
        gv = gv + torch.where(has, acc, torch.zeros_like(acc))
    bc = gs if flip else gv
    if vmax is not None:
        vmax.append(float((bc ** 2).sum(dim=1).max()))
    r = torch.arange(sc.nodes, device=dev) - off
    ix = torch.stack([r // (wid * wid), (r // wid) % wid, r % wid], dim=1) - 2
    wall = ((ix < PAD) | (ix > (ncell - PAD)[:, None])).any(dim=1, keepdim=True) if isinstance(ncell, torch.Tensor) \
        else ((ix < PAD) | (ix > ncell - PAD)).any(dim=1, keepdim=True)
    bc = torch.where(wall, torch.zeros_like(bc), bc)
    if sc.colliders:
        bc = torch.where(has, _collide(bc, ix.to(x.dtype) * sc.single[0]), bc)
    if flip:
        gs = bc
    else:
        gv = bc
    pv = torch.zeros_like(x)
    ps = torch.zeros_like(x)
    G = torch.zeros_like(C)
    for o in offs:
        W = (w[o[0]][:, 0] * w[o[1]][:, 1] * w[o[2]][:, 2])[:, None]
        at = node(o)
        a = gv[at]
        s = gs[at] if flip else a
        pv = pv + W * a
        if flip:
            ps = ps + W * s
        if sc.transfer == "flip":
            gw = torch.stack([dw[o[0]][:, 0] * w[o[1]][:, 1] * w[o[2]][:, 2], w[o[0]][:, 0] * dw[o[1]][:, 1] * w[o[2]][:, 2],
                              w[o[0]][:, 0] * w[o[1]][:, 1] * dw[o[2]][:, 2]], dim=1) / dx
            G = G + s[:, :, None] * gw[:, None, :]
        else:
            d = (torch.tensor(o, device=dev, dtype=x.dtype) - f) * dx
            G = G + (W * s)[:, :, None] * d[:, None, :] * (4.0 / two(sc.dx) ** 2)
    if flip:
        dv = v - pv
        vn = ps + 0.99 * dv
        xn = x + dt * (ps + (sc.beta[:, None] * 0.99 * dv if sc.transfer == "aflip" else 0.0))
    else:
        vn, xn = pv, x + dt * pv
    step = two(sc.dt) * G
    Fn, Jn = F, J
    if sol.numel():
        Fn = F + step[sol] @ F
        if sc.solid == "sand":
            Fn = _drucker_prager(Fn, mu, lam)
    if flu.numel():
        Jn = (1.0 + step[flu].diagonal(dim1=1, dim2=2).sum(dim=1)) * J
    return xn, vn, (C if sc.transfer == "flip" else G), Fn, Jn


def _lame(E, nu):
    return E / (2.0 * (1.0 + nu)), E * nu / ((1.0 + nu) * (1.0 - 2.0 * nu))


def _one_scene(dx, dt, cells, m, vol, **more):
    nodes = (cells + 8) ** 3
    sc = _Scene(dx, dt, cells, 0, m, vol, nodes, single=(dx, cells), **more)
    sc.node_dt, sc.node_cells, sc.node_base, sc.node_width = dt, cells, 0, cells + 8
    return sc


def _many_scenes(descs, mats, scene):
    d = dict(device=DEV, dtype=torch.float64)
    cells = torch.tensor([q["n_cells"] for q in descs], device=DEV)
    width = cells + 8
    size = width ** 3
    base = torch.cumsum(size, 0) - size
    of = torch.repeat_interleave(torch.arange(len(descs), device=DEV), size)
    s = scene.long()
    dx, dt = torch.tensor([q["dx"] for q in descs], **d), torch.tensor([q["dt"] for q in descs], **d)
    vol = torch.tensor([q["vol"] for q in mats], **d)
    sc = _Scene(dx[s], dt[s], cells[s], base[s], (RHO * vol)[s], vol[s], int(size.sum()))
    sc.node_dt, sc.node_cells, sc.node_base, sc.node_width = dt[of][:, None], cells[of], base[of], width[of]
    return sc


def _soa(t):
    return t.reshape(t.shape[0], -1).t().contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "morton":
        return None
    d = lambda t: t.double().t().contiguous()  # noqa: E731
    if kind in ("frame", "nodes"):
        cells, dt = case["cells"], _dt(case["cells"])
        if kind == "frame":
            st, dx, mats = _frame_inputs(case, seed)
            x, v, C, F9 = d(st["x"]), d(st["v"]), d(st["C"]).view(-1, 3, 3), d(st["F"]).view(-1, 3, 3)
            sol, flu = (st["mat"] == 1).nonzero()[:, 0], (st["mat"] == 0).nonzero()[:, 0]
            fiber = st["a"].double().t()[sol].contiguous() if "a" in st else None
            vol = mats[0]["vol"]
            sc = _one_scene(dx, dt, cells, RHO * vol, vol, transfer=case["transfer"], solid=case["solid"], fiber=fiber,
                            colliders=case["colliders"], beta=st["beta"].double() if "beta" in st else None)
            steps = case["steps"]
        else:
            objs, dx, mats = _nodes_inputs(case, seed)
            cat = lambda a, b: torch.cat([d(o[a:b]) for o in objs])  # noqa: E731
            x, v, C = cat(1, 4), cat(4, 7), cat(8, 17).view(-1, 3, 3)
            nf = objs[0].shape[1]
            F9 = torch.zeros_like(C)
            F9[:nf, 0, 0], F9[nf:] = objs[0][19].double(), d(objs[1][19:28]).view(-1, 3, 3)
            flu, sol = torch.arange(nf, device=DEV), torch.arange(nf, x.shape[0], device=DEV)
            sc = _one_scene(dx, dt, cells, cat(0, 1)[:, 0], cat(7, 8)[:, 0])
            steps = 1
        mu, lam = _lame(1e5, 0.3)
        F, J, vmax = F9[sol], F9[flu, 0, 0], []
        for _ in range(steps):
            x, v, C, F, J = _substep(sc, x, v, C, F, J, mu, lam, sol, vmax if kind == "nodes" else None)
        F9 = torch.zeros_like(C)
        F9[sol] = F
        F9[flu, 0, 0] = J
        if kind == "frame":
            return dict(x=_soa(x), v=_soa(v), C=_soa(C), F=_soa(F9))
        out = []
        for k, (o, sel) in enumerate(zip(objs, (flu, sol))):
            planes = o.double()
            planes[1:4], planes[4:7], planes[8:17] = _soa(x[sel]), _soa(v[sel]), _soa(C[sel])
            planes[19:] = J[None, :] if k == 0 else _soa(F)
            out.append(_tiles(planes, o.shape[0]))
        return dict(fluid=out[0], solid=out[1], vmax=vmax[0])
    if kind == "batch":
        st, descs, mats = _batch_inputs(case, seed)
        sc = _many_scenes(descs, mats, st["mat"])
        lame = torch.tensor([_lame(q["E"], q["nu"]) for q in mats], device=DEV, dtype=torch.float64)[st["mat"].long()]
        x, v, C, F = d(st["x"]), d(st["v"]), d(st["C"]).view(-1, 3, 3), d(st["F"]).view(-1, 3, 3)
        sol, J = torch.arange(x.shape[0], device=DEV), torch.zeros(0, device=DEV, dtype=torch.float64)
        for _ in range(case["steps"]):
            x, v, C, F, J = _substep(sc, x, v, C, F, J, lame[:, 0], lame[:, 1], sol)
        return dict(x=_soa(x), v=_soa(v), C=_soa(C), F=_soa(F))
    st, descs, mats, E, nu, xbar = _grad_inputs(case, seed)
    sc = _many_scenes(descs, mats, st["mat"])
    E = E.to(DEV).double().requires_grad_(True)
    nu = nu.to(DEV).double().requires_grad_(True)
    v0 = st["v"].double().requires_grad_(True)
    s = st["mat"].long()
    mu, lam = _lame(E, nu)
    mu, lam = mu[s], lam[s]
    x, v, C, F = d(st["x"]), v0.t(), d(st["C"]).view(-1, 3, 3), d(st["F"]).view(-1, 3, 3)
    x = x.requires_grad_(True)
    sol, J = torch.arange(x.shape[0], device=DEV), torch.zeros(0, device=DEV, dtype=torch.float64)

    def step(x, v, C, F, mu, lam):
        return _substep(sc, x, v, C, F, J, mu, lam, sol)[:4]

    for _ in range(case["steps"]):
        x, v, C, F = checkpoint(step, x, v, C, F, mu, lam, use_reentrant=False)
    g = torch.autograd.grad(x, (v0, E, nu), xbar.double().t())
    return dict(x=_soa(x.detach()), v0=g[0], E=g[1].cpu(), nu=g[2].cpu())
