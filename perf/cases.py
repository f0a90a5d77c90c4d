"""Timed workloads of the jbgpu library, each through its public Python entry points.

A case is a dict of plain values; ``prepare`` builds what a program holds before the call (a context with its world or
proxies, rays, a model), ``run`` is one pass as such a program calls it, ``work`` the bytes and operations the pass
cannot do without, ``tolerance`` and ``exact`` what its results may differ by and what they are in 64 bits.

Simulation results are compared exactly: a step's arithmetic and the order in which rows are solved are fixed (the
library promises the bits of a sequential solver given the reported order), so bodies, pairs, manifolds and hits are
the same whatever the launch shape.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "libgdx-jbullet_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "libgdx-jbullet_amd"))

import jbgpu  # noqa: E402
from jbgpu import scenes  # noqa: E402

DT = 1.0 / 60.0
BODY_STATIC = 1  # flag word of a fixed body
PILE_LAYERS = 20  # lattice layers a pile is dropped from


def listed():
    return [
        # a handful of objects, one step a frame, their state read back: the smallest world a game steps
        {"name": "boxes_27", "kind": "boxes", "side": 3, "steps": 1},
        # the 10 x 10 x 10 box grid over a plane, at rest, one step a frame
        {"name": "boxes_1000", "kind": "boxes", "side": 10, "steps": 1},
        # one room's worth of mixed convex debris, one step a frame, 20 solver iterations
        {"name": "pile_3000", "kind": "pile", "bodies": 3000, "iterations": 20, "steps": 1},
        # the large mixed pile, two substeps per state read-back
        {"name": "pile_100000", "kind": "pile", "bodies": 100_000, "iterations": 20, "steps": 2},
        # many small independent worlds (agents trained in parallel): eight substeps per read-back, captured steps
        {"name": "towers_4096", "kind": "towers", "worlds": 4096, "graph": True, "steps": 8},
        # hanging and swinging chains with boxes falling on them: constraints beside contacts
        {"name": "chains_64", "kind": "chains", "side": 8, "links": 8, "drops": 200, "steps": 1},
        # the broadphase alone behind another engine, boxes resident on the device, pair keys read back
        {"name": "pairs_1000000_dbvt", "kind": "pairs", "boxes": 1_000_000, "mode": "dbvt", "device": True},
        # the broadphase alone for a host-side engine: boxes uploaded, pairs and their changes read back
        {"name": "pairs_20011_sap32", "kind": "pairs", "boxes": 20_011, "mode": "sap32", "device": False},
        # closest-hit rays of sensors over a pile, rays and results on the device
        {"name": "rays_262144", "kind": "rays", "bodies": 20_000, "rays": 262_144},
        # convex sweeps (character and camera probes) through a pile, host arrays
        {"name": "sweeps_4099", "kind": "sweeps", "bodies": 5000, "queries": 4099},
        # narrowphase and solver as plugins of a host-side world: dispatch its pair cache, then solve its islands
        {"name": "seams_3000", "kind": "seams", "bodies": 3000, "iterations": 10},
        # one full-batch gradient of the warm-start model (forward and backward)
        {"name": "mlp_grad_65536", "kind": "mlp", "contacts": 65_536, "grad": True},
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["boxes", "pile", "pile", "towers", "chains", "pairs", "pairs", "rays", "sweeps", "seams", "mlp"])
    if kind == "boxes":
        return {"kind": kind, "side": rng.randint(2, 16), "steps": rng.randint(1, 4)}
    if kind == "pile":
        return {"kind": kind, "bodies": _spread(rng, 300, 60_000), "iterations": rng.choice([4, 10, 20]),
                "steps": rng.randint(1, 2)}
    if kind == "towers":
        return {"kind": kind, "worlds": _spread(rng, 8, 3000), "graph": rng.random() < 0.6, "steps": rng.randint(1, 8)}
    if kind == "chains":
        return {"kind": kind, "side": rng.randint(2, 14), "links": rng.randint(3, 12), "drops": rng.randint(20, 400),
                "steps": rng.randint(1, 3)}
    if kind == "pairs":
        return {"kind": kind, "boxes": _spread(rng, 500, 900_000), "mode": rng.choice(["dbvt", "sap32", "sap16", "simple"]),
                "device": rng.random() < 0.5}
    if kind == "rays":
        return {"kind": kind, "bodies": _spread(rng, 1000, 30_000), "rays": _spread(rng, 64, 250_000)}
    if kind == "sweeps":
        return {"kind": kind, "bodies": _spread(rng, 1000, 20_000), "queries": _spread(rng, 16, 8_000)}
    if kind == "seams":
        return {"kind": kind, "bodies": _spread(rng, 300, 6000), "iterations": rng.choice([4, 10, 20])}
    return {"kind": kind, "contacts": _spread(rng, 100, 200_000), "grad": rng.random() < 0.5}


# ---- scenes -----------------------------------------------------------------------------------------------------


class _Palette:
    """Shapes that many bodies share, each with its density: records, masses and inertias are made once per shape."""

    def __init__(self, entries, verts=None):
        self.verts = np.zeros((1, 3), np.float32) if verts is None else np.asarray(verts, np.float32)
        self.rec = np.stack([jbgpu.make_shape(t, (list(p) + [0.0] * 4)[:4], self.verts) for t, p, _ in entries])
        self.mass = np.array([m for _, _, m in entries], np.float32)
        self.inertia = np.stack([jbgpu.shape_inertia(r, float(m), self.verts) if m else np.zeros(3, np.float32)
                                 for r, m in zip(self.rec, self.mass)])

    def bodies(self, shape, basis, origin):
        n = len(shape)
        b = np.zeros((n, jbgpu.BODY_WORDS), np.float32)
        b[:, 0:9] = basis
        b[:, 9:12] = origin
        one, zero = np.float32(1.0), np.float32(0.0)
        with np.errstate(divide="ignore", invalid="ignore"):
            inv = np.where(self.mass != 0, one / self.mass, zero)
            inv_inertia = np.where(self.inertia != 0, one / self.inertia, zero)
            gravity = np.where(self.mass[:, None] != 0, scenes.GRAVITY[None, :] * (one / inv)[:, None], zero)
        b[:, 18] = inv[shape]
        b[:, 19:22] = inv_inertia[shape]
        b[:, 22:25] = gravity[shape]
        b[:, 25] = 0.5
        words = b.view(np.int32)
        words[:, 27] = shape
        words[:, 28] = np.where(self.mass[shape] != 0, 0, BODY_STATIC)
        words[:, 29] = scenes.ACTIVE_TAG
        return b


def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    x, y, z, w = q.T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1).astype(np.float32)


def _mixed_palette(rng, walls):
    """Floor, walls, then 200 dynamic shapes of the mixed pile's sizes: 40% spheres (r log-uniform 0.1-1), 30% boxes
    (half extents U(0.1, 1)), 15% capsules, 15% hulls of 16-32 points; density U(500, 2000)."""
    entries = [(scenes.PLANE, [0.0, 1.0, 0.0, 0.0], 0.0)] + [(scenes.BOX, list(h), 0.0) for h in walls]
    verts, nv = [], 0
    for k in range(200):
        rho = rng.uniform(500, 2000)
        if k < 80:
            r = float(np.exp(rng.uniform(np.log(0.1), 0.0)))
            entries.append((scenes.SPHERE, [r], rho * 4 / 3 * np.pi * r ** 3))
        elif k < 140:
            h = rng.uniform(0.1, 1.0, 3)
            entries.append((scenes.BOX, list(h), rho * 8 * h.prod()))
        elif k < 170:
            r, height = float(np.exp(rng.uniform(np.log(0.1), np.log(0.5)))), float(rng.uniform(0.2, 2.0))
            entries.append((scenes.CAPSULE, [r, height], rho * (np.pi * r * r * height + 4 / 3 * np.pi * r ** 3)))
        else:
            axes, m = rng.uniform(0.1, 1.0, 3), int(rng.integers(16, 33))
            d = rng.normal(size=(m, 3))
            verts.append(d / np.linalg.norm(d, axis=1, keepdims=True) * axes)
            entries.append((scenes.HULL, [nv, m], rho * 4 / 3 * np.pi * axes.prod()))
            nv += m
    return _Palette(entries, np.concatenate(verts).astype(np.float32))


def _pile(seed, n, iterations, settle):
    """n mixed convex bodies dropped from a 2.2 m lattice into a walled bin, stepped until they lie in a pile."""
    rng = np.random.default_rng(seed)
    per = max(2, int(math.ceil(math.sqrt(n / PILE_LAYERS))))
    half, t, hw = 1.1 * per + 1.1, 1.0, 15.0
    walls = [(t, hw, half + t), (t, hw, half + t), (half + t, hw, t), (half + t, hw, t)]
    pal = _mixed_palette(rng, walls)
    i = np.arange(n)
    lattice = np.stack([(i % per - (per - 1) / 2.0) * 2.2, 2.0 + (i // (per * per)) * 2.2,
                        ((i // per) % per - (per - 1) / 2.0) * 2.2], 1) + rng.uniform(-0.1, 0.1, (n, 3))
    fixed = np.array([[0, 0, 0], [half + t, hw, 0], [-half - t, hw, 0], [0, hw, half + t], [0, hw, -half - t]])
    shape = np.concatenate([np.arange(5), 5 + rng.integers(0, 200, n)]).astype(np.int32)
    basis = np.concatenate([np.tile(scenes.IDENT, (5, 1)), _rotations(rng, n)])
    ctx = jbgpu.Context(num_iterations=iterations)
    ctx.world_create(pal.rec, pal.verts, pal.bodies(shape, basis, np.concatenate([fixed, lattice]).astype(np.float32)))
    ctx.step(DT, settle)
    return ctx, pal, half


def _boxes(seed, side):
    """A side^3 grid of 1 m boxes with random yaw just above a plane, stepped to rest."""
    rng = np.random.default_rng(seed)
    n = side ** 3
    pal = _Palette([(scenes.PLANE, [0.0, 1.0, 0.0, 0.0], 0.0), (scenes.BOX, [0.5, 0.5, 0.5], 1.0)])
    i = np.arange(n)
    pos = np.stack([(i % side) * 1.2, 0.55 + (i // (side * side)) * 1.2, ((i // side) % side) * 1.2], 1)
    yaw = rng.uniform(0, 2 * np.pi, n)
    basis = np.zeros((n + 1, 9), np.float32)
    basis[:, 4] = 1.0
    basis[1:, 0], basis[1:, 2], basis[1:, 6], basis[1:, 8] = np.cos(yaw), np.sin(yaw), -np.sin(yaw), np.cos(yaw)
    basis[0, 0] = basis[0, 8] = 1.0
    origin = np.concatenate([np.zeros((1, 3)), pos + rng.uniform(-0.05, 0.05, (n, 3))]).astype(np.float32)
    ctx = jbgpu.Context(num_iterations=10)
    ctx.world_create(pal.rec, pal.verts, pal.bodies(np.minimum(np.arange(n + 1), 1), basis, origin))
    ctx.step(DT, 150)
    return ctx


def _towers(seed, worlds, graph):
    """Independent worlds of 16-512 spheres and boxes (log-uniform) in towers of 4-20 on a 3 m grid."""
    rng = np.random.default_rng(seed)
    entries = [(scenes.PLANE, [0.0, 1.0, 0.0, 0.0], 0.0)]
    ext = [0.0]
    for k in range(140):
        rho = rng.uniform(500, 2000)
        if k < 80:
            r = float(np.exp(rng.uniform(np.log(0.1), 0.0)))
            entries.append((scenes.SPHERE, [r], rho * 4 / 3 * np.pi * r ** 3))
            ext.append(r)
        else:
            h = rng.uniform(0.1, 1.0, 3)
            entries.append((scenes.BOX, list(h), rho * 8 * h.prod()))
            ext.append(float(h[1]))
    pal, ext = _Palette(entries), np.array(ext)
    # world sizes spread evenly over the logarithm of their range, the same for every seed
    count = np.floor(np.exp(np.log(16) + np.log(513 / 16) * (np.arange(worlds) * 0.6180339887 % 1.0))).astype(np.int64)
    total = int(count.sum())
    world = np.repeat(np.arange(worlds), count)
    place = np.arange(total) - np.repeat(np.cumsum(count) - count, count)  # number inside its world
    # tower heights per world: the j-th boundary of world w is the sum of its first j random heights
    heights = rng.integers(4, 21, (worlds, 128))
    bound = np.cumsum(heights, 1)
    tower = np.empty(total, np.int64)
    for w0 in range(0, worlds, 256):
        sel = slice(int(count[:w0].sum()), int(count[:w0 + 256].sum()))
        tower[sel] = (bound[world[sel]] <= place[sel][:, None]).sum(1)
    base = np.where(tower > 0, bound[world, np.maximum(tower - 1, 0)], 0)
    shape = 1 + rng.integers(0, 140, total)
    size = 2 * ext[shape] + 0.01
    top = np.cumsum(size)
    before = top - size  # height of everything before, in all towers; its value at the tower's first body is the floor
    y = before - before[np.arange(total) - (place - base)] + ext[shape] + 0.01
    origin = np.stack([(tower % 8) * 3.0, y, (tower // 8) * 3.0], 1)
    # each world's floor comes first among its bodies
    at = np.arange(total) + world + 1
    n = total + worlds
    all_shape, all_origin, all_world = np.zeros(n, np.int32), np.zeros((n, 3), np.float32), np.empty(n, np.int32)
    all_shape[at], all_origin[at], all_world[at] = shape, origin, world
    all_world[np.cumsum(count) - count + np.arange(worlds)] = np.arange(worlds)
    ctx = jbgpu.Context(num_iterations=10)
    ctx.world_create(pal.rec, pal.verts, pal.bodies(all_shape, np.tile(scenes.IDENT, (n, 1)), all_origin), all_world)
    ctx.solver_set_world_blocks(512, 128, False)
    ctx.step(DT, 100)
    if graph:
        ctx.set_step_graph(True)
        ctx.step(DT, 50)
    return ctx


def _chains(seed, side, links, drops):
    sc = scenes.chains(seed=seed, nx=side, nz=side, links=links, drops=drops)
    shapes, verts, bodies = scenes.build_records(sc, jbgpu)
    bodies[:, 12:15] = sc.meta["velocity"]
    ctx = jbgpu.Context(num_iterations=10)
    ctx.world_create(shapes, verts, bodies)
    ctx.add_point2point(*sc.meta["joints"])
    ctx.step(DT, 120)
    return ctx


def _cloud(seed, n, frames):
    """AABB frames on the device: centres in a cube of one per (10 m)^3, lognormal half extents, N(0, 5 m/s)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    side = 10.0 * n ** (1.0 / 3.0)
    c = torch.rand(n, 3, generator=g, device="cuda") * side
    h = torch.exp(0.7 * torch.randn(n, 3, generator=g, device="cuda"))
    v = 5.0 * torch.randn(n, 3, generator=g, device="cuda")
    out = []
    for _ in range(frames):
        out.append(torch.cat([c - h, c + h], 1).contiguous())
        c = c + v * DT
    return out, side


_MODES = {"dbvt": jbgpu.BP_DBVT, "sap16": jbgpu.BP_SAP16, "sap32": jbgpu.BP_SAP32, "simple": jbgpu.BP_SIMPLE}
_MLP_SIZES = [(64, 16), (64,), (64, 64), (64,), (64, 64), (64,), (3, 64), (3,)]


def _mlp_data(seed, n):
    """A He-uniform model, its normalisation, and contacts of that normalisation's spread."""
    rng = np.random.default_rng(seed)
    parts = [rng.uniform(-1, 1, s) * math.sqrt(6.0 / s[1]) if len(s) == 2 else rng.normal(0, 0.1, s) for s in _MLP_SIZES]
    params = np.concatenate([p.reshape(-1) for p in parts]).astype(np.float32)
    mean, std, so, mo = rng.normal(0, 1, 16), rng.uniform(0.5, 2.0, 16), rng.uniform(0.5, 3.0, 3), rng.normal(0, 1, 3)
    norm = np.concatenate([mean, 1.0 / std, so, mo]).astype(np.float32)
    x = (rng.standard_normal((n, 16), dtype=np.float32) * std.astype(np.float32) + mean.astype(np.float32))
    t = (rng.standard_normal((n, 3), dtype=np.float32) * so.astype(np.float32) + mo.astype(np.float32))
    return params, norm, x.astype(np.float32), t.astype(np.float32)


def _islands(bodies, keys, man):
    """Manifolds with points and a dynamic body, as one list: islands share no dynamic body, so the host may record
    them in any grouping."""
    static = bodies[:, 28].view(np.int32) & 1
    lo = (keys >> np.uint64(32)).astype(np.int64) - 1
    hi = (keys & np.uint64(0xffffffff)).astype(np.int64) - 1
    return np.nonzero((man[:, 0].view(np.int32) > 0) & ((static[lo] & static[hi]) == 0))[0].astype(np.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "boxes":
        return {"case": case, "ctx": _boxes(seed, case["side"])}
    if kind == "pile":
        return {"case": case, "ctx": _pile(seed, case["bodies"], case["iterations"], 260)[0]}
    if kind == "towers":
        return {"case": case, "ctx": _towers(seed, case["worlds"], case["graph"])}
    if kind == "chains":
        return {"case": case, "ctx": _chains(seed, case["side"], case["links"], case["drops"])}
    if kind == "pairs":
        n = case["boxes"]
        frames, side = _cloud(seed, n, 9)
        ctx = jbgpu.Context(bp_mode=_MODES[case["mode"]], world_min=(-0.1 * side - 20,) * 3, world_max=(1.1 * side + 20,) * 3)
        ctx.bp_create_proxies(frames[0].cpu().numpy())
        if not case["device"]:
            frames = [f.cpu().numpy() for f in frames]
        st = {"case": case, "ctx": ctx, "frames": frames[1:], "at": 0}
        for k in ("keys",) if case["device"] else ("keys", "added", "removed"):  # the program's own tables
            st[k] = np.zeros(n // 4 + 256, np.int64)
            st["n_" + k] = 0
        torch.cuda.synchronize()
        for _ in range(2):  # the pair cache a running program holds
            _set_frame(st)
            ctx.bp_calculate_overlapping_pairs()
        return st
    if kind == "rays":
        ctx, _, half = _pile(seed, case["bodies"], 10, 150)
        g = torch.Generator(device="cuda").manual_seed(seed + 1)
        n = case["rays"]
        lo, span = torch.tensor([-half, 0.0, -half], device="cuda"), torch.tensor([2 * half, 30.0, 2 * half], device="cuda")
        a = lo + span * torch.rand(n, 3, generator=g, device="cuda")
        b = lo + span * torch.rand(n, 3, generator=g, device="cuda")
        down = torch.rand(n, generator=g, device="cuda") < 0.5  # half of them look straight down
        b[down, 0], b[down, 2] = a[down, 0], a[down, 2]
        a[down, 1], b[down, 1] = 30.0, -1.0
        st = {"case": case, "ctx": ctx, "from": a.contiguous(), "to": b.contiguous(),
              "obj": torch.empty(n, dtype=torch.int32, device="cuda"), "fraction": torch.empty(n, device="cuda"),
              "normal": torch.empty(n, 3, device="cuda"), "point": torch.empty(n, 3, device="cuda")}
        torch.cuda.synchronize()
        return st
    if kind == "sweeps":
        ctx, _, half = _pile(seed, case["bodies"], 10, 150)
        rng = np.random.default_rng(seed + 1)
        n = case["queries"]
        basis = _rotations(rng, n)
        a = np.stack([rng.uniform(-half, half, n), rng.uniform(0.5, 25.0, n), rng.uniform(-half, half, n)], 1)
        b = a + rng.normal(0.0, 5.0, (n, 3))
        shape = jbgpu.make_shape(scenes.CAPSULE, [0.4, 1.0, 0.0, 0.0])
        return {"case": case, "ctx": ctx, "shape": shape, "from": np.concatenate([basis, a], 1).astype(np.float32),
                "to": np.concatenate([basis, b], 1).astype(np.float32)}
    if kind == "seams":
        ctx, _, _ = _pile(seed, case["bodies"], case["iterations"], 260)
        ctx.step_until(1, DT)  # the host's own predict, AABBs and pair cache: four pairs a body, lowest keys first
        keys, man = ctx.pairs()
        n = 4 * case["bodies"]
        if len(keys) < n:
            raise RuntimeError(f"the pile has {len(keys)} pairs, fewer than {n}")
        keys, man = keys[:n].copy(), man[:n].copy()
        return {"case": case, "ctx": ctx, "keys": keys, "man": man, "bodies": ctx.bodies()}
    params, norm, x, t = _mlp_data(seed, case["contacts"])
    ctx = jbgpu.Context()
    ctx.mlp_set_params(params, norm)
    return {"case": case, "ctx": ctx, "x": x, "t": t}


def _set_frame(st):
    f = st["frames"][st["at"] % len(st["frames"])]
    st["at"] += 1
    if st["case"]["device"]:
        st["ctx"].bp_set_aabbs_device(f.data_ptr(), st["case"]["boxes"])
    else:
        st["ctx"].bp_set_aabbs(f)


def _keep(st, name, keys):
    """The keys in the program's table of that name: as many as there are, then zeros."""
    table, n = st[name], len(keys)
    table[:n] = keys.view(np.int64)
    table[n:st["n_" + name]] = 0
    st["n_" + name] = n
    return table


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind in ("boxes", "pile", "towers", "chains"):
        ctx.step(DT, case["steps"])
        return ctx.bodies()
    if kind == "pairs":
        _set_frame(st)
        ctx.bp_calculate_overlapping_pairs()
        out = {"keys": _keep(st, "keys", ctx.bp_pairs())}
        if not case["device"]:
            added, removed = ctx.bp_pair_deltas()
            out.update(added=_keep(st, "added", added), removed=_keep(st, "removed", removed))
        return out
    if kind == "rays":
        ctx.ray_test_device(case["rays"], st["from"].data_ptr(), st["to"].data_ptr(), st["obj"].data_ptr(),
                            st["fraction"].data_ptr(), st["normal"].data_ptr(), st["point"].data_ptr())
        return {k: st[k] for k in ("obj", "fraction", "normal", "point")}
    if kind == "sweeps":
        obj, fraction, normal, point = ctx.convex_sweep(st["shape"], st["from"], st["to"])
        return {"obj": obj, "fraction": fraction, "normal": normal, "point": point}
    if kind == "seams":
        ctx.set_bodies(st["bodies"])
        man = ctx.np_dispatch(st["keys"], st["man"])
        ctx.solver_prepare(len(st["bodies"]), len(man))
        ctx.solver_add_island(_islands(st["bodies"], st["keys"], man))
        ctx.solver_all_solved(DT)
        return {"bodies": ctx.bodies(), "manifolds": ctx.pairs()[1]}
    if case["grad"]:
        grad, loss = ctx.mlp_grad(st["x"], st["t"])
        return {"grad": grad, "loss": loss}
    return ctx.mlp_infer(st["x"])


# ---- what a pass cannot do without --------------------------------------------------------------------------------
# Bytes per unit (32-bit records, each read and written once): predict 208, AABB 88, proxy 128, integrate 156 and state
# read-back 128 per body; a pair 1056 (bodies, shapes, manifold); a contact's solver set-up 552; a solver row 180 per
# sweep, three rows per contact.  Pairs and contacts per body are the settled scenes' own.


def _step_bytes(n, pairs, contacts, iterations):
    return n * (208 + 88 + 128 + 156) + n * pairs * 1064 + n * contacts * (552 + 540 * iterations)


def work(case):
    kind = case["kind"]
    if kind == "boxes":
        n = case["side"] ** 3 + 1
        return {"bytes": case["steps"] * _step_bytes(n, 5.0, 6.0, 10) + 128 * n, "flops": 0}
    if kind == "pile":
        n = case["bodies"] + 5
        return {"bytes": case["steps"] * _step_bytes(n, 9.0, 3.5, case["iterations"]) + 128 * n, "flops": 0}
    if kind == "towers":
        n = case["worlds"] * 144
        return {"bytes": case["steps"] * _step_bytes(n, 2.3, 1.8, 10) + 128 * n, "flops": 0}
    if kind == "chains":
        n = case["side"] ** 2 * case["links"] + case["drops"] + 1
        return {"bytes": case["steps"] * (_step_bytes(n, 4.0, 2.0, 10) + 400 * 10 * n) + 128 * n, "flops": 0}
    if kind == "pairs":
        return {"bytes": 128 * case["boxes"] + 16 * 0.08 * case["boxes"], "flops": 0}
    if kind == "rays":
        return {"bytes": 56 * case["rays"] + 200 * case["bodies"], "flops": 0}
    if kind == "sweeps":
        return {"bytes": 128 * case["queries"] + 200 * case["bodies"], "flops": 0}
    if kind == "seams":
        n = case["bodies"] + 5
        return {"bytes": n * 128 * 2 + n * 4.0 * (2 * 528 + 1064) + n * 2.0 * (552 + 540 * case["iterations"]), "flops": 0}
    flop = 2 * (16 * 64 + 64 * 64 + 64 * 64 + 64 * 3) * case["contacts"]
    return {"bytes": 76 * case["contacts"], "flops": 3 * flop if case["grad"] else flop}


def tolerance(case):
    if case["kind"] != "mlp":
        return "exact"
    # bf16 operands with 32-bit sums: four times the largest difference seen between 32-bit sums in another order and
    # 64-bit sums of the same rounded operands (a hidden activation near a rounding boundary changes by one bf16 step)
    return {"rel": 3e-4, "max": 0.05}


def exact(case, seed):
    """The unrounded model in 64 bits; simulation results have no closed form."""
    if case["kind"] != "mlp":
        return None
    params, norm, x, t = _mlp_data(seed, case["contacts"])
    p, o = [], 0
    for s in _MLP_SIZES:
        k = int(np.prod(s))
        p.append(params[o:o + k].astype(np.float64).reshape(s))
        o += k
    nm = norm.astype(np.float64)
    h = [(x.astype(np.float64) - nm[:16]) * nm[16:32]]
    z = []
    for k in range(3):
        z.append(h[-1] @ p[2 * k].T + p[2 * k + 1])
        h.append(np.maximum(z[-1], 0.0))
    y = h[3] @ p[6].T + p[7]
    if not case["grad"]:
        return y * nm[32:35] + nm[35:38]
    d = y - (t.astype(np.float64) - nm[35:38]) / nm[32:35]
    g = 2.0 * d / d.size
    parts = [g.sum(0), g.T @ h[3]]
    for k in (2, 1, 0):
        g = np.where(z[k] > 0, g @ p[2 * k + 2], 0.0)
        parts += [g.sum(0), g.T @ h[k]]
    return {"grad": np.concatenate([q.reshape(-1) for q in parts[::-1]]), "loss": float(np.mean(d * d))}
