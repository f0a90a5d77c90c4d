"""GPU parity of the contact sweeps where their launch form changes: all sweeps of a solve in one launch, groups of 16
slots of one colour at a time, against one launch per colour (a colour past a body's 64-bit colour mask, a body
flagged static that has a mass).  Bit for bit against the oracle fed the device's order."""
import numpy as np
import pytest

import jbgpu
import pyoracle
from jbgpu import scenes
from test_gpu_parity import _compare_world, _sync_and_step, _world_pair

pytestmark = pytest.mark.gpu


def _floor(name):
    b = scenes._Builder(name)
    b.body(b.shape(scenes.PLANE, [0.0, 1.0, 0.0, 0.0]), scenes.IDENT, np.zeros(3, np.float32), 0.0)
    return b


def _separate(n):
    """n boxes resting on the floor, none touching another: n slots of one colour."""
    b = _floor("separate")
    box = b.shape(scenes.BOX, [0.5, 0.5, 0.5])
    for i in range(n):
        b.body(box, scenes.IDENT, np.array([2.0 * (i % 8), 0.499, 2.0 * (i // 8)], np.float32), 1.0)
    return b.done(dt=1 / 60, iterations=10)


def _hub(m):
    """A plate lying on m boxes: the plate has one slot in each of m colours."""
    b = _floor("hub")
    box = b.shape(scenes.BOX, [0.25, 0.25, 0.25])
    side = int(np.ceil(np.sqrt(m)))
    plate = b.shape(scenes.BOX, [0.5 * side + 0.5, 0.2, 0.5 * side + 0.5])
    mid = (side - 1) / 2.0
    b.body(plate, scenes.IDENT, np.array([0.0, 0.697, 0.0], np.float32), 20.0)
    for i in range(m):
        b.body(box, scenes.IDENT, np.array([i % side - mid, 0.249, i // side - mid], np.float32), 1.0)
    return b.done(dt=1 / 60, iterations=10)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 33])
def test_one_colour_group_edges(n):
    ctx, orc = _world_pair(_separate(n))
    for step in range(20):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"separate {n} step {step}")
    assert ctx.stats()["colors"] == 1 and ctx.stats()["manifolds"] == n
    ctx.close()


@pytest.mark.parametrize("m,tail", [(5, 0), (60, 0), (72, 0), (72, 1024), (80, 4)])
def test_body_with_many_slots(m, tail):
    """Up to 64 colours the sweeps are one launch, past them one launch per colour (with and without the tail's)."""
    ctx, orc = _world_pair(_hub(m))
    ctx.solver_set_tail(tail)
    most = 0
    for step in range(12):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"hub {m} step {step}")
        most = max(most, ctx.stats()["colors"])
    print(f"[hub {m}] most colours {most}", flush=True)
    assert most >= m and (most > 64) == (m > 64)
    ctx.close()


def test_tolerance_mode_past_64_colours():
    ctx, orc = _world_pair(_hub(70))
    ctx.solver_set_params(tolerance=1e-3, max_iterations=40, num_iterations=10)
    orc.set_solver(jbgpu.ORDER_EXPLICIT, 1e-3, 40, 10)
    for step in range(6):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"hub tolerance step {step}")
        assert ctx.stats()["iterations"] == orc.stats()["iterations"]
    ctx.close()


def test_static_flag_with_mass_steps():
    """A static-flagged box that has a mass, with one box lying on it: one slot touches it, as the oracle solves it."""
    b = _floor("odd")
    box = b.shape(scenes.BOX, [0.5, 0.5, 0.5])
    b.body(box, scenes.IDENT, np.array([0.0, 0.5, 0.0], np.float32), 1.0)
    b.body(box, scenes.IDENT, np.array([0.0, 1.498, 0.0], np.float32), 1.0)
    sc = b.done(dt=1 / 60, iterations=10)
    shapes, verts, bodies = scenes.build_records(sc, jbgpu)
    bodies.view(np.int32)[1, 28] = 1
    ctx = jbgpu.Context(num_iterations=10)
    ctx.world_create(shapes, verts, bodies)
    orc = pyoracle.World(shapes, verts, bodies, iterations=10, order=jbgpu.ORDER_EXPLICIT)
    for step in range(10):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"static flag step {step}")
    assert ctx.stats()["manifolds"] == 1
    ctx.close()


def test_island_list_with_a_static_pair():
    """A caller's island list that holds a pair of static boxes: that slot is ordered by nothing but its own
    impulses; the dynamic box's solve is the one without it."""
    b = _floor("static pair")
    box = b.shape(scenes.BOX, [0.5, 0.5, 0.5])
    b.body(box, scenes.IDENT, np.array([0.0, 0.5, 0.0], np.float32), 0.0)
    b.body(box, scenes.IDENT, np.array([0.9, 0.5, 0.0], np.float32), 0.0)
    b.body(box, scenes.IDENT, np.array([0.0, 1.498, 0.0], np.float32), 1.0)
    shapes, verts, bodies = scenes.build_records(b.done(dt=1 / 60, iterations=10), jbgpu)
    keys = np.array([(2 << 32) | 3, (2 << 32) | 4], np.uint64)
    got = []
    for islands in ([1], [0, 1]):
        ctx = jbgpu.Context(num_iterations=10)
        ctx.world_create(shapes, verts, bodies)
        rec = np.zeros((2, jbgpu.MANIFOLD_WORDS), np.float32)
        rec.view(np.int32)[:, 1:4] = [[1, 2, 2], [1, 3, 2]]  # bodies, convex-convex
        man = ctx.np_dispatch(keys, rec)
        assert (man[:, 0].view(np.int32) > 0).all()
        ctx.solver_prepare(len(bodies), 2)
        ctx.solver_add_island(islands)
        ctx.solver_all_solved()
        got.append((ctx.bodies(), ctx.pairs()[1][1]))
        ctx.close()
    assert np.array_equal(got[0][0].view(np.uint32), got[1][0].view(np.uint32))
    assert np.array_equal(got[0][1].view(np.uint32), got[1][1].view(np.uint32))


@pytest.mark.parametrize("n", [1, 3, 64, 65, 16383, 16384, 16385])
def test_ray_counts_around_the_lane_split(n):
    """A ray's result does not depend on how many rays are asked for: a wave per ray below 16,384 rays, half a wave
    from there on; long rays along a row of boxes and the floor (many candidates, out of their lanes' share)."""
    b = _floor("row")
    box = b.shape(scenes.BOX, [0.3, 0.3, 0.3])
    for i in range(700):
        b.body(box, scenes.IDENT, np.array([float(i), 0.5, 0.0], np.float32), 1.0)
    shapes, verts, bodies = scenes.build_records(b.done(dt=1 / 60, iterations=10), jbgpu)
    ctx = jbgpu.Context()
    ctx.world_create(shapes, verts, bodies)
    rng = np.random.default_rng(3)
    m = 40  # distinct rays: along the whole row (700 candidates), along parts of it, straight down, past everything
    frm = np.stack([rng.uniform(-5, 705, m), rng.uniform(0.3, 3.0, m), rng.uniform(-0.2, 0.2, m)], 1)
    to = np.stack([rng.uniform(-5, 705, m), rng.uniform(-1.0, 0.7, m), rng.uniform(-0.2, 0.2, m)], 1)
    frm[0], to[0] = [-5.0, 0.75, 0.25], [705.0, 0.79, 0.28]  # above every box, inside their margins' AABBs
    to[1:10, [0, 2]] = frm[1:10, [0, 2]]
    frm[10], to[10] = [0.0, 50.0, 0.0], [10.0, 60.0, 0.0]
    frm, to = frm.astype(np.float32), to.astype(np.float32)
    orc = pyoracle.World(shapes, verts, bodies, iterations=10, order=0)
    want = orc.ray_test(frm, to)
    pick = np.arange(n) % m
    got = ctx.ray_test(frm[pick], to[pick])
    for g, w in zip(got, want):
        assert np.array_equal(np.asarray(g).view(np.uint32), np.asarray(w)[pick].view(np.uint32))
    ctx.close()


@pytest.mark.parametrize("n", [1023, 1025, 5119, 5120])
def test_small_step_limits(n):
    """n boxes at rest and the floor on both sides of a thousand manifolds and of the bodies the one-launch solve order
    holds (5120 with the floor)."""
    ctx, orc = _world_pair(_separate(n))
    for step in range(2):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"separate {n} step {step}")
    assert ctx.stats()["manifolds"] == n
    ctx.close()


def test_more_manifolds_than_the_small_order_holds():
    """4400 boxes stacked two and two on a row of plates: over 8192 manifolds among few bodies, then fewer again."""
    b = _floor("stacks")
    box = b.shape(scenes.BOX, [0.5, 0.5, 0.5])
    side = 16
    for k in range(side * side * 17):  # a close-packed block: about three manifolds a box
        x, z, y = k % side, (k // side) % side, k // (side * side)
        b.body(box, scenes.IDENT, np.array([0.999 * x, 0.499 + 0.998 * y, 0.999 * z], np.float32), 1.0)
    ctx, orc = _world_pair(b.done(dt=1 / 60, iterations=4), iterations=4)
    seen = 0
    for step in range(2):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"stacks step {step}")
        seen = max(seen, ctx.stats()["manifolds"])
    assert seen > 8192
    bodies = ctx.bodies()
    bodies[2000:, 9] += 5.0 * np.arange(len(bodies) - 2000)  # most of them flung apart
    ctx.set_bodies(bodies)
    for step in range(2):
        _sync_and_step(ctx, orc)
        _compare_world(ctx, orc, f"stacks apart step {step}")
    assert ctx.stats()["manifolds"] <= 8192
    ctx.close()
