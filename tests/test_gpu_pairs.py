"""GPU parity of the pair search where it changes form: small proxy sets are tested pair by pair (256 proxies against a
chunk at a time), larger ones through the tree; pair sets bit for bit against the oracle."""
import numpy as np
import pytest

import jbgpu
import pyoracle
from test_gpu_parity import MODES, WMAX, WMIN

pytestmark = pytest.mark.gpu


def _both(mode, boxes, group, mask, world):
    ctx = jbgpu.Context(bp_mode=MODES[mode], world_min=WMIN, world_max=WMAX)
    ctx.bp_create_proxies(boxes, group, mask, world)
    orc = pyoracle.Broadphase(MODES[mode], np.array(WMIN, np.float32), np.array(WMAX, np.float32))
    orc.create(boxes, group, mask)
    if world is not None:
        orc.set_worlds(world)
    return ctx, orc


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 2049])
def test_pair_by_pair_tile_edges(mode, n):
    """Both sides of a tile and a chunk, with filters, worlds, boxes that touch exactly, coincident boxes and one box
    around everything."""
    rng = np.random.default_rng(n)
    side = 3.0 * n ** (1.0 / 3.0)
    c = rng.integers(0, max(2, int(side)), (n, 3)).astype(np.float32)  # on a grid: faces touch, some boxes coincide
    h = rng.choice(np.array([0.25, 0.5, 1.0], np.float32), (n, 3))
    v = rng.normal(0, 5, (n, 3)).astype(np.float32)
    h[n // 2] = 500.0
    group = rng.integers(1, 4, n).astype(np.int16)
    mask = rng.integers(0, 4, n).astype(np.int16)
    mask[rng.random(n) < 0.3] = -1
    world = rng.integers(0, 3, n).astype(np.int32)
    ctx, orc = _both(mode, np.concatenate([c - h, c + h], 1), group, mask, world)
    for step in range(4):
        boxes = np.concatenate([c - h, c + h], 1).astype(np.float32)
        ctx.bp_set_aabbs(boxes)
        orc.set_all(boxes)
        ctx.bp_calculate_overlapping_pairs()
        assert np.array_equal(ctx.bp_pairs(), orc.step()), f"{mode} {n} step {step}"
        c = (c + v * np.float32(1.0 / 60.0)).astype(np.float32)
    ctx.close()


@pytest.mark.parametrize("mode", ["dbvt", "sap16"])
@pytest.mark.parametrize("n", [24576, 24577])
def test_both_sides_of_the_tree_limit(mode, n):
    rng = np.random.default_rng(7)
    c = rng.uniform(0, 250, (n, 3)).astype(np.float32)
    h = rng.lognormal(0.0, 0.7, (n, 3)).astype(np.float32)
    boxes = np.concatenate([c - h, c + h], 1).astype(np.float32)
    ctx, orc = _both(mode, boxes, None, None, None)
    for step in range(2):
        ctx.bp_set_aabbs(boxes)
        orc.set_all(boxes)
        ctx.bp_calculate_overlapping_pairs()
        assert np.array_equal(ctx.bp_pairs(), orc.step(cap=1 << 21)), f"{mode} {n} step {step}"
    ctx.close()


def test_dense_tiles_past_their_staging():
    """Every box overlaps every other: a tile finds more pairs than its staging holds, and the pair capacity grows."""
    n = 700
    boxes = np.tile(np.array([[0, 0, 0, 1, 1, 1]], np.float32), (n, 1))
    ctx, orc = _both("dbvt", boxes, None, None, None)
    ctx.bp_set_aabbs(boxes)
    orc.set_all(boxes)
    assert ctx.bp_calculate_overlapping_pairs() == n * (n - 1) // 2
    assert np.array_equal(ctx.bp_pairs(), orc.step(cap=1 << 19))
    ctx.close()


@pytest.mark.parametrize("n", [300, 30000])
def test_proxies_destroyed_between_set_aabb_and_the_query(n):
    """destroyProxy after setAabb and before the pair query: the destroyed proxies pair no more."""
    rng = np.random.default_rng(4)
    c = rng.uniform(0, 3.0 * n ** (1.0 / 3.0), (n, 3)).astype(np.float32)
    boxes = np.concatenate([c - 1, c + 1], 1).astype(np.float32)
    ctx, orc = _both("dbvt", boxes, None, None, None)
    ctx.bp_set_aabbs(boxes)
    orc.set_all(boxes)
    dead = rng.choice(n, n // 5, replace=False) + 1
    ctx.bp_destroy_proxies(dead)
    orc.destroy(dead)
    ctx.bp_calculate_overlapping_pairs()
    got = ctx.bp_pairs()
    lo, hi = (got >> np.uint64(32)).astype(np.int64), (got & np.uint64(0xffffffff)).astype(np.int64)
    assert len(got) and not (np.isin(lo, dead) | np.isin(hi, dead)).any()
    assert np.array_equal(got, orc.step())
    ctx.close()


@pytest.mark.parametrize("couples", [(0, 1, 2, 3), (4095, 4096, 4097, 4096), (5000, 10, 1025, 1024)])
def test_pair_counts_around_the_small_sort(couples):
    """Exactly so many pairs in successive queries (the first of a size is met with the expectation of the last), uids
    shuffled; the sorted keys are known."""
    rng = np.random.default_rng(5)
    most = max(couples)
    c = np.repeat(np.stack([np.arange(most) * 4.0, np.zeros(most), np.zeros(most)], 1), 2, 0).astype(np.float32)
    perm = rng.permutation(2 * most)
    place = np.argsort(perm)  # body of couple k: uids place[2k] + 1, place[2k + 1] + 1
    ctx = jbgpu.Context(bp_mode=jbgpu.BP_DBVT, world_min=WMIN, world_max=WMAX)
    half = np.float32(0.5)
    ctx.bp_create_proxies(np.concatenate([c - half, c + half], 1)[perm])
    for k in couples:
        d = c.copy()
        d[2 * k + 1::2, 1] = 50.0  # the other couples come apart
        ctx.bp_set_aabbs(np.concatenate([d - half, d + half], 1).astype(np.float32)[perm])
        ctx.bp_calculate_overlapping_pairs()
        u = np.sort(place[:2 * k].reshape(-1, 2) + 1, 1).astype(np.uint64)
        assert np.array_equal(ctx.bp_pairs(), np.sort(u[:, 0] << np.uint64(32) | u[:, 1]))
    ctx.close()
