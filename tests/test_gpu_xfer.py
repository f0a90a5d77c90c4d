"""Host copies through the pinned slots at the edges of their pieces (512 KiB and 4 MiB; a body has 128 bytes, a
manifold 528), bit for bit, and from several threads at once."""
import threading

import numpy as np
import pytest

import jbgpu
from jbgpu import scenes

pytestmark = pytest.mark.gpu


def _context(n):
    sc = scenes.boxes_grid(nx=n - 1, ny=1, nz=1)
    shapes, verts, bodies = scenes.build_records(sc, jbgpu)
    ctx = jbgpu.Context(num_iterations=1)
    ctx.world_create(shapes, verts, bodies)
    return ctx


def _bodies(n, seed, ok):
    ctx = _context(n)
    b = ctx.bodies().copy()
    b[:, 9:18] = np.random.default_rng(seed).normal(0, 1, (n, 9))
    ctx.set_bodies(b)
    ok.append(ctx.bodies().tobytes() == b.tobytes())
    ctx.close()


@pytest.mark.parametrize("n", [2, 511, 4095, 4096, 4097, 8193, 131071, 131073])
def test_bodies_round_trip(n):
    ok = []
    _bodies(n, n, ok)
    assert ok == [True]


@pytest.mark.parametrize("n", [1, 992, 993, 994, 7944, 31776])
def test_pairs_round_trip(n):
    ctx = _context(n + 3)
    lo = np.arange(2, n + 2, dtype=np.uint64)  # neighbours on the line; uid 1 is the plane
    keys = lo << np.uint64(32) | (lo + np.uint64(1))
    keys = keys[:n]
    man = np.random.default_rng(n).normal(0, 1, (n, jbgpu.MANIFOLD_WORDS)).astype(np.float32)
    head = man.view(np.int32)
    head[:, 0] = np.arange(n) % 5
    head[:, 1], head[:, 2], head[:, 3] = lo[:n] - np.uint64(1), lo[:n], 2  # convex against convex
    ctx.set_pairs(keys, man)
    k, m = ctx.pairs()
    assert np.array_equal(k, keys) and m.tobytes() == man.tobytes()
    ctx.close()


def test_copies_from_several_threads():
    ok = []
    threads = [threading.Thread(target=_bodies, args=(40001 + 977 * k, k, ok)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert ok == [True] * 4
