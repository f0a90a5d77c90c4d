"""The pair search of convex shapes against the oracle, bit for bit: hulls with every remainder of the support map's
vertex groups (eight at a time), pair counts on both sides of the lines where waves take more pairs (4096 and 8192) and
where the order by type takes another form (32768), and shapes apart, touching and overlapping, so that the simplex passes through every region of triangles and tetrahedra."""
import numpy as np
import pytest

import jbgpu
import pyoracle
from jbgpu import scenes
from test_gpu_seams import _masked, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 127, 1024, 4096, 4097, 8191, 8193, 32768, 32769])
def test_random_convex_pairs(n):
    rng = np.random.default_rng(n)
    b = scenes._Builder("cluster")
    kinds = [b.hull(rng.normal(0, 0.6, (k, 3))) for k in (1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 33)]
    kinds += [b.shape(scenes.BOX, [0.5, 0.7, 0.3]), b.shape(scenes.CAPSULE, [0.3, 0.5]), b.shape(scenes.SPHERE, [0.5])]
    m = 131 if n < 8500 else 260
    b.bodies([kinds[i % len(kinds)] for i in range(m)], scenes._quat_basis(scenes._random_quats(rng, m)),
             rng.uniform(-3, 3, (m, 3)).astype(np.float32), np.ones(m, np.float32))
    shapes, verts, bodies = scenes.build_records(b.done(dt=1 / 60, iterations=10), jbgpu)
    lo, hi = np.triu_indices(m, 1)
    pick = np.sort(rng.permutation(len(lo))[:n])
    lo, hi = lo[pick], hi[pick]
    keys = (lo + 1).astype(np.uint64) << np.uint64(32) | (hi + 1).astype(np.uint64)
    rec = np.zeros((n, jbgpu.MANIFOLD_WORDS), np.float32)
    head = rec.view(np.int32)
    head[:, 1], head[:, 2] = lo, hi
    sphere = np.array([i % len(kinds) == len(kinds) - 1 for i in range(m)])
    head[:, 3] = np.where(sphere[lo] & sphere[hi], 0, 2)
    ctx = jbgpu.Context(num_iterations=10)
    ctx.world_create(shapes, verts, bodies)
    orc = pyoracle.World(shapes, verts, bodies, iterations=10, order=jbgpu.ORDER_EXPLICIT)
    got = ctx.np_dispatch(keys, rec)
    orc.set_pairs(keys, rec)
    orc.phase(2)
    _, want = orc.pairs()
    assert _same(_masked(got), _masked(want))
    assert n < 100 or (got[:, 0].view(np.int32) > 0).any()
    ctx.close()
