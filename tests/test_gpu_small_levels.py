"""Small levels are started 16 lanes a ray and scanned a wavefront a ray.  The same rays asked for in
batches on both sides of the limit (8 192 rays, 32 768 in 2D and 3D; half of it where the count is
exact) have to end alike, ray by ray, and at the oracle's vertices; short 16-NN lists and a tree of
one node are the smallest cases.  Leaves of other sizes than 32 keep the packet scan."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context
from oracle_py import Oracle

pytestmark = pytest.mark.gpu


def rays_of(keys, coords, n, count):
    d = coords.shape[1]
    v, p = np.divmod(np.arange(len(keys) * (d + 1)), d + 1)
    first = np.where(p == 0, keys[v, 1], keys[v, 0])
    v, p = v[first <= n], p[first <= n]
    v, p = np.resize(v, count), np.resize(p, count)
    return keys[v].astype(np.int64), p.astype(np.int32), coords[v]


@pytest.mark.parametrize("d,n,limit", [(2, 3000, 16384), (3, 1500, 16384), (4, 400, 4096), (5, 150, 4096), (6, 60, 4096)])
@pytest.mark.parametrize("precision", ["fp64", "bf16"])
def test_rays_end_alike_in_small_and_large_batches(d, n, limit, precision):
    x = synth.uniform(d, n, 19)
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(*synth.cube_planes(d))
    m = ctx.build_mesh(precision=precision)
    keys, coords = m.export()
    m.free()
    ok, _, _ = Oracle(x, *synth.cube_planes(d)).voronoi()
    assert np.array_equal(keys, ok[np.lexsort(ok.T[::-1])])
    sig, drop, r = rays_of(keys, coords, n, limit + 1)
    large = ctx.raycast_batch(sig, drop, r, precision=precision)
    for lo, hi in ((0, limit), (limit, limit + 1), (7, 8), (3, 260)):
        small = ctx.raycast_batch(sig[lo:hi], drop[lo:hi], r[lo:hi], precision=precision)
        for a, b in zip(small, large):
            assert np.array_equal(a, b[lo:hi], equal_nan=True)


@pytest.mark.parametrize("d,n", [(2, 3), (3, 5), (4, 16), (5, 18)])
def test_smallest_sets(d, n):
    x = synth.uniform(d, n, 23)
    base, normal = synth.cube_planes(d)
    ok, oc, _ = Oracle(x, base, normal).voronoi()
    o = np.lexsort(ok.T[::-1])
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(base, normal)
    for leaf in (0, 8):
        m = ctx.build_mesh(precision="fp64", leaf_size=leaf)
        k, c = m.export()
        m.free()
        assert np.array_equal(k, ok[o])
        assert np.max(np.abs(c - oc[o])) < 1e-10
