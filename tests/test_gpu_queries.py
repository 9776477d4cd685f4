"""Half-space nearest and range queries against brute force in FP64 (ids exact, distances to a few
roundings), at the edges of the leaves (32 points), of the 8-ary tree's levels (256 and 2 048
points) and of the list a wavefront sorts in LDS (512 hits); and across what makes a context's
kept search tree stale."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context

pytestmark = pytest.mark.gpu


def context(xs):
    ctx = Context(0)
    ctx.set_points(xs)
    ctx.set_boundary(*synth.cube_planes(xs.shape[1]))
    return ctx


def brute_nearest(xs, q, u, c):
    d2 = ((q[:, None] - xs[None]) ** 2).sum(2)
    d2[~(u @ xs.T > c[:, None])] = np.inf
    i = d2.argmin(1)
    best = d2[np.arange(len(q)), i]
    return np.where(best < np.inf, i + 1, 0), np.sqrt(best)


def check_nearest(ctx, xs, q, u, c):
    idx, dist = ctx.nn_halfspace(q, u, c)
    ri, rd = brute_nearest(xs, q, u, c)
    assert np.array_equal(idx, ri)
    assert np.allclose(dist, rd, rtol=1e-14, atol=0)


def check_range(ctx, xs, q, rad):
    ptr, ids = ctx.inrange(q, rad)
    d2 = ((q[:, None] - xs[None]) ** 2).sum(2)
    hit = d2 <= (rad ** 2)[:, None]
    assert np.array_equal(np.diff(ptr), hit.sum(1))
    for k in range(len(q)):
        assert np.array_equal(ids[ptr[k]:ptr[k + 1]], np.nonzero(hit[k])[0] + 1)


def queries(d, n, nq, seed):
    rng = np.random.default_rng(seed)
    q = rng.uniform(-0.2, 1.2, (nq, d))
    u = rng.standard_normal((nq, d))
    c = (u * q).sum(1)
    c[::3] = -np.inf
    c[1::7] = 1e9   # nothing ahead
    return q, u, c


@pytest.mark.parametrize("d,n,nq", [(2, 3, 1), (2, 32, 5), (3, 33, 64), (3, 255, 257), (4, 256, 3), (4, 2049, 130),
                                    (5, 2047, 66), (6, 3000, 65)])
def test_queries_match_brute_force(d, n, nq):
    xs = synth.uniform(d, n, 40 + d)
    ctx = context(xs)
    q, u, c = queries(d, n, nq, 9)
    check_nearest(ctx, xs, q, u, c)
    rng = np.random.default_rng(3)
    check_range(ctx, xs, q, rng.uniform(0.0, 1.0, nq))   # from no hit to more than a wavefront sorts in LDS


def test_equal_distances_give_the_smaller_id():
    g = np.stack(np.meshgrid(*[np.arange(1, 8) / 8.0] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    xs = np.ascontiguousarray(g[np.random.default_rng(1).permutation(len(g))])
    ctx = context(xs)
    q = (np.floor(np.random.default_rng(2).random((50, 3)) * 6) + 1.5) / 8.0   # cell centres: 8 nearest each
    u = np.tile([1.0, 0.0, 0.0], (50, 1))
    c = np.full(50, -np.inf)
    idx, _ = ctx.nn_halfspace(q, u, c)
    d2 = ((q[:, None] - xs[None]) ** 2).sum(2)      # exact in binary
    assert np.array_equal(idx, d2.argmin(1) + 1)


def test_a_kept_tree_follows_points_planes_and_integrals():
    d = 3
    a, b = synth.uniform(d, 700, 1), synth.uniform(d, 700, 2)
    ctx = context(a)
    q, u, c = queries(d, 700, 40, 5)
    check_nearest(ctx, a, q, u, c)
    ctx.set_points(b)                                 # the same size: written in place
    check_nearest(ctx, b, q, u, c)
    m = ctx.build_mesh(precision="bf16")
    check_nearest(ctx, b, q, u, c)
    ctx.set_points(a)                                 # the mesh keeps b
    check_range(ctx, a, q, np.full(40, 0.3))
    ctx.integrate(m, "points", nsamples=20000, seed=1)   # a tree over b in the same tables
    check_nearest(ctx, a, q, u, c)
    m.free()
    base, normal = synth.cube_planes(d, -1.0, 2.0)
    ctx.set_boundary(base, normal)
    check_nearest(ctx, a, q, u, c)
    check_range(ctx, a, q, np.full(40, 0.2))


@pytest.mark.parametrize("first,second", [("fp64", "bf16"), ("bf16", "fp32"), ("fp32", "fp64")])
def test_rays_on_a_kept_tree_equal_rays_on_a_fresh_one(first, second):
    d, n = 4, 900
    xs = synth.uniform(d, n, 12)
    ctx = context(xs)
    m = ctx.build_mesh()
    keys, coords = m.export()
    m.free()
    v = np.arange(0, len(keys), 7)
    sig, r = keys[v], coords[v]
    drop = np.full(len(sig), d, dtype=np.int32)       # a key's first id is a generator
    ctx2 = context(xs)
    q, u, c = queries(d, n, 9, 6)
    ctx2.nn_halfspace(q, u, c)                        # leaves a tree without neighbour lists
    ctx2.raycast_batch(sig, drop, r, precision=first)
    kept = ctx2.raycast_batch(sig, drop, r, precision=second)
    fresh = context(xs).raycast_batch(sig, drop, r, precision=second)
    for x, y in zip(kept, fresh):
        assert np.array_equal(x, y, equal_nan=x.dtype.kind == "f")
