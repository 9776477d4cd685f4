"""Calls small enough for the pinned block (2 MiB, arguments and results together) are worked on there,
larger ones are copied: one call of each kind on both sides of that limit has to give, piece by
piece, what many small ones give; a refused ray is named, and nothing is written, on either side."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context, HVError

pytestmark = pytest.mark.gpu


def context(d, n):
    ctx = Context(0)
    ctx.set_points(synth.uniform(d, n, 3))
    ctx.set_boundary(*synth.cube_planes(d))
    return ctx


def pieces(n):
    return ((0, 1), (1, 1000), (n - 700, n))


@pytest.mark.parametrize("d,nq", [(2, 37000), (2, 37600), (5, 20000), (5, 20500)])
def test_nearest(d, nq):
    ctx, rng = context(d, 3000), np.random.default_rng(1)
    q, u = rng.random((nq, d)), rng.standard_normal((nq, d))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    c = (u * q).sum(1)
    idx, dist = ctx.nn_halfspace(q, u, c)
    for a, b in pieces(nq):
        i, t = ctx.nn_halfspace(q[a:b], u[a:b], c[a:b])
        assert np.array_equal(i, idx[a:b]) and np.array_equal(t, dist[a:b])


@pytest.mark.parametrize("d,nq", [(3, 5000), (3, 60000)])
def test_inrange(d, nq):
    ctx, rng = context(d, 3000), np.random.default_rng(2)
    q, r = rng.random((nq, d)), rng.uniform(0.0, 0.15, nq)
    ptr, idx = ctx.inrange(q, r)
    for a, b in pieces(nq):
        p, i = ctx.inrange(q[a:b], r[a:b])
        assert np.array_equal(p, ptr[a:b + 1] - ptr[a]) and np.array_equal(i, idx[ptr[a]:ptr[b]])


@pytest.mark.parametrize("count", [50, 40000])
def test_rays(count):
    d, n = 3, 2000
    ctx = context(d, n)
    m = ctx.build_mesh(precision="fp64")
    keys, coords = m.export()
    m.free()
    keep = keys[:, 1] <= n
    sig = np.resize(keys[keep].astype(np.int64), (count, d + 1))
    r = np.resize(coords[keep], (count, d))
    drop = (np.arange(count) % (d + 1)).astype(np.int32)
    res = ctx.raycast_batch(sig, drop, r)
    for a, b in pieces(max(count, 701)):
        a, b = min(a, count - 1), min(b, count)
        for x, y in zip(ctx.raycast_batch(sig[a:b], drop[a:b], r[a:b]), res):
            assert np.array_equal(x, y[a:b], equal_nan=True)
    for j, value, text in ((1, n + 2 * d + 1, "out of range"), (1, int(sig[-1, 0]), "sorted"), (-1, d + 1, "drop position")):
        s, p = sig.copy(), drop.copy()
        if j < 0:
            p[-1] = value
        else:
            s[-1, j] = value
        with pytest.raises(HVError, match=text):
            ctx.raycast_batch(s, p, r)
    again = ctx.raycast_batch(sig, drop, r)
    for x, y in zip(again, res):
        assert np.array_equal(x, y, equal_nan=True)
