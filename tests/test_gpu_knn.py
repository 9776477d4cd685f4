"""The 16-NN lists feed every ray's start: the mesh must not depend on the leaves they were found in
(below, at and above 32 points, up to the 64 a scan stages), and sets with fewer
than 17 points, or in one block of 64, have short lists."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context
from oracle_py import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf", [8, 31, 32, 33, 64])
@pytest.mark.parametrize("d,n", [(2, 700), (3, 1500), (5, 400)])
def test_mesh_does_not_depend_on_the_leaves(d, n, leaf):
    xs = synth.uniform(d, n, 21)
    ctx = Context(0)
    ctx.set_points(xs)
    ctx.set_boundary(*synth.cube_planes(d))
    a = ctx.build_mesh(precision="fp64", leaf_size=leaf)
    ka, ca = a.export()
    a.free()
    b = ctx.build_mesh(precision="bf16")
    kb, cb = b.export()
    b.free()
    assert np.array_equal(ka, kb) and np.array_equal(ca, cb)


@pytest.mark.parametrize("d,n", [(2, 3), (3, 16), (4, 17), (3, 63), (2, 64), (2, 65), (6, 66)])
def test_short_lists(d, n):
    xs = synth.uniform(d, n, 33)
    base, normal = synth.cube_planes(d)
    ctx = Context(0)
    ctx.set_points(xs)
    ctx.set_boundary(base, normal)
    m = ctx.build_mesh(precision="bf16")
    k, c = m.export()
    m.free()
    ok, oc, _ = Oracle(xs, base, normal).voronoi()
    o = np.lexsort(ok.T[::-1])
    assert np.array_equal(k, ok[o])
    assert np.max(np.abs(c - oc[o])) < 1e-10
