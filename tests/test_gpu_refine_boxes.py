"""The old vertices a refinement keeps are found with boxes of 32 and of 1 024 new points: the refined
table has to be the fresh table of the union for counts of new points on both sides of those sizes,
spread and all in one corner (vertices far from every box, and boxes within many spheres)."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,m,side", [(2, 3000, 1, 1.0), (3, 1500, 31, 0.3), (3, 1500, 33, 1.0), (2, 2000, 1024, 1.0),
                                        (2, 2000, 1025, 0.2), (4, 500, 65, 0.5), (5, 200, 20, 1.0)])
def test_refined_is_the_fresh_mesh(d, n, m, side):
    x, y = synth.uniform(d, n, 41), side * synth.uniform(d, m, 42)
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(*synth.cube_planes(d))
    a = ctx.build_mesh(precision="bf16")
    r, _ = ctx.refine(a, y, precision="bf16")
    kr, xr = r.export()
    a.free()
    r.free()
    ctx.set_points(np.vstack([x, y]))
    f = ctx.build_mesh(precision="bf16")
    kf, xf = f.export()
    f.free()
    assert np.array_equal(kr, kf) and np.max(np.abs(xr - xf)) < 1e-12
