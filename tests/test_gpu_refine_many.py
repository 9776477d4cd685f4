"""Which old vertices a refinement drops, for many new points: on both sides of the line between the
boxes of the new points and the tree of the union (2 and 16 times the old points in 2D and 3D), and of the
counts from which a third and a fourth level of boxes is tested (2^15 and 2^20).  The refined table has to
be the fresh table of the union, and the vertices dropped the old ones that it does not hold."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,m", [(2, 40, 80), (2, 40, 81), (3, 30, 480), (3, 30, 481), (4, 20, 2000), (2, 16500, 32768),
                                   (2, 16500, 32769), (3, 3000, 33000), (4, 100, 33000), (2, 525000, 1048577)])
def test_refined_is_the_fresh_mesh(d, n, m):
    x, y = synth.uniform(d, n, 51), synth.uniform(d, m, 52)
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(*synth.cube_planes(d))
    a = ctx.build_mesh(precision="bf16")
    na = len(a.export()[0])
    r, removed = ctx.refine(a, y, precision="bf16")
    kr, xr = r.export()
    a.free()
    r.free()
    ctx.set_points(np.vstack([x, y]))
    f = ctx.build_mesh(precision="bf16")
    kf, xf = f.export()
    f.free()
    assert np.array_equal(kr, kf) and np.max(np.abs(xr - xf)) < 1e-12
    old = np.sum(~np.any((kf > n) & (kf <= n + m), axis=1))   # vertices of old generators and planes alone
    assert na - removed == old
