"""hv_build_mesh_batch over more meshes in one walk than the limit of a level's ray buckets (2048):
the levels of few rays end too, and every mesh equals its single build bit for bit."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context, build_mesh_batch

pytestmark = pytest.mark.gpu


def test_batch_of_more_meshes_than_buckets():
    pts = [synth.uniform(2, 4 + k % 9, 1000 + k) for k in range(2600)]
    planes = [synth.cube_planes(2)] * len(pts)
    out, status = build_mesh_batch(pts, planes, precision="bf16")
    assert not np.any(status)
    ctx = Context(0)
    for k, (m, x) in enumerate(zip(out, pts)):
        got = m.export()
        m.free()
        if k % 20 == 0:
            ctx.set_points(x)
            ctx.set_boundary(*planes[0])
            s = ctx.build_mesh(precision="bf16")
            want = s.export()
            s.free()
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        # Euler: n cells, every vertex of degree 3, the square's four corners of degree 2
        assert len(got[0]) == 2 * len(x) + 2
