"""The order a level's rays are scanned in, and the emission of the next level's before its counts
are known, must not change the mesh: the default walk (rays counted into buckets along the
generators' Morton order) against the one that sorts every ray's code (chunks=1).  Sizes: a handful
of generators, one bucket per several generators, several buckets per generator, and counts on both
sides of the one-workgroup scan; clustered points crowd the buckets; one plane family without
images, and cells of a periodic box."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context
from hvgpu.geometry import cuboid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,points,precision", [
    (2, 4, "uniform", "fp64"), (3, 17, "uniform", "bf16"), (2, 4095, "mixture", "fp32"), (2, 4097, "uniform", "bf16"),
    (3, 20011, "mixture", "fp64"), (4, 3000, "uniform", "bf16"), (5, 1200, "mixture", "fp32"), (6, 120, "uniform", "bf16")])
def test_mesh_does_not_depend_on_the_scan_order(d, n, points, precision):
    x = synth.uniform(d, n, 5) if points == "uniform" else synth.gaussian_mixture_5d(n, seed=4, d=d)
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(*synth.cube_planes(d))
    a = ctx.build_mesh(precision=precision)
    ka, xa = a.export()
    sa = a.stats()
    a.free()
    b = ctx.build_mesh(precision=precision, chunks=1)
    kb, xb = b.export()
    b.free()
    assert np.array_equal(ka, kb) and np.array_equal(xa, xb)
    assert sa["vertices"] == len(ka)


@pytest.mark.parametrize("d,n", [(2, 60), (3, 150)])
def test_periodic_mesh_does_not_depend_on_the_scan_order(d, n):
    ctx = Context(0)
    tables = []
    for chunks in (0, 1):
        ctx.set_points(synth.uniform(d, n, 8))
        ctx.set_boundary(*cuboid(d, periodic=None).arrays())
        m = ctx.build_mesh(precision="bf16", chunks=chunks)
        tables.append(m.export())
        m.free()
    assert np.array_equal(tables[0][0], tables[1][0]) and np.array_equal(tables[0][1], tables[1][1])
