"""hv_mesh_export sorts on the device: rows strictly ascending in lexicographic key order, every
coordinate row with its own key, for keys of one, two and three sort words (ids of 6 .. 17 bits,
3 .. 7 ids per key) and a table exported in more than one chunk."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context

pytestmark = pytest.mark.gpu


def check(d, n, precision="bf16"):
    xs = synth.uniform(d, n, 700 + d)
    base, normal = synth.cube_planes(d)
    ctx = Context(0)
    ctx.set_points(xs)
    ctx.set_boundary(base, normal)
    m = ctx.build_mesh(precision=precision)
    keys, coords = m.export()
    nv = m.counts()[0]
    m.free()
    assert keys.shape == (nv, d + 1) and coords.shape == (nv, d)
    assert np.all(np.diff(keys, axis=1) > 0) and keys.min() >= 1 and keys.max() <= n + 2 * d
    # strictly ascending rows: the first column that differs from the row above is larger
    diff = np.diff(keys, axis=0)
    lead = (diff != 0).argmax(axis=1)
    assert np.all(diff[np.arange(nv - 1), lead] > 0)
    # the coordinates belong to the key: equal distances to its generators, planes met
    r0 = np.linalg.norm(coords - xs[keys[:, 0] - 1], axis=1)
    for j in range(1, d + 1):
        gen = keys[:, j] <= n
        r = np.linalg.norm(coords[gen] - xs[keys[gen, j] - 1], axis=1)
        assert np.max(np.abs(r - r0[gen]), initial=0.0) < 1e-8
        p = keys[~gen, j] - n - 1
        off = np.sum(normal[p] * (coords[~gen] - base[p]), axis=1)
        assert np.max(np.abs(off), initial=0.0) < 1e-8


@pytest.mark.parametrize("d,n", [(2, 40), (2, 70000), (3, 58), (3, 59), (4, 900), (5, 300), (6, 120), (6, 500)])
def test_rows_sorted_and_paired(d, n):
    check(d, n)


def test_table_of_several_chunks():
    check(5, 25000)   # about 3.6 million rows of 88 bytes
