"""Face grouping where several faces share a grouping key (their smallest id and a hash of the others): a
generator in the middle of a noisy sphere of others is the smallest id of tens of thousands of edges, several
of which fall on one hash value.  Against the oracle, and, for so many ids that fewer hash bits are left,
against a mesh of a few of the cells, whose ids are few.  An integral outlives its context and its mesh.

Bounds: measures of size at most 1, formed from heights that a projection between normals at an angle down
to about 1e-5 divides, so rounding grows to some 1e5 times 2e-16 and, over the terms of a face, stays
below 1e-9."""
import ctypes as C

import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context, lib
from oracle_py import polytope

pytestmark = pytest.mark.gpu

TOL = 1e-9


def star(d, n, seed=1):
    rng = np.random.default_rng(seed)
    v = rng.normal(size=(n, d))
    v /= np.linalg.norm(v, axis=1)[:, None]
    x = 0.5 + v * (0.4 * (1 + 1e-3 * rng.uniform(-1, 1, size=(n, 1))))
    x[0] = 0.5
    return x


def setup(x):
    ctx = Context(0)
    ctx.set_points(x)
    ctx.set_boundary(*synth.cube_planes(x.shape[1]))
    return ctx


@pytest.mark.parametrize("d,n", [(3, 6000), (4, 700)])
def test_shared_keys_match_the_oracle(d, n):
    x = star(d, n)
    ctx = setup(x)
    m = ctx.build_mesh()
    keys, coords = m.export()
    got = ctx.integrate(m, "polytope")
    m.free()
    vol, ptr, nbr, area = polytope(x, *synth.cube_planes(d), keys, coords)
    assert ptr[1] > 600                          # neighbours of the middle cell
    assert np.array_equal(got["nbr_ptr"], ptr) and np.array_equal(got["neighbors"], nbr)
    assert np.max(np.abs(got["volumes"] - vol)) < TOL and np.max(np.abs(got["areas"] - area)) < TOL


def test_many_ids_match_a_mesh_of_few_cells():
    n, cells = 300_000, np.array([1, 2, 77, 150_000, 300_000])   # 19 bits an id: 13 of hash
    ctx = setup(star(3, n))
    m = ctx.build_mesh()
    a = ctx.integrate(m, "polytope")
    m.free()
    m = ctx.build_mesh_cells(cells)
    b = ctx.integrate(m, "polytope")
    m.free()
    assert abs(a["volumes"].sum() - 1.0) < TOL
    for c in cells - 1:
        ra, rb = slice(a["nbr_ptr"][c], a["nbr_ptr"][c + 1]), slice(b["nbr_ptr"][c], b["nbr_ptr"][c + 1])
        assert np.array_equal(a["neighbors"][ra], b["neighbors"][rb])
        assert np.max(np.abs(a["areas"][ra] - b["areas"][rb])) < TOL
        assert abs(a["volumes"][c] - b["volumes"][c]) < TOL


def test_integral_outlives_its_context():
    x = synth.uniform(3, 500, 9)
    ctx = setup(x)
    m = ctx.build_mesh()
    want = ctx.integrate(m, "polytope")
    h = C.c_void_p()
    assert lib().hv_integrate_polytope(ctx._h, m._h, C.byref(h)) == 0
    m.free()
    del m, ctx
    vol = np.zeros(500)
    area = np.zeros(len(want["areas"]))
    dp = C.POINTER(C.c_double)
    assert lib().hv_integral_export(h, vol.ctypes.data_as(dp), None, None, area.ctypes.data_as(dp), None) == 0
    lib().hv_integral_free(h)
    assert np.array_equal(vol, want["volumes"]) and np.array_equal(area, want["areas"])
