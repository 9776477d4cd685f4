"""A context may take over the stream and the device tables of one that is gone: whatever they were
used for before (another dimension, size, precision, an integral, a refused set), its results have to be
those of a fresh one, also while another context lives and after the kept tables were given back."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context, HVError, lib

pytestmark = pytest.mark.gpu


def pass_of(d, n, precision, seed=6):
    ctx = Context(0)
    ctx.set_points(synth.uniform(d, n, seed))
    ctx.set_boundary(*synth.cube_planes(d))
    m = ctx.build_mesh(precision=precision)
    table = m.export()
    r = ctx.integrate(m, "polytope")
    m.free()
    return table + (r["volumes"], r["neighbors"], r["areas"])


def test_contexts_after_contexts():
    shapes = [(3, 900, "fp64"), (2, 50, "bf16"), (5, 200, "fp32"), (2, 4000, "fp64"), (4, 300, "bf16")]
    first = {}
    for s in shapes:
        assert lib().hv_batch_release(-1) == 0
        first[s] = pass_of(*s)
    for s in shapes[::-1] + shapes:
        with pytest.raises(HVError):
            bad = Context(0)
            bad.set_points(synth.uniform(s[0], 40, 1) + 0.7)
            bad.set_boundary(*synth.cube_planes(s[0]))
            bad.build_mesh(precision=s[2])
        bad = None
        got = pass_of(*s)
        for a, b in zip(got[:2] + (got[3],), first[s][:2] + (first[s][3],)):
            assert np.array_equal(a, b)
        for a, b in zip((got[2], got[4]), (first[s][2], first[s][4])):
            assert np.allclose(a, b, rtol=1e-12, atol=0.0)


def test_two_contexts_side_by_side():
    a, b = Context(0), Context(0)
    for ctx, d in ((a, 2), (b, 3)):
        ctx.set_points(synth.uniform(d, 500, 9))
        ctx.set_boundary(*synth.cube_planes(d))
    ma, mb = a.build_mesh(precision="bf16"), b.build_mesh(precision="bf16")
    ka, kb = ma.export()[0], mb.export()[0]
    del a   # its mesh lives on
    c = Context(0)
    c.set_points(synth.uniform(4, 300, 9))
    c.set_boundary(*synth.cube_planes(4))
    mc = c.build_mesh(precision="bf16")
    assert np.array_equal(ma.export()[0], ka) and np.array_equal(mb.export()[0], kb)
    for m in (ma, mb, mc):
        m.free()
