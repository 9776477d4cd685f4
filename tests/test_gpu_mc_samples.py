"""The sampling kernel's matrix filter must not lose a neighbour: its samples are drawn again here
(the same strata and stream), and each is given to its nearest generator by brute force in 64 bits.
A lost nearest generator moves a sample to another cell, so the counts, hence the volumes, have to
agree exactly: what the kernel measures in FP32 only picks the two generators it measures in FP64,
and three within 1e-7 of one distance do not occur among these samples.  Sizes: within one leaf of
32, one point more, several levels of the tree with a ragged last leaf; a box away from the origin;
clustered points (wide and narrow packets); the periodic box, whose images are looked up."""
import numpy as np
import pytest

from hvgpu import synth
from hvgpu._lib import Context
from hvgpu.geometry import cuboid

pytestmark = pytest.mark.gpu


def mix(z):
    for mul in (0xff51afd7ed558ccd, 0xc4ceb9fe1a85ec53):
        z = z ^ (z >> np.uint64(33))
        z = z * np.uint64(mul)
    return z ^ (z >> np.uint64(33))


def samples(d, nsamples, seed, lo, hi):
    G = max(1, int(np.floor((nsamples / 256.0) ** (1.0 / d))))
    per = -(-nsamples // G ** d)
    per = (per + 63) // 64 * 64
    s = np.arange(G ** d * per, dtype=np.uint64)
    b = s // np.uint64(per)
    p = np.empty((len(s), d))
    for k in range(d):
        ck = (b % np.uint64(G)).astype(float)
        b //= np.uint64(G)
        with np.errstate(over="ignore"):
            idx = s * np.uint64(d) + np.uint64(k) + np.uint64(1)
            u = mix(np.uint64(seed) ^ (idx * np.uint64(0x9E3779B97F4A7C15)))
        p[:, k] = lo + (ck + (u >> np.uint64(11)).astype(float) / 2.0 ** 53) * ((hi - lo) / G)
    return p


def counts(x, p, box):
    c = np.zeros(len(x), dtype=np.int64)
    step = max(1, int(2e7 / (len(x) * x.shape[1])))
    for a in range(0, len(p), step):
        d2 = np.zeros((len(p[a:a + step]), len(x)))
        for k in range(x.shape[1]):
            t = np.abs(p[a:a + step, k, None] - x[None, :, k])
            if box:
                t = np.minimum(t, box - t)
            d2 += t * t
        c += np.bincount(d2.argmin(1), minlength=len(x))
    return c


@pytest.mark.parametrize("d,n,lo,hi,points,periodic", [
    (2, 32, 0.0, 1.0, "uniform", False), (2, 33, 0.0, 1.0, "uniform", False), (3, 2049, -1.0, 2.0, "uniform", False),
    (4, 777, 0.0, 1.0, "mixture", False), (5, 300, 0.0, 1.0, "mixture", False), (6, 255, 0.0, 1.0, "uniform", False),
    (2, 150, 0.0, 1.0, "uniform", True), (4, 200, 0.0, 1.0, "uniform", True), (6, 40, 0.0, 1.0, "uniform", True)])
def test_samples_go_to_their_nearest_generator(d, n, lo, hi, points, periodic):
    x = synth.uniform(d, n, 77) if points == "uniform" else synth.gaussian_mixture_5d(n, seed=3, d=d)
    x = lo + (hi - lo) * x
    ctx = Context(0)
    ctx.set_points(x)
    if periodic:
        ctx.set_boundary(*cuboid(d, periodic=None).arrays())
    else:
        ctx.set_boundary(*synth.cube_planes(d, lo, hi))
    m = ctx.build_mesh(precision="bf16")
    r = ctx.integrate(m, "points", nsamples=40000, seed=5)
    m.free()
    p = samples(d, 40000, 5, lo, hi)
    want = counts(x, p, (hi - lo) if periodic else 0.0)
    got = r["volumes"] * (len(p) / (hi - lo) ** d)
    assert np.max(np.abs(got - np.rint(got))) < 1e-6
    assert np.array_equal(np.rint(got).astype(np.int64), want)
