"""The list passes (csrc/nbr_passes.hip) with 16 and with 4 lanes per
particle: the sums are taken in the list's order, so lists, overflow scans,
single instances and batches agree bit for bit, at counts that leave a
wavefront's groups and a group's lanes partly empty."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

FIELDS = ("density", "dstress_dt", "density_dt", "balsara", "acc", "xvel", "maxvsig")


def workload(kind, n):
    if kind == "solid":
        return ics.collision(n, seed=n, gap=-2.0, gravity=False)
    h, prm = ics.liquid_blob(n, seed=n, gravity=False,
                             fields=("posm", "pos64", "vel", "acc", "density", "density_dt", "balsara", "maxvsig", "xvel"))
    h["vel"][:, :3] = np.random.default_rng(n).normal(0.0, 0.1, size=(n, 3))
    if kind == "xsph":
        prm.flags |= g.XSPH
        prm.xsph_factor = 0.5
    else:  # artificial pressure, no Balsara switch
        prm.flags |= g.ARTIFICIAL_STRESS
        prm.flags &= ~g.BALSARA_SWITCH
    return h, prm


def run(h, prm, capacity):
    ctx = g.Context(0)
    if capacity:
        ctx.set_option("max_neighbours_grow", 0)
        ctx.set_option("max_neighbours", capacity)
    d = g.DeviceParticles.from_host(h)
    ctx.compute_derivatives(d, prm)
    g.hip.synchronize()
    out = d.download([f for f in FIELDS if f in h])
    d.free()
    ctx.close()
    return out


@pytest.mark.parametrize("kind", ["solid", "xsph", "pressure"])
@pytest.mark.parametrize("n", [2, 5, 17, 333, 10240, 10241])
def test_lists_scans_and_batches_agree(kind, n):
    print("passes kind=%s n=%d" % (kind, n), flush=True)
    h, prm = workload(kind, n)
    a = run(h, prm, 0)
    assert np.all(np.isfinite(a["acc"]))
    b = run(h, prm, 33)  # the particles inside overflow, those at the surface don't
    for f in a:
        assert np.array_equal(a[f], b[f]), f
    if n > 400:
        h2, prm2 = workload(kind, 37)  # a batch walks with 4 lanes: against 16 of the single instance
        host, offsets = g.pack_batch([h2, h, h2])
        ctx = g.Context(0)
        d = g.DeviceParticles.from_host(host)
        ctx.batch_compute_derivatives(d, ctx.batch(offsets, [prm2, prm, prm2]))
        g.hip.synchronize()
        got = g.unpack_batch(d.download(list(a)), offsets)
        d.free()
        ctx.close()
        for f in a:
            assert np.array_equal(got[1][f], a[f]), f
            assert np.array_equal(got[0][f], got[2][f]), f


@pytest.mark.parametrize("kind", ["solid", "xsph"])
def test_overflow_scans_in_a_batch(kind):
    """Scans of the second and third instance's own boxes of 512 slots."""
    print("passes batch overflow kind=%s" % kind, flush=True)
    sizes = (700, 1025, 2500)
    inst = [workload(kind, n) for n in sizes]
    host, offsets = g.pack_batch([h for h, _ in inst])
    ctx = g.Context(0)
    ctx.set_option("max_neighbours_grow", 0)
    ctx.set_option("max_neighbours", 33)
    d = g.DeviceParticles.from_host(host)
    ctx.batch_compute_derivatives(d, ctx.batch(offsets, [p for _, p in inst]))
    g.hip.synchronize()
    a = [run(h, p, 0) for h, p in inst]
    got = g.unpack_batch(d.download(list(a[0])), offsets)
    d.free()
    ctx.close()
    for k in range(len(sizes)):
        for f in a[k]:
            assert np.array_equal(got[k][f], a[k][f]), (k, f)


def test_rigid_rotation_counts_the_same_pairs():
    """In a rigid rotation v . r of every pair is FP32 rounding, whose sign
    decides whether the pair counts for maxvsig: evaluated as the FP32 oracle
    rounds it, the same particles have none."""
    n = 4000
    print("passes rigid rotation n=%d" % n, flush=True)
    h, prm = ics.large_sphere(n, seed=3, noise=0.0, spin=0.3)
    prm.flags &= ~g.SELF_GRAVITY
    got = run(h, prm, 0)["maxvsig"]
    ref = O.compute_derivatives(prm, h, "f32")["maxvsig"]
    assert np.array_equal(got == 0, ref == 0)
    # 2 c and a wij of rounding
    assert np.allclose(got, ref, rtol=1e-6, atol=0)


@pytest.mark.parametrize("kind,n", [("solid", 65536), ("solid", 65537), ("xsph", 65599), ("solid", 98500)])
def test_long_list_capacity_changes_nothing(kind, n):
    """A capacity past 512 takes 16 lanes a particle and, from 65537 particles on, blocks dealt to the XCDs in runs
    (whole runs up to 65536 and 98304 slots' worth of them, and what is left at the end)."""
    print("long lists kind=%s n=%d" % (kind, n), flush=True)
    h, prm = workload(kind, n)
    a = run(h, prm, 0)
    b = run(h, prm, 544)
    for f in a:
        assert np.array_equal(a[f], b[f]), f
