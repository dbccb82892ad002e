"""Batches of many small instances: counts around the passes' blocks of 64 slots, the
list kernel's of 32 and the in-group gravity's of 64 and 256, against the
single-instance path; and an instance's gravity among few blocks (of 64) and among
many (of 256), bit for bit."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

from tests._util import vec_errors

pytestmark = pytest.mark.gpu

FIELDS = ("density", "balsara", "maxvsig", "dstress_dt", "acc")


def batch_of(inst, options=()):
    host, offsets = g.pack_batch([h for h, _ in inst])
    ctx = g.Context(0)
    for k, v in options:
        ctx.set_option(k, v)
    d = g.DeviceParticles.from_host(host)
    ctx.batch_compute_derivatives(d, ctx.batch(offsets, [p for _, p in inst]))
    g.hip.synchronize()
    out = g.unpack_batch(d.download([f for f in FIELDS if f in host]), offsets)
    d.free()
    ctx.close()
    return out


@pytest.mark.parametrize("symmetric", [1, 0])
def test_small_instances(symmetric):
    print("small batch symmetric=%d" % symmetric, flush=True)
    sizes = [2, 20, 31, 32, 33, 63, 64, 65, 95, 97, 127, 129, 191, 193, 255, 256, 257, 319, 511, 513] * 3
    inst = [ics.collision(n, seed=k) for k, n in enumerate(sizes)]
    got = batch_of(inst, [("batch_symmetric", symmetric)])
    one = g.Context(0)
    one.set_option("sweep_slices", 1)
    for k, (h, prm) in enumerate(inst):
        d = g.DeviceParticles.from_host(h)
        one.compute_derivatives(d, prm)
        g.hip.synchronize()
        ref = d.download(FIELDS)
        d.free()
        for f in FIELDS:
            if f == "acc" and symmetric:  # sums of at most 64 plain FP32 terms, in other shares
                mx, norm = vec_errors(got[k][f], ref[f])
                assert norm < 1e-6, (sizes[k], mx, norm)
            else:
                assert np.array_equal(got[k][f].view(np.uint32), ref[f].view(np.uint32)), (sizes[k], f)
    one.close()


@pytest.mark.parametrize("soft", [True, False])
def test_in_group_blocks_of_64_and_256(soft):
    print("in-group blocks soft=%s" % soft, flush=True)
    few = [ics.plummer(n, seed=n) for n in (256, 250, 1, 1024, 1500)]
    for h, prm in few:
        prm.H = prm.H if soft else 0.0
    filler = ics.plummer(256, seed=9)
    filler[1].H = few[0][1].H
    a, b = batch_of(few), batch_of(few + [filler] * 520)
    for k in range(len(few)):
        assert np.array_equal(a[k]["acc"].view(np.uint32), b[k]["acc"].view(np.uint32)), k
