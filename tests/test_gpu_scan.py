"""The scan of a particle whose list overflowed (csrc/nbr_passes.hip) collects
its neighbours 16 or 4 at a time: capacity 1 against ample capacity, bit for
bit, for lists of every length around those, in the boxes of 64 and 512 slots
that end inside the instance, single and in a batch (4 lanes)."""
import numpy as np
import pytest

import grasph2_amd as g

from tests.test_gpu_passes import run, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["solid", "xsph"])
@pytest.mark.parametrize("n,reach", [(3, 4.0), (6, 4.0), (18, 4.0), (40, 1.0), (65, 0.6), (65, 4.0), (513, 0.5), (577, 1.0),
                                     (1100, 1.3), (25000, 0.8)])
def test_scan_equals_list(kind, n, reach):
    print("scan kind=%s n=%d reach=%g" % (kind, n, reach), flush=True)
    h, prm = workload(kind, n)
    prm.H *= reach
    full, scan = run(h, prm, 4096), run(h, prm, 1)
    for f in full:
        assert np.array_equal(full[f].view(np.uint32), scan[f].view(np.uint32)), f
    host, offsets = g.pack_batch([h, h])
    ctx = g.Context(0)
    ctx.set_option("max_neighbours", 1)
    d = g.DeviceParticles.from_host(host)
    ctx.batch_compute_derivatives(d, ctx.batch(offsets, [prm, prm]))
    g.hip.synchronize()
    for got in g.unpack_batch(d.download(list(full)), offsets):
        for f in full:
            assert np.array_equal(full[f].view(np.uint32), got[f].view(np.uint32)), f
    d.free()
    ctx.close()
