"""The lists' layout (list_entry, csrc/internal.hpp): capacities that are multiples
of 4 and not, lists that fill them, just do not and overflow, with 16 and 4 lanes
per particle and in a batch whose instances begin inside a tile of 64 slots: the
same bits as with ample capacity."""
import numpy as np
import pytest

import grasph2_amd as g

from tests.test_gpu_passes import run, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 3000, 25000])
def test_capacities(n):
    h, prm = workload("solid", n)
    full = run(h, prm, 1024)
    ctx = g.Context(0)
    for kmax in (3, 4, 30, 57, 62, 64, 66, 100, 101, 600):
        print("list layout n=%d kmax=%d" % (n, kmax), flush=True)
        got = run(h, prm, kmax)
        for f in full:
            assert np.array_equal(full[f].view(np.uint32), got[f].view(np.uint32)), (kmax, f)
        if n > 3000:
            continue
        host, offsets = g.pack_batch([h, h, h])
        ctx.set_option("max_neighbours", kmax)
        d = g.DeviceParticles.from_host(host)
        ctx.batch_compute_derivatives(d, ctx.batch(offsets, [prm] * 3))
        g.hip.synchronize()
        for one in g.unpack_batch(d.download(list(full)), offsets):
            for f in full:
                assert np.array_equal(full[f].view(np.uint32), one[f].view(np.uint32)), (kmax, f)
        d.free()
    ctx.close()
