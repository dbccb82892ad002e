"""Shapes of the one-sided sweep's automatic choice (own_plan, csrc/capi.hip):
one and four slots per lane, full and half workgroups, several planes, a last
share and a last workgroup that are partly empty, against the same sweep in
one share per slot block (sweep_slices = 1)."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 127, 128, 511, 512, 1025, 1537, 4096, 4097, 5500, 9473, 11000, 14337])
def test_automatic_shares(n):
    print("one-sided shares n=%d" % n, flush=True)
    h, prm = ics.plummer(n, seed=n)
    out = []
    for slices in (0, 1):
        ctx = g.Context(0)
        ctx.set_option("sweep_symmetric", 0)
        ctx.set_option("sweep_slices", slices)
        d = g.DeviceParticles.from_host(h)
        ctx.compute_derivatives(d, prm)
        g.hip.synchronize()
        out.append(d.download(["acc"])["acc"])
        d.free()
        ctx.close()
    if n == 1:
        assert np.array_equal(out[0], out[1])
        return
    mx, norm = vec_errors(out[0], out[1])
    # sums of 128 terms in plain FP32 (rounding ~ sqrt(128) / 2 ulp = 3.4e-7 of their magnitude), compensated
    # from there, on both sides: well below 1e-6 norm-wise over the shares' independent roundings
    assert norm < 1e-6 and mx < 2e-5, (mx, norm)
