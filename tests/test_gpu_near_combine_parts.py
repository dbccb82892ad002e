"""In-group gravity and combine in one launch (near_combine_kernel, 8 parts of the
combine) against the two launches (option sym_near_shares) where those take 4 and 2
parts: counts from 24576 to 65535, the last group and workgroup partly empty."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [24577, 40001, 49153, 65535])
def test_other_parts(n):
    print("near combine parts n=%d" % n, flush=True)
    h, prm = ics.plummer(n, seed=n)
    out = []
    for shares in (0, 4):
        ctx = g.Context(0)
        ctx.set_option("sweep_symmetric", 1)
        ctx.set_option("sym_near_shares", shares)
        d = g.DeviceParticles.from_host(h)
        ctx.compute_derivatives(d, prm)
        g.hip.synchronize()
        out.append(d.download(["acc"])["acc"])
        d.free()
        ctx.close()
    # the same terms in both, compensated but for the far field's chains, which are the same:
    # two roundings of the result and second-order ones of the sums
    mx, norm = vec_errors(out[0], out[1])
    assert norm < 2.4e-7 and mx < 1e-6, (mx, norm)
