"""In-group gravity and combine in one launch (near_combine_kernel) against the
two launches (option sym_near_shares set), which add the same terms in another
number of parts, and against the FP64 oracle: a last group that is partly
empty, a last workgroup that is."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 5000, 12345])
def test_one_launch_and_two(n):
    print("near combine n=%d" % n, flush=True)
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
    if n == 1:
        assert np.all(out[0] == 0) and np.all(out[1] == 0)
        return
    ref = O.compute_derivatives(prm, h, "f64")["acc"]
    for got in out:  # sums of up to 512 plain FP32 terms, compensated from there (sqrt(512) / 2 ulp = 7e-7 of the parts)
        mx, norm = vec_errors(got, ref)
        assert mx < 1e-5 and norm < 1e-6, (mx, norm)
