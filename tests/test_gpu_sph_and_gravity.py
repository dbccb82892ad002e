"""SPH terms and gravity meet in one rounding at the counts where the symmetric
sweep has taken the one-sided sweep's place: with gravity 10^-5 of the pressure
forces, what the two sweeps' gravity differs by (10^-7 of it) is 10^-5 of an ulp
of the result, so their accelerations have the same bits but for about one
component in 10^5; rounding the pressure forces before gravity joins them would
change about one in four."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [10752, 16383])
def test_one_rounding(n):
    print("sph and gravity n=%d" % n, flush=True)
    h, prm = ics.liquid_blob(n, seed=n)
    prm.flags &= ~g.ARTIFICIAL_VISCOSITY
    prm.SOUNDSPEED = 1000.0
    out = []
    for symmetric in (2, 0):
        ctx = g.Context(0)
        ctx.set_option("sweep_symmetric", symmetric)
        d = g.DeviceParticles.from_host(h)
        ctx.compute_derivatives(d, prm)
        g.hip.synchronize()
        out.append(d.download(["acc"])["acc"][:, :3])
        d.free()
        ctx.close()
    assert np.abs(out[0]).max() > 1e4
    assert np.mean(out[0].view(np.uint32) != out[1].view(np.uint32)) < 0.01
