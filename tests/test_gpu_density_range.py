"""The acceleration pass divides by mean densities over FP32's whole range:
sums of two densities above 2^126 (whose reciprocal is denormal) and below
2^-126, against the FP64 oracle, with one lane count after the other."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [300, 25000])  # 16 and 4 lanes per particle
@pytest.mark.parametrize("rho,mass,speed", [(1.5e38, 1e20, 1e9), (1.0, 1e-3, 1.0), (2.0e-39, 1e-38, 1.0)])
def test_mean_density(n, rho, mass, speed):
    print("density range n=%d rho=%g" % (n, rho), flush=True)
    rng = np.random.default_rng(n)
    h, prm = ics.liquid_blob(n, seed=n, gravity=False)
    prm.flags |= g.XSPH
    prm.alpha = 1.0
    h["posm"][:, 3] = mass
    h["density"][:] = rho
    h["vel"][:, :3] = rng.normal(0.0, speed, size=(n, 3))
    ctx = g.Context(0)
    d = g.DeviceParticles.from_host(h)
    ctx.calc_acceleration(d, prm)
    g.hip.synchronize()
    got = d.download(["acc", "xvel"])
    d.free()
    ctx.close()
    ref = O.calc_acceleration(prm, h, "f64")
    # a pair's term carries about 10 FP32 roundings (6e-7), a sum of ~60 of either sign 8 times a term
    mx, norm = vec_errors(got["xvel"], ref["xvel"])
    assert norm < 1e-6, (mx, norm)
    if rho >= 1.0:  # below, rho^2 is 0 and the pressure term has no value
        mx, norm = vec_errors(got["acc"], ref["acc"])
        assert norm < 1e-6, (mx, norm)
