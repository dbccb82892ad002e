"""Artificial viscosity in large units: with H of 10^8 m and speeds of mm/s the
viscosity times the kernel gradient lies below FP32's range (10^-40), times the
mass too it does not.  At rest density nothing else acts; against the FP64 oracle."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solid", [False, True])
@pytest.mark.parametrize("n", [300, 25000])  # 16 and 4 lanes per particle
def test_slow_flow_of_large_bodies(n, solid):
    print("viscosity range n=%d solid=%s" % (n, solid), flush=True)
    rng = np.random.default_rng(n)
    h, prm = ics.liquid_blob(n, seed=n, gravity=False, fields=ics.SOLID_FIELDS)
    scale, rho = 1e8 / prm.H, 1000.0
    if solid:
        prm = ics.solid_params(prm.H, gravity=False)
    prm.H, prm.rho0, prm.SOUNDSPEED = 1e8, rho, 1e-3
    prm.alpha = 1.0
    h["posm"][:, :3] *= np.float32(scale)
    h["pos64"][:] = h["posm"][:, :3].astype(np.float64).T
    h["posm"][:, 3] = rho * (4.2 / n) * scale ** 3
    h["density"][:] = rho
    h["balsara"][:] = 1.0
    h["vel"][:, :3] = rng.normal(0.0, 1e-3, size=(n, 3))
    ctx = g.Context(0)
    d = g.DeviceParticles.from_host(h)
    ctx.calc_acceleration(d, prm)
    g.hip.synchronize()
    got = d.download(["acc"])["acc"]
    d.free()
    ctx.close()
    # a pair's term carries about 10 FP32 roundings (6e-7), a sum of ~60 of either sign 8 times a term
    mx, norm = vec_errors(got, O.calc_acceleration(prm, h, "f64")["acc"])
    assert norm < 1e-6, (mx, norm)
