"""Gravity of unequal masses in units far from 1: m / r is in FP32's range where
1 / r^3 alone is not (separations of 10^15: 1 / r^3 is 0; of 10^-15: infinite).
The one-sided sweep in its shapes, the pairs inside a group, and the symmetric
sweep at the counts where it has taken the one-sided sweep's place, against the
FP64 oracle."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("soft", [True, False])
@pytest.mark.parametrize("scale", [1e15, 1e-15])
@pytest.mark.parametrize("n,symmetric,call", [
    (100, 2, "compute_derivatives"), (1000, 2, "compute_derivatives"), (1000, 1, "compute_derivatives"),
    (7000, 2, "compute_derivatives"), (9000, 2, "compute_derivatives_noalloc"), (12345, 2, "compute_derivatives")])
def test_unequal_masses(n, symmetric, call, scale, soft):
    print("gravity range n=%d sym=%d scale=%g soft=%s" % (n, symmetric, scale, soft), flush=True)
    h, prm = ics.plummer(n, seed=n)
    h["posm"][:, :3] *= np.float32(scale)
    h["pos64"][:] = h["posm"][:, :3].astype(np.float64).T
    h["posm"][:, 3] *= np.random.default_rng(n).uniform(0.5, 2.0, size=n).astype(np.float32) * np.float32(scale)
    prm.H = prm.H * scale if soft else 0.0
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", symmetric)
    d = g.DeviceParticles.from_host(h)
    getattr(ctx, call)(d, prm)
    g.hip.synchronize()
    got = d.download(["acc"])["acc"]
    d.free()
    ctx.close()
    mx, norm = vec_errors(got, O.compute_derivatives(prm, h, "f64")["acc"])
    # a pair's factor carries 3 roundings and the root's error, the sums a few more: 5e-7 at most of a term;
    # without softening the closest pairs' FP32 separations carry up to 2^-24 |x| / r each
    assert (mx < 1e-5 and norm < 1e-6) if soft else (mx < 1e-3 and norm < 1e-4), (mx, norm)
