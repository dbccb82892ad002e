"""Shapes of the one-sided sweep (own_plan, csrc/capi.hip) at larger counts, with
256 compute units: counts where four lanes a slot would be chosen but for the
equal-mass rule, equal and unequal masses, against the symmetric sweep; and four
slots per lane against two with the same shares."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


def acc_of(h, prm, options):
    ctx = g.Context(0)
    for k, v in options.items():
        ctx.set_option(k, v)
    d = g.DeviceParticles.from_host(h)
    ctx.compute_derivatives(d, prm)
    g.hip.synchronize()
    a = d.download(["acc"])["acc"]
    d.free()
    ctx.close()
    return a


def case(n, uniform):
    h, prm = ics.plummer(n, seed=n)
    if not uniform:
        h["posm"][:, 3] *= np.random.default_rng(n).uniform(0.5, 2.0, size=n).astype(np.float32)
    return h, prm


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("n", [24575, 24576, 40000, 45000])
def test_past_the_mass_check(n, uniform):
    print("one-sided shapes n=%d uniform=%s" % (n, uniform), flush=True)
    h, prm = case(n, uniform)
    # both within 1e-7 of the exact sums norm-wise: chains of at most 128 plain FP32 terms, compensated
    mx, norm = vec_errors(acc_of(h, prm, {"sweep_symmetric": 0}), acc_of(h, prm, {"sweep_symmetric": 1}))
    assert norm < 1e-6 and mx < 2e-5, (mx, norm)


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("slices", [6, 7, 8])
def test_four_slots_a_lane(slices, uniform):
    """At 33000 particles 6 to 8 shares are taken by four slots a lane, in one
    plane; by two with sweep_i_per_lane = 2."""
    print("four slots a lane slices=%d uniform=%s" % (slices, uniform), flush=True)
    h, prm = case(33000, uniform)
    a = acc_of(h, prm, {"sweep_symmetric": 0, "sweep_slices": slices})
    b = acc_of(h, prm, {"sweep_symmetric": 0, "sweep_slices": slices, "sweep_i_per_lane": 2})
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
