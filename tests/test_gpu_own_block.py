"""The one-sided gravity of csrc/own_block.hpp (one-sided sweep, batches,
pairs inside a group) at the edges of its tiles and shares: particle counts
around 64, 256 and the shares' lengths, both sides of the equal-mass rule and
of the one / four slots per lane rule, against the FP64 oracle; and shares,
lanes and wavefronts that must not change a bit."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


def acc_of(ctx, h, prm):
    d = g.DeviceParticles.from_host(h)
    ctx.compute_derivatives(d, prm)
    g.hip.synchronize()
    a = d.download(["acc"])["acc"]
    d.free()
    return a


def case(n, uniform, soft=True):
    h, prm = ics.plummer(n, seed=n)
    if not uniform:
        h["posm"][:, 3] *= np.random.default_rng(n).uniform(0.5, 2.0, size=n).astype(np.float32)
    if not soft:
        prm.H = 0.0
        h["posm"][n // 2, :3] = h["posm"][0, :3]  # coincident: nothing between them
        h["pos64"][:, n // 2] = h["pos64"][:, 0]
    return h, prm


@pytest.mark.parametrize("soft", [True, False])
@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 129, 1001, 6143, 6145, 8200])
def test_one_sided_matches_fp64(n, uniform, soft):
    print("own block n=%d uniform=%s soft=%s" % (n, uniform, soft), flush=True)
    h, prm = case(n, uniform, soft)
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", 0)
    got = acc_of(ctx, h, prm)
    ctx.close()
    ref = O.compute_derivatives(prm, h, "f64")["acc"]
    if not np.any(ref):  # one particle, or two in one place
        assert not np.any(got)
        return
    # at most 128 plain FP32 terms before they are compensated
    mx, norm = vec_errors(got, ref)
    assert mx < 1e-5 and norm < 1e-6, (mx, norm)


@pytest.mark.parametrize("n", [700, 7001])
def test_lanes_do_not_change_a_bit(n):
    """One, two or four slots per lane meet the same partners in the same order."""
    print("own block lanes n=%d" % n, flush=True)
    h, prm = case(n, False)
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", 0)
    ctx.set_option("sweep_slices", 4)
    a = acc_of(ctx, h, prm)
    ctx.set_option("sweep_i_per_lane", 2)
    b = acc_of(ctx, h, prm)
    ctx.close()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n", [1024, 2500])
@pytest.mark.parametrize("shares", [1, 3, 16])
def test_in_group_shares(n, shares):
    print("own block in-group n=%d shares=%d" % (n, shares), flush=True)
    h, prm = case(n, True)
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", 1)
    ctx.set_option("sym_near_shares", shares)
    got = acc_of(ctx, h, prm)
    ctx.close()
    mx, norm = vec_errors(got, O.compute_derivatives(prm, h, "f64")["acc"])
    assert mx < 1e-5 and norm < 1e-6, (mx, norm)
