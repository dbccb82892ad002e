"""Neighbour lists where the slot order keeps no neighbours together
(csrc/lists.hip: the boxes of 64 slots taken whole): particles in random order
that are never sorted, and a body that one stray particle leaves in a few cells
of the curve; counts against an all-pairs search, sums against the FP64 oracle."""
import numpy as np
import pytest

import grasph2_amd as g
from oracle import pyoracle as O

from tests.test_gpu_lists import brute_counts, particles

pytestmark = pytest.mark.gpu


# more than 32 boxes of 64 (from 2049 particles), rounds of 64 and 128 of them, through boxes of 512 from 8193
@pytest.mark.parametrize("how", ["unsorted", "stray"])
@pytest.mark.parametrize("n,spacings", [(2048, 2.5), (2049, 2.5), (2111, 2.5), (4161, 2.5), (8193, 2.5), (8193, 6.0), (16500, 2.5)])
def test_counts_without_order(how, n, spacings):
    print("list order %s n=%d spacings=%g" % (how, n, spacings), flush=True)
    rng = np.random.default_rng(n)
    h, prm = particles("ball", n, rng)
    prm.H = spacings * (4.2 / n) ** (1.0 / 3.0)
    mix = rng.permutation(n)
    h["posm"] = h["posm"][mix]
    ctx = g.Context(0)
    if how == "unsorted":
        ctx.set_option("reorder_interval", 0)
    else:
        h["posm"][n // 3, :3] = 3000.0
    h["pos64"][:] = h["posm"][:, :3].astype(np.float64).T
    d = g.DeviceParticles.from_host(h)
    ctx.calc_density(d, prm)
    pairs, mx, over = ctx.neighbour_stats()
    rho = d.download(["density"])["density"]
    d.free()
    ctx.close()
    want = brute_counts(h["posm"][:, :3], prm.H)
    assert (pairs, mx) == (int(want.sum()), int(want.max()))
    assert over == int(np.count_nonzero(want > 160))
    ref = O.calc_density(prm, h, "f64")["density"]
    # half-ulp terms, compensated sums
    assert np.linalg.norm(rho - ref) <= 1e-6 * np.linalg.norm(ref)
