"""The far field's softened pair block (csrc/far_rotation.hpp) at the edges of
its tiles: one far group of a single particle, a last chunk that is partly
empty, whole groups, equal and unequal masses, against the FP64 oracle."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("n", [1025, 1039, 2048, 2065, 3583])
def test_far_pairs_match_fp64(n, uniform):
    print("far rotation n=%d uniform=%s" % (n, uniform), flush=True)
    h, prm = ics.plummer(n, seed=n)
    if not uniform:
        h["posm"][:, 3] *= np.random.default_rng(n).uniform(0.5, 2.0, size=n).astype(np.float32)
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", 1)
    d = g.DeviceParticles.from_host(h)
    ctx.compute_derivatives(d, prm)
    g.hip.synchronize()
    got = d.download(["acc"])["acc"]
    d.free()
    ctx.close()
    ref = O.compute_derivatives(prm, h, "f64")["acc"]
    mx, norm = vec_errors(got, ref)
    # a slot adds at most 512 terms in plain FP32 before they are compensated: random-walk rounding of
    # sqrt(512) half-ulps is 7e-7 of the partial sums, a tenth of that norm-wise over ~10 partials
    assert mx < 1e-5 and norm < 1e-6, (mx, norm)


# Rows cut into shares of 16 partners: a last group of one particle (all its
# shares but one lie past the end), of one whole chunk, of one particle more;
# folds every 128 partners (below 131072 particles) and every 512 (from there),
# against the one-sided sweep, which is compensated.
@pytest.mark.parametrize("n", [17 * 1024 + 1, 18 * 1024 + 16, 18 * 1024 + 17, 131071, 128 * 1024 + 1])
def test_far_shares(n):
    print("far shares n=%d" % n, flush=True)
    h, prm = ics.plummer(n, seed=n)
    h["posm"][:, 3] *= np.random.default_rng(n).uniform(0.5, 2.0, size=n).astype(np.float32)
    out = []
    for symmetric in (1, 0):
        ctx = g.Context(0)
        ctx.set_option("sweep_symmetric", symmetric)
        d = g.DeviceParticles.from_host(h)
        ctx.compute_derivatives(d, prm)
        g.hip.synchronize()
        out.append(d.download(["acc"])["acc"])
        d.free()
        ctx.close()
    mx, norm = vec_errors(out[0], out[1])
    # both sides within the bound above of the exact sums
    assert mx < 2e-5 and norm < 1e-6, (mx, norm)


# Below 65536 particles every run of partners decides for itself whether its
# row's slots have one mass and its partners one: two masses (most runs have
# one on each side, some another on each), one particle that differs, all.
@pytest.mark.parametrize("masses", ["two", "one differs", "none equal"])
@pytest.mark.parametrize("soft", [True, False])
def test_far_runs_of_one_mass(masses, soft):
    n = 5000
    print("far masses %s soft=%s" % (masses, soft), flush=True)
    h, prm = ics.plummer(n, seed=7)
    m = h["posm"][:, 3]
    if masses == "two":
        m[n // 3:] *= np.float32(1.7)
    elif masses == "one differs":
        m[n - 40] *= np.float32(3.0)
    else:
        m *= np.random.default_rng(7).uniform(0.5, 2.0, size=n).astype(np.float32)
    if not soft:
        prm.H = 0.0
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", 1)
    d = g.DeviceParticles.from_host(h)
    ctx.compute_derivatives(d, prm)
    g.hip.synchronize()
    got = d.download(["acc"])["acc"]
    d.free()
    ctx.close()
    mx, norm = vec_errors(got, O.compute_derivatives(prm, h, "f64")["acc"])
    # as above; without softening the closest pairs' FP32 separations carry up to 2^-24 |x| / r each
    assert (mx < 1e-5 and norm < 1e-6) if soft else (mx < 1e-3 and norm < 1e-4), (mx, norm)
