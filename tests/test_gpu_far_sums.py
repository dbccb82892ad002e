"""Plain FP32 chains of the gravity sums, alone.  The far field's own side
(csrc/sym_sweep.hip): every group but
the last in one point, the last group's particles in another, so that each far
pair's factor is a power of two (r^2 + H^2 = 16, dx = 2: m_j / 32 exactly) or
nothing.  What a slot of the first groups is off by is the rounding of its sum
of the last group's masses, and no two rows cut those partners the same way."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

pytestmark = pytest.mark.gpu


def own_sums(n, masses):
    """32 acc_x of every slot before the last group, whose particles have `masses`."""
    first = (n - 1) // 1024 * 1024
    h = g.host_particles(n, ("posm", "vel", "acc"))
    h["posm"][:, 3] = np.random.default_rng(n).uniform(1.0, 2.0, size=n).astype(np.float32)
    h["posm"][first:, :3] = 2.0
    h["posm"][first:, 3] = masses[:n - first]
    prm = ics.plummer_params(2.0)
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", 1)
    d = g.DeviceParticles.from_host(h)
    ctx.compute_derivatives(d, prm)
    g.hip.synchronize()
    a = d.download(["acc"])["acc"][:first, :3].astype(np.float64)
    d.free()
    ctx.close()
    assert np.array_equal(a[:, 0], a[:, 1]) and np.array_equal(a[:, 0], a[:, 2])
    return 32.0 * a[:, 0]


@pytest.mark.parametrize("n", [5 * 1024, 11 * 1024, 16 * 1024])  # a wavefront has 16, 32 and 64 partners
def test_merged_wavefronts_lose_nothing(n):
    """Integer masses of 18 bits: a wavefront's sum (at most 64 of them) is
    exact, eight wavefronts' need up to 27 bits, and the whole one, an odd
    number just below the middle between two floats, has to round down."""
    print("far merge n=%d" % n, flush=True)
    m = np.random.default_rng(n).integers(1 << 17, 1 << 18, size=1024)
    total = int(m.sum())
    ulp = 1 << (total.bit_length() - 24)
    m[0] += ulp // 2 - 1 - total % ulp
    total = int(m.sum())
    assert total % ulp == ulp // 2 - 1
    got = own_sums(n, m.astype(np.float32))
    assert np.all(got == total - total % ulp)


@pytest.mark.parametrize("groups", [162, 196, 256])
def test_own_chains(groups):
    """Masses in [1, 2).  Adding k like terms in plain FP32 is off by
    2^-23 0.12 sqrt(k) of the sum (rms; half a unit in the last place, uniform,
    a step).  128 at most a chain: 1.6e-7 / sqrt(1024 / 128), then at most 16 such
    sums, 5.7e-8, and the result's own 1.7e-8: 8.2e-8 in all.  Rows differ in
    where their chains begin; the bound leaves a factor 1.4 for the sample."""
    n = 1024 * groups
    print("far chains groups=%d" % groups, flush=True)
    m = np.random.default_rng(groups).uniform(1.0, 2.0, size=1024).astype(np.float32)
    got = own_sums(n, m)[::1024]
    total = m.astype(np.float64).sum()
    rms = np.sqrt(np.mean((got / total - 1.0) ** 2))
    assert rms < 1.15e-7, rms


@pytest.mark.parametrize("symmetric,waves,slices", [(1, 0, 0), (1, 4, 0), (0, 0, 1), (0, 0, 3)])
def test_in_group_and_one_sided_chains(symmetric, waves, slices):
    """Inside a group, or one-sided, 64 slots in one point and the 960 others, masses in
    [1, 2), in the other.  As above with 64 a chain, 15 of them: 1.15e-7 /
    sqrt(960 / 64), and the result's own 1.7e-8: 3.4e-8, times 1.4 for the sample."""
    print("in-group chains sym=%d waves=%d slices=%d" % (symmetric, waves, slices), flush=True)
    ctx = g.Context(0)
    ctx.set_option("sweep_symmetric", symmetric)
    ctx.set_option("sym_near_shares", waves)
    ctx.set_option("sweep_slices", slices)
    prm = ics.plummer_params(2.0)
    off = []
    for seed in range(64):
        h = g.host_particles(1024, ("posm", "vel", "acc"))
        h["posm"][:, 3] = np.random.default_rng(seed).uniform(1.0, 2.0, size=1024).astype(np.float32)
        h["posm"][:960, :3] = 2.0
        d = g.DeviceParticles.from_host(h)
        ctx.compute_derivatives(d, prm)
        g.hip.synchronize()
        got = 32.0 * d.download(["acc"])["acc"][960:, 0].astype(np.float64)
        d.free()
        off.append(got / h["posm"][:960, 3].astype(np.float64).sum() - 1.0)
    ctx.close()
    rms = np.sqrt(np.mean(np.square(off)))
    assert rms < 4.8e-8, rms
