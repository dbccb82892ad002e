"""The neighbour lists (csrc/lists.hip) at the edges of their boxes and tiles:
counts against a plain FP32 search over all pairs (the test rounds every
product and sum, so the counts are equal, not close), and the sums over the
lists against the FP64 oracle."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def brute_counts(pos, H):
    """Partners j of every i with 0 < r^2 <= H^2 in FP32, as the oracle rounds them."""
    p = np.ascontiguousarray(pos, dtype=np.float32)
    H2 = np.float32(H) * np.float32(H)
    out = np.zeros(len(p), dtype=np.int64)
    for i in range(len(p)):
        d = p[i] - p
        r2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
        out[i] = np.count_nonzero((r2 > 0) & (r2 <= H2))
    return out


def particles(kind, n, rng):
    if kind == "ball":
        h, prm = ics.liquid_blob(n, seed=n)
    else:
        h, prm = ics.liquid_blob(max(n, 2), seed=n)
        x = rng.uniform(-1, 1, size=(n, 3))
        if kind == "far":  # two clumps a thousand radii apart
            x[n // 2:] += [1000.0, 3.0, -2.0]
        elif kind == "plane":
            x[:, 2] = 0.25
        elif kind == "coincident":
            x = np.repeat(x[: max(1, n // 4)], 4, axis=0)[:n]
            x = np.concatenate([x, rng.uniform(-1, 1, size=(n - len(x), 3))])
        h = {f: a[..., :n] if a.ndim == 2 and f in ("pos64",) else a[:n] for f, a in h.items()}
        h = {f: np.ascontiguousarray(a) for f, a in h.items()}
        h["posm"][:, :3] = x
        h["pos64"][:] = h["posm"][:, :3].astype(np.float64).T
        prm.H = 0.3
    prm.flags &= ~g.SELF_GRAVITY
    return h, prm


@pytest.mark.parametrize("kind", ["ball", "far", "plane", "coincident"])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 64, 65, 511, 513, 1500])
def test_counts_equal_all_pairs_search(kind, n):
    print("lists kind=%s n=%d" % (kind, n), flush=True)
    h, prm = particles(kind, n, np.random.default_rng(n))
    ctx = g.Context(0)
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
    # half-ulp terms, compensated sum (norm-wise: single partners at the kernel's edge leave densities near 0)
    assert np.linalg.norm(rho - ref) <= 1e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("sizes", [(1, 513, 8, 700), (64, 1, 1, 1025)])
def test_batch_counts_equal_single_instances(sizes):
    print("lists batch sizes=%s" % (sizes,), flush=True)
    inst = [particles("ball" if n > 1 else "plane", n, np.random.default_rng(n)) for n in sizes]
    host, offsets = g.pack_batch([h for h, _ in inst])
    ctx = g.Context(0)
    d = g.DeviceParticles.from_host(host)
    ctx.batch_compute_derivatives(d, ctx.batch(offsets, [p for _, p in inst]))
    g.hip.synchronize()
    got = g.unpack_batch(d.download(["density", "acc"]), offsets)
    d.free()
    one = g.Context(0)
    for k, (h, prm) in enumerate(inst):
        dk = g.DeviceParticles.from_host(h)
        one.compute_derivatives(dk, prm)
        g.hip.synchronize()
        ref = dk.download(["density", "acc"])
        dk.free()
        assert np.array_equal(got[k]["density"], ref["density"])
        assert np.array_equal(got[k]["acc"], ref["acc"])
    ctx.close()
    one.close()


@pytest.mark.parametrize("kind", ["ball", "coincident"])  # all keys differ; many are the same
@pytest.mark.parametrize("n", [31, 33, 1025, 16384, 16385])
def test_order_by_rank_and_by_sort(kind, n):
    """Slots from the rank kernel (up to 16384 particles) and from the sort: a
    slot left out or filled twice would change the counts."""
    print("order kind=%s n=%d" % (kind, n), flush=True)
    h, prm = particles(kind, n, np.random.default_rng(n))
    prm.H = min(prm.H, 2.5 * (4.2 / n) ** (1.0 / 3.0))
    ctx = g.Context(0)
    d = g.DeviceParticles.from_host(h)
    ctx.calc_density(d, prm)
    pairs, mx, _ = ctx.neighbour_stats()
    d.free()
    ctx.close()
    want = brute_counts(h["posm"][:, :3], prm.H)
    assert (pairs, mx) == (int(want.sum()), int(want.max()))


# boxes of 64 tested directly up to 8192 particles, from there through the boxes of 512 (64 of them a round: two
# rounds from 32769); with H of 12 spacings every box is near and the collected ones are worked off in between
@pytest.mark.parametrize("n,spacings", [(4097, 12.0), (8192, 2.5), (8193, 2.5), (8193, 12.0), (33000, 2.5)])
def test_counts_at_edges_of_the_box_search(n, spacings):
    print("box search n=%d spacings=%g" % (n, spacings), flush=True)
    h, prm = particles("ball", n, np.random.default_rng(n))
    prm.H = spacings * (4.2 / n) ** (1.0 / 3.0)
    ctx = g.Context(0)
    d = g.DeviceParticles.from_host(h)
    ctx.calc_density(d, prm)
    pairs, mx, over = ctx.neighbour_stats()
    d.free()
    ctx.close()
    want = brute_counts(h["posm"][:, :3], prm.H)
    assert (pairs, mx) == (int(want.sum()), int(want.max()))
    assert over == int(np.count_nonzero(want > 160))
