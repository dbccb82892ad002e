"""The batched far field's rows in 4, 8 and 16 pieces (sym_batch_tables,
csrc/sym_sweep.hip: finer where a batch has fewer pieces than wavefronts), rows with
fewer groups than pieces and a last group partly empty: every instance against the
same in the one-sided sweep."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

from tests._util import vec_errors

pytestmark = pytest.mark.gpu


# pieces a row at most, with 2048 wavefronts: 16 (few rows), 8 (1225 pieces at 4, 2345 at 8), 4
@pytest.mark.parametrize("sizes", [(2049, 17500, 1024, 30001), (30001,) * 11 + (1500,) * 4, (9000,) * 100])
def test_pieces(sizes):
    print("batch pieces sizes=%s..." % (sizes[:4],), flush=True)
    made = {n: ics.plummer(n, seed=n) for n in set(sizes)}
    for n, (h, _) in made.items():
        h["posm"][:, 3] *= np.random.default_rng(n).uniform(0.5, 2.0, size=n).astype(np.float32)
    inst = [made[n] for n in sizes]
    host, offsets = g.pack_batch([h for h, _ in inst])
    ctx = g.Context(0)
    d = g.DeviceParticles.from_host(host)
    b = ctx.batch(offsets, [p for _, p in inst])
    out = []
    for symmetric in (1, 0):
        ctx.set_option("batch_symmetric", symmetric)
        ctx.batch_compute_derivatives(d, b)
        g.hip.synchronize()
        out.append(g.unpack_batch(d.download(["acc"]), offsets))
    d.free()
    ctx.close()
    for n, x, y in zip(sizes, *out):
        # 512 plain FP32 terms a chain in the far field (sqrt(512) / 2 ulp = 7e-7 of the parts), compensated from there
        mx, norm = vec_errors(x["acc"], y["acc"])
        assert norm < 1e-6 and mx < 2e-5, (n, mx, norm)
