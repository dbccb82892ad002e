"""A captured evaluation reports no overflowed lists: replays in a state whose
lists overflow, then an eager call in a state whose lists do not, leave the
list capacity (and so the arrays the graph points to) as they were, and the
graph still gives the eager results."""
import numpy as np
import pytest

import grasph2_amd as g
from grasph2_amd import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["compute_derivatives", "calc_density"])
def test_replays_do_not_grow_the_lists(call):
    n = 3000
    print("capture lists %s n=%d" % (call, n), flush=True)
    h, prm = ics.collision(n, seed=11)
    dense = dict(h, posm=h["posm"].copy())
    dense["posm"][:, :3] *= np.float32(0.5)  # 8 times the neighbours
    ctx, ref = g.Context(0), g.Context(0)
    for c in (ctx, ref):
        c.set_option("max_neighbours", 128)
        c.set_option("reorder_interval", 1000)
    ref.set_option("max_neighbours_grow", 0)
    d, s = g.DeviceParticles.from_host(h), g.hip.Stream()
    for c in (ctx, ref):
        getattr(c, call)(d, prm, s)  # eager: slot order and work arrays
    s.synchronize()
    graph = g.hip.Graph(s, lambda st: getattr(ctx, call)(d, prm, st))
    for _ in range(3):
        d.upload(dense)
        getattr(ref, call)(d, prm, s)
        s.synchronize()
        assert ref.neighbour_stats()[1] > 128  # overflows
        want = d.download(["acc", "density"])
        d.upload(dense)
        graph.launch(s)
        s.synchronize()
        got = d.download(["acc", "density"])
        for f in want:
            assert np.array_equal(got[f].view(np.uint32), want[f].view(np.uint32)), f
        d.upload(h)
        for _ in range(2):
            getattr(ctx, call)(d, prm, s)  # eager, nothing overflows
            s.synchronize()
        assert ctx.get_option("max_neighbours") == 128
    d.free()
    ctx.close()
    ref.close()
