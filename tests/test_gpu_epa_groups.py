"""EPA by lane groups: batches around a group's and a block's size, of pairs
whose polytopes stay small, outgrow the small store, or reach the reference's
own limits, bit for bit against the oracle."""
import numpy as np
import pytest

import fcl_amd as F
import fclo
from fcl_amd import workloads as W
from test_gpu_shapes import check_parity

pytestmark = pytest.mark.gpu


def _curved(n, seed, flat):
    """Cylinder pairs and large convex pairs, most of them overlapping."""
    rng = np.random.default_rng(seed)
    types = np.where(np.arange(n) % 3 == 2, F.CONVEX, F.CYLINDER).repeat(2)
    dims = rng.uniform(0.3, 1.0, (2 * n, 3))
    dims[:, 1] *= flat
    conv = []
    for k in np.flatnonzero(types == F.CONVEX):
        v = rng.standard_normal((1 + k % 90, 3))  # one vertex, a few, more than the lanes
        conv.append(0.6 * v / np.linalg.norm(v, axis=1, keepdims=True))
    rec, pool = F.shape_table(types, dims, conv)
    ps = np.arange(2 * n, dtype=np.int32).reshape(n, 2)
    return rec, pool, ps, W.random_poses(n, rng, 0.25), W.random_poses(n, rng, 0.25)


@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("n", [1, 65, 2000])
def test_long_queues_run_a_lane_each(ctx, n, over):
    """On both sides of the queue length from which EPA runs a lane per pair."""
    rec, pool, ps, tf1, tf2 = _curved(n, 11 * n, 1.0)
    queue = int((fclo.shape_collide_batch(fclo.shapes_from_table(rec, pool), ps, tf1, tf2, 1, True,
                                          passes=True)[2][:, 1] > 0).sum())
    ctx.set_engine_param("epa_lanes_min", max(queue, 1) + over)
    try:
        check_parity(ctx, rec, pool, ps, tf1, tf2, 1, True, "lanes from %d EPA pairs" % (queue + over))
    finally:
        ctx.set_engine_param("epa_lanes_min", 240000)


@pytest.mark.parametrize("n", [1, 2, 15, 17, 33, 257, 6000])
@pytest.mark.parametrize("flat", [1.0, 0.02])
def test_small_and_full_stores(ctx, n, flat):
    rec, pool, ps, tf1, tf2 = _curved(n, 7 * n, flat)
    check_parity(ctx, rec, pool, ps, tf1, tf2, 1, True, "curved flat=%g" % flat)
    if n > 200:  # some pairs stay in the small store's 64 faces and some leave it
        passes = fclo.shape_collide_batch(fclo.shapes_from_table(rec, pool), ps, tf1, tf2, 1, True,
                                          passes=True)[2][:, 1]
        assert (passes > 32).sum() > n // 100 and ((passes > 0) & (passes < 12)).sum() > n // 100
