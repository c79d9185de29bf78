"""distance() by a wavefront per query (single calls, and FAST batches of
contexts holding merged BVs) against the one-lane kernel and the oracle: the
smallest meshes, every output and statistic, ties, merged BVs."""
import numpy as np
import pytest
import torch

import fcl_amd as F
import fclo
from test_gpu_parity import _t

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _batch(ctx, m, tf1, tf2, engine):
    n = len(tf1)
    d = torch.zeros(n, dtype=torch.float64, device=DEV)
    p = torch.zeros((n, 6), dtype=torch.float64, device=DEV)
    i = torch.zeros((n, 2), dtype=torch.int32, device=DEV)
    st = [torch.zeros(n, dtype=torch.int64, device=DEV) for _ in range(2)]
    s = torch.cuda.current_stream().cuda_stream
    ctx.distance_batch_async(_t(np.tile(np.array(m, np.int32), (n, 1)), torch.int32),
                             _t(tf1, torch.float64), _t(tf2, torch.float64), d, p, i,
                             engine=engine, bv_tests=st[0], leaf_tests=st[1], stream=s)
    ctx.sync(s)
    return [x.cpu().numpy() for x in (d, p, i, st[0], st[1])]


@pytest.mark.parametrize("bv", [F.RSS, F.OBBRSS])
@pytest.mark.parametrize("ka,kb,lo,hi", [(1, 1, 0.0, 3.0), (1, 9, 1.0, 3.0), (9, 9, 1.5, 2.6),
                                         (17, 5, 2.2, 6.0)])
def test_single_calls_match_the_oracle(ctx, bv, ka, kb, lo, hi):
    A, B = F.icosphere(ka, 0.15, 31), F.icosphere(kb, 0.15, 32)
    print("case: clearance %d %d %g %g bv=%d" % (ka, kb, lo, hi, bv), flush=True)
    m = [ctx.mesh(*A, bv), ctx.mesh(*B, bv)]
    o = [fclo.OracleMesh(*A, bv), fclo.OracleMesh(*B, bv)]
    tf1, tf2 = F.poses(12, 1, lo, hi, 0xD15)
    want = _batch(ctx, m, tf1, tf2, F.ENGINE_PLAIN)
    od = fclo.distance_batch(o, np.tile([0, 1], (12, 1)), tf1, tf2)[0]
    assert np.array_equal(want[0], od)
    for q in range(12):
        d, pts, ids, stats = ctx.distance(m[0], tf1[q], m[1], tf2[q])
        assert d == want[0][q] and np.array_equal(pts.reshape(6), want[1][q])
        assert np.array_equal(ids, want[2][q])
        assert stats.tolist() == [want[3][q], want[4][q]]


def test_ties_keep_the_first_pair(ctx):
    """Two flat grids face to face: whole rows of triangle pairs at one
    distance."""
    V, T = F.heightfield(9, 0.0, 1)
    m = [ctx.mesh(V, T, F.RSS), ctx.mesh(V, T, F.RSS)]
    print("case: clearance ties", flush=True)
    tf = np.tile(np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0], float), (5, 1))
    tf2 = tf.copy()
    tf2[:, 11] = [0.5, 0.25, 1.0, 2.0, 0.0]
    want = _batch(ctx, m, tf, tf2, F.ENGINE_PLAIN)
    for q in range(5):
        d, pts, ids, stats = ctx.distance(m[0], tf[q], m[1], tf2[q])
        assert d == want[0][q] and np.array_equal(ids, want[2][q])
        assert np.array_equal(pts.reshape(6), want[1][q])
        assert stats.tolist() == [want[3][q], want[4][q]]


def test_merged_bvs_follow_the_reference_order(ctx):
    A, B = F.icosphere(9, 0.15, 41), F.icosphere(8, 0.15, 42)
    local = F.Context(0)
    print("case: clearance, merged BVs", flush=True)
    m = [local.mesh(*A, F.RSS), local.mesh(*B, F.RSS)]
    local.mesh_refit(m[0], torch.from_numpy(A[0] * 1.05).to(DEV), bottomup=True)
    tf1, tf2 = F.poses(150, 1, 1.9, 3.0, 0xD16)
    want = _batch(local, m, tf1, tf2, F.ENGINE_PLAIN)
    got = _batch(local, m, tf1, tf2, F.ENGINE_FAST)
    assert all(np.array_equal(a, b) for a, b in zip(got, want))
    local.close()


@pytest.mark.parametrize("mode,n", [(2, 300), (0, 2047), (0, 2048), (0, 65536 + 5)])
def test_lanes_give_the_wavefronts_answers(mode, n):
    """Merged BVs with a lane per query -- forced, and by the rule with light
    and heavy queries and bad ids in one batch -- against wavefronts."""
    print("case: clearance lanes mode=%d n=%d" % (mode, n), flush=True)
    local = F.Context(0)
    tri = np.array([[0.9, 0, 0], [-0.4, 0.8, 0], [-0.4, -0.8, 0.1]]), np.array([[0, 1, 2]])
    heavy = F.icosphere(3, 0.15, 8)
    m = np.array([local.mesh(*x, F.RSS) for x in (tri, F.icosphere(1, 0.1, 9), heavy)], np.int32)
    local.mesh_refit(int(m[1]), torch.from_numpy(F.icosphere(1, 0.1, 9)[0] * 1.05).to(DEV),
                     bottomup=True)
    qm = m[np.random.default_rng(n).integers(0, 3, (n, 2))]
    qm[5::500, 1] = -1
    tf1, tf2 = F.poses(n, 1, 1.9, 4.0, 0xD17)
    out = []
    for v in (1, mode):
        local.set_engine_param("ordered_lanes", v)
        d = torch.full((n,), -1, dtype=torch.float64, device=DEV)
        p = torch.zeros((n, 6), dtype=torch.float64, device=DEV)
        i = torch.full((n, 2), -7, dtype=torch.int32, device=DEV)
        st = [torch.full((n,), -1, dtype=torch.int64, device=DEV) for _ in range(2)]
        s = torch.cuda.current_stream().cuda_stream
        local.distance_batch_async(_t(qm, torch.int32), _t(tf1, torch.float64),
                                   _t(tf2, torch.float64), d, p, i, engine=F.ENGINE_FAST,
                                   bv_tests=st[0], leaf_tests=st[1], stream=s)
        assert local.sync_status(s) != 0
        good = torch.from_numpy((qm >= 0).all(1)).to(DEV)
        out.append([d, i] + st + [p[good]])
    assert all(torch.equal(a, b) for a, b in zip(*out))
    local.close()
