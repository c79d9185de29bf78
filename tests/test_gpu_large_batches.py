"""Batches beyond 2^26 queries (a wavefront each would be 2^32 threads, which
HIP refuses) and around the blocks that one launch takes: every query's answer
is that of the same pose in a small batch."""
import numpy as np
import pytest
import torch

import fcl_amd as F
from test_gpu_parity import collide_gpu

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
BLOCKS = 1 << 20  # most blocks of a launch
PAST = (1 << 26) + 33
PERIOD = 64  # poses that the batches repeat



@pytest.fixture(scope="module")
def poses():
    return F.poses(PERIOD, 0, 1.8, 0, 0xB16)


def _tiled(a, n, dtype):
    t = torch.from_numpy(np.ascontiguousarray(a)).to(DEV, dtype)
    out = torch.empty((n,) + t.shape[1:], dtype=dtype, device=DEV)
    out[:n - n % PERIOD].view(-1, *t.shape).copy_(t)
    out[n - n % PERIOD:] = t[:n % PERIOD]
    return out


def _repeats(got, want):
    """got is want over and over."""
    n = got.shape[0]
    w = torch.from_numpy(np.ascontiguousarray(want)).to(DEV)
    whole = got[:n - n % PERIOD].view(-1, *w.shape)
    return bool((whole == w).all()) and bool((got[n - n % PERIOD:] == w[:n % PERIOD]).all())


@pytest.mark.parametrize("n,cap,contact,lanes",
                         [(BLOCKS + 77, 2, True, 1), (4 * BLOCKS + 77, 1, False, 1),
                          (PAST, 2, False, 1), (PAST, 2, True, 1), (PAST, 1, False, 2)])
def test_collide(poses, n, cap, contact, lanes):
    print("case: %d collide queries, contact=%d lanes=%d" % (n, contact, lanes), flush=True)
    ctx = F.Context(0)
    ctx.set_engine_param("ordered_lanes", lanes)
    m = [ctx.mesh(*F.icosphere(2, 0.15, k)) for k in (1, 2)]
    want = collide_gpu(ctx, np.tile(np.array(m, np.int32), (PERIOD, 1)), *poses, cap)[1]
    if contact:
        want = np.array([len(ctx.collide_contact(m[0], poses[0][q], m[1], poses[1][q], cap=cap)[0])
                         for q in range(PERIOD)], np.int32)
    assert 0 < (want > 0).mean() < 1
    counts = torch.full((n,), -1, dtype=torch.int32, device=DEV)
    num = torch.zeros(1, dtype=torch.int64, device=DEV)
    rows = 1000
    pairs = torch.zeros((rows, 3), dtype=torch.int32, device=DEV)
    geo = tuple(torch.zeros((rows,) + k, dtype=torch.float64, device=DEV)
                for k in ((3,), (3,), ())) if contact else None
    qm = torch.tensor(m, dtype=torch.int32, device=DEV).repeat(n, 1)
    s = torch.cuda.current_stream().cuda_stream
    ctx.collide_batch_async(qm, _tiled(poses[0], n, torch.float64),
                            _tiled(poses[1], n, torch.float64), cap, counts, pairs, num,
                            engine=F.ENGINE_FAST, contact=geo, stream=s)
    ctx.sync_status(s)  # (more contacts than rows)
    assert _repeats(counts, want) and int(num.item()) == int(counts.long().sum())
    ctx.close()


@pytest.mark.parametrize("n", [PAST])
def test_distance_over_merged_bvs(n):
    print("case: %d distance queries" % n, flush=True)
    local = F.Context(0)
    local.set_engine_param("ordered_lanes", 1)
    V, T = F.icosphere(1, 0.0, 1)
    m = [local.mesh(V, T, F.RSS), local.mesh(*F.icosphere(1, 0.15, 2), F.RSS)]
    local.mesh_refit(m[0], torch.from_numpy(V * 0.1).to(DEV), bottomup=True)
    poses = F.poses(PERIOD, 1, 3.0, 6.0, 0xB16)
    want = [local.distance(m[0], poses[0][q], m[1], poses[1][q]) for q in range(PERIOD)]
    d = torch.zeros(n, dtype=torch.float64, device=DEV)
    points = torch.zeros((n, 6), dtype=torch.float64, device=DEV)
    ids = torch.zeros((n, 2), dtype=torch.int32, device=DEV)
    tests = torch.zeros((2, n), dtype=torch.int64, device=DEV)
    s = torch.cuda.current_stream().cuda_stream
    local.distance_batch_async(torch.tensor(m, dtype=torch.int32, device=DEV).repeat(n, 1),
                               _tiled(poses[0], n, torch.float64),
                               _tiled(poses[1], n, torch.float64), d, points, ids,
                               engine=F.ENGINE_FAST, bv_tests=tests[0], leaf_tests=tests[1],
                               stream=s)
    local.sync(s)
    assert _repeats(d, np.array([w[0] for w in want]))
    assert _repeats(points, np.stack([w[1].reshape(6) for w in want]))
    assert _repeats(ids, np.stack([w[2] for w in want]).astype(np.int32))
    for k in (0, 1):
        assert _repeats(tests[k], np.stack([w[3] for w in want])[:, k])
    local.close()


@pytest.mark.parametrize("n,lanes", [(BLOCKS + 77, 1), (PAST, 1), (PAST, 2)])
def test_mesh_against_primitives(poses, n, lanes):
    print("case: %d mesh-shape queries, lanes=%d" % (n, lanes), flush=True)
    ctx = F.Context(0)
    ctx.set_engine_param("ordered_lanes", lanes)
    mesh = ctx.mesh(*F.icosphere(4, 0.15, 1))
    rec, pool = F.shape_table([F.BOX], [(0.6, 0.4, 0.5)])
    shapes = torch.from_numpy(np.ascontiguousarray(rec).view(np.uint8)).to(DEV)
    pool = torch.from_numpy(pool).to(DEV)
    s = torch.cuda.current_stream().cuda_stream

    def run(k):
        counts = torch.full((k,), -1, dtype=torch.int32, device=DEV)
        zero = torch.zeros(k, dtype=torch.int32, device=DEV)
        ctx.mesh_shape_collide_batch_async(zero + mesh, shapes, pool, zero,
                                           _tiled(poses[0], k, torch.float64),
                                           _tiled(poses[1], k, torch.float64), 1, counts, stream=s)
        ctx.sync(s)
        return counts

    want = run(PERIOD).cpu().numpy()
    assert 0 < want.mean() < 1
    assert _repeats(run(n), want)
    ctx.close()


@pytest.mark.parametrize("n", [(1 << 24) + 5, 1 << 28])
def test_broadphase_sweep(ctx, n):
    """Unit boxes three apart in x, but for the last of each 1,024, which
    touches the first of the next."""
    print("case: %d boxes" % n, flush=True)
    lo = 3.0 * torch.arange(n, device=DEV, dtype=torch.float64)
    boxes = torch.zeros((n, 6), dtype=torch.float64, device=DEV)
    boxes[:, 0], boxes[:, 3], boxes[:, 4:] = lo, lo + 1, 1
    boxes[1023::1024, 3] += 2
    pairs = torch.full((n // 512, 2), 7, dtype=torch.int32, device=DEV)
    num = torch.zeros(1, dtype=torch.int64, device=DEV)
    s = torch.cuda.current_stream().cuda_stream
    ctx.broadphase_pairs_async(boxes, pairs, num, stream=s)
    ctx.sync(s)
    first = torch.arange(1023, n - 1, 1024, device=DEV, dtype=torch.int32)
    k = len(first)
    assert int(num.item()) == k
    assert bool((pairs[:k, 0] == first).all()) and bool((pairs[:k, 1] == first + 1).all())
    assert bool((pairs[k:] == -1).all())
