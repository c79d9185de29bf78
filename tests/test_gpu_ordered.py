"""The lane-group collide kernel against the one-lane FP64 kernel (PLAIN, which
the parity tests compare with the oracle): both group widths, list bounds,
matrices that are no rotations, and contact mode; every answer, order and
count equal."""
import numpy as np
import pytest
import torch

import fcl_amd as F
from fcl_amd import workloads as W
from test_gpu_parity import _t, collide_gpu

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.fixture(scope="module")
def pair(ctx):
    V, T = F.heightfield(24, 0.05, 5)
    return [ctx.mesh(*F.icosphere(7, 0.15, 3)), ctx.mesh(F.scale_to_radius(V, 1.0), T)]


def _same(ctx, qm, tf1, tf2, cap, stats):
    a = collide_gpu(ctx, qm, tf1, tf2, cap, engine=F.ENGINE_PLAIN, stats=stats)
    b = collide_gpu(ctx, qm, tf1, tf2, cap, engine=F.ENGINE_FAST, stats=stats)
    assert a[0] == b[0] == 0 and a[5] == b[5]
    assert np.array_equal(a[1], b[1])
    assert a[2].keys() == b[2].keys() and all(np.array_equal(a[2][q], b[2][q]) for q in a[2])
    assert np.array_equal(a[3], b[3]) and np.array_equal(a[4], b[4])
    return a


@pytest.mark.parametrize("n,cap,stats", [(65535, 1, False), (65536, 1, False), (65539, 1, False),
                                         (65536, 1, True), (1, 64, True), (257, 2, True),
                                         (300, 64, True), (300, 64, False)])
def test_groups_match_the_one_lane_kernel(ctx, pair, n, cap, stats):
    print("case: ordered groups n=%d cap=%d stats=%d" % (n, cap, stats), flush=True)
    tf1, tf2 = F.poses(n, 0, 1.7, 0, 0x0D + n)
    got = _same(ctx, np.tile(np.array(pair, np.int32), (n, 1)), tf1, tf2, cap, stats)
    assert n == 1 or 0 < (got[1] > 0).mean() < 1


def test_bad_queries_in_a_narrow_batch(ctx, pair):
    n = 65537
    print("case: ordered groups, bad queries n=%d" % n, flush=True)
    tf1, tf2 = F.poses(n, 0, 1.7, 0, 0xBAD)
    qm = np.tile(np.array(pair, np.int32), (n, 1))
    bad = np.arange(0, n, 5)
    qm[bad, 1] = 9999
    rc, counts, per_q, _, _, _ = collide_gpu(ctx, qm, tf1, tf2, 1, engine=F.ENGINE_FAST,
                                             stats=False)
    assert rc != 0 and not counts[bad].any()
    good = np.setdiff1d(np.arange(n), bad)
    _, want, _, _, _, _ = collide_gpu(ctx, qm[good], tf1[good], tf2[good], 1, stats=False)
    assert np.array_equal(counts[good], want)


@pytest.mark.parametrize("scale", [1.0, 1.3, 40.0])
def test_matrices_that_are_no_rotations(ctx, pair, scale):
    """A scaled or sheared matrix is outside the FP32 cull's margin: the
    single call and the batches answer as FP64 does."""
    n = 60
    print("case: ordered groups, scale %g" % scale, flush=True)
    tf1, tf2 = F.poses(n, 0, 1.7, 0, 0x5CA1)
    tf2[:, :9] *= scale
    tf1[:, 1] += 0.2 * (scale - 1)
    qm = np.tile(np.array(pair, np.int32), (n, 1))
    want = _same(ctx, qm, tf1, tf2, 3, True)
    for q in range(0, n, 7):
        pairs, stats = ctx.collide(pair[0], tf1[q], pair[1], tf2[q], cap=3)
        assert np.array_equal(pairs, want[2].get(q, np.zeros((0, 2))))
        assert stats.tolist() == [want[3][q], want[4][q]]


def test_a_full_list_of_hits(ctx):
    """Two terrains through each other with a cap no query reaches: hits pile
    up in the list behind open nodes."""
    m = [ctx.mesh(*F.heightfield(20, 0.05, s)) for s in (9, 10)]
    print("case: ordered groups, dense contacts", flush=True)
    tf1, tf2 = F.poses(1, 0, 0.0, 0, 1)
    tf2[0] = tf1[0]
    n = 3
    qm = np.tile(np.array(m, np.int32), (n, 1))
    a = collide_gpu(ctx, qm, np.tile(tf1, (n, 1)), np.tile(tf2, (n, 1)), 100000, capacity=1 << 16)
    pairs, stats = ctx.collide(m[0], tf1[0], m[1], tf2[0], cap=100000)
    assert len(pairs) > 200 and np.array_equal(pairs, a[2][0])
    assert stats.tolist() == [a[3][0], a[4][0]]


@pytest.mark.parametrize("scale", [1e-45, 1e-41, 1e-30, 1e30, 1e38])
def test_sizes_at_the_ends_of_floats(scale):
    """Coordinates that floats hold badly or not at all: the single calls and
    every batch answer as FP64 does."""
    n = 80
    print("case: ordered groups, sizes of %g" % scale, flush=True)
    local = F.Context(0)
    A, B = F.icosphere(5, 0.15, 3), F.icosphere(5, 0.15, 4)
    m = [local.mesh(A[0] * scale, A[1]), local.mesh(B[0] * scale, B[1])]
    tf1, tf2 = F.poses(n, 0, 1.7, 0, 0xE4D)
    tf1[:, 9:] *= scale
    tf2[:, 9:] *= scale
    qm = np.tile(np.array(m, np.int32), (n, 1))
    for cap in (1, 5):
        _same(local, qm, tf1, tf2, cap, True)
    # every contact: the batch gives each query's in any order
    want, got = [collide_gpu(local, qm, tf1, tf2, 100000, engine=e, capacity=1 << 20)
                 for e in (F.ENGINE_PLAIN, F.ENGINE_FAST)]
    assert want[0] == got[0] == 0 and want[5] == got[5]
    assert all(np.array_equal(want[k], got[k]) for k in (1, 3, 4))
    for q, pairs in want[2].items():
        assert np.array_equal(*[p[np.lexsort(p.T)] for p in (pairs, got[2][q])])
    assert 0 < (want[1] > 0).mean() < 1
    for q in range(0, n, 3):
        pairs, stats = local.collide(m[0], tf1[q], m[1], tf2[q], cap=100000)
        assert np.array_equal(pairs, want[2].get(q, np.zeros((0, 2))))
        assert stats.tolist() == [want[3][q], want[4][q]]
    local.close()


@pytest.mark.parametrize("carry_max", [1, 9, 300])
def test_counts_at_the_carry_limit(pair, ctx, carry_max):
    """Test counts are summed in 64 bits, whatever the list may carry ahead."""
    n = 200
    print("case: ordered groups, carry limit %d" % carry_max, flush=True)
    tf1, tf2 = F.poses(n, 0, 1.7, 0, 0xCA)
    qm = np.tile(np.array(pair, np.int32), (n, 1))
    ctx.set_engine_param("ordered_carry_max", carry_max)
    try:
        for cap in (1, 3, 64):
            want = _same(ctx, qm, tf1, tf2, cap, True)
        _, stats = ctx.collide(pair[0], tf1[5], pair[1], tf2[5], cap=64)
        assert stats.tolist() == [want[3][5], want[4][5]]
    finally:
        ctx.set_engine_param("ordered_carry_max", 2**31)
    assert ctx.get_engine_param("ordered_carry_max") == 2**31


TRIANGLE = np.array([[0.9, 0, 0], [-0.4, 0.8, 0], [-0.4, -0.8, 0.1]]), np.array([[0, 1, 2]])
BOX = W.box_mesh(np.zeros(3), np.array([1.0, 1.1, 0.9]), 0.3)


def _answers(local, m, n, cap, contact, seed=5):
    tf1, tf2 = F.poses(n, 0, 1.4, 0, seed)
    counts = torch.full((n,), -1, dtype=torch.int32, device=DEV)
    num = torch.zeros(1, dtype=torch.int64, device=DEV)
    rows = n * min(cap, 12)
    pairs = torch.full((rows, 3), n, dtype=torch.int32, device=DEV)
    geo = [torch.zeros((rows,) + k, dtype=torch.float64, device=DEV) for k in ((3,), (3,), ())]
    tests = [torch.full((n,), -1, dtype=torch.int64, device=DEV) for _ in range(2)]
    s = torch.cuda.current_stream().cuda_stream
    local.collide_batch_async(_t(m, torch.int32), _t(tf1, torch.float64), _t(tf2, torch.float64),
                              cap, counts, pairs, num, engine=F.ENGINE_FAST, bv_tests=tests[0],
                              leaf_tests=tests[1], contact=geo if contact else None, stream=s)
    rc = local.sync_status(s)
    order = torch.argsort(pairs[:, 0], stable=True)
    return rc, [t.cpu().numpy() for t in [counts, num] + tests + [pairs[order]] +
                [g[order] for g in geo]]


@pytest.mark.parametrize("cap,contact", [(1, False), (3, False), (1, True), (4, True)])
@pytest.mark.parametrize("mode", [0, 2])
def test_lanes_give_the_groups_answers(cap, contact, mode):
    """A lane per query -- forced, and by the rule with light and heavy queries
    and bad ids in one batch -- against lane groups, all outputs equal."""
    n = 4000 if mode == 2 else 131072 + 77
    print("case: ordered lanes mode=%d cap=%d contact=%d" % (mode, cap, contact), flush=True)
    local = F.Context(0)
    m = [local.mesh(*TRIANGLE), local.mesh(*BOX), local.mesh(*F.icosphere(4, 0.15, 8))]
    qm = np.random.default_rng(cap).integers(0, 3, (n, 2)).astype(np.int32)
    qm = np.array(m, np.int32)[qm]
    qm[::1001, 0] = 77
    got = []
    for v in (1, mode):
        local.set_engine_param("ordered_lanes", v)
        got.append(_answers(local, qm, n, cap, contact))
    assert got[0][0] == got[1][0] != 0
    assert all(np.array_equal(a, b) for a, b in zip(got[0][1], got[1][1]))
    assert not got[0][1][0][::1001].any() and 0 < (got[0][1][0] > 0).mean() < 1
    local.close()


@pytest.mark.parametrize("n", [511, 512, 513, 32768])
@pytest.mark.parametrize("meshes", [(TRIANGLE, TRIANGLE), (TRIANGLE, BOX)])
def test_light_contexts(n, meshes):
    """Contexts whose every query is light, around the sizes where the rule
    changes, scaled matrices among them."""
    print("case: ordered lanes, light context n=%d" % n, flush=True)
    local = F.Context(0)
    m = np.array([local.mesh(*x) for x in meshes], np.int32)
    qm = np.tile(m, (n, 1))
    tf1, tf2 = F.poses(n, 0, 1.2, 0, n)
    tf2[::7, :9] *= 1.3
    _same(local, qm, tf1, tf2, 1, True)
    _same(local, qm, tf1, tf2, 5, True)
    local.close()


def test_single_calls_with_many_contacts():
    """More records than a call's pinned room: through device memory, the
    page-locked memory stays as it is, and small answers follow large ones."""
    print("case: single calls with many contacts", flush=True)
    local = F.Context(0)
    A, B = F.icosphere(32, 0.05, 9), F.icosphere(32, 0.05, 10)
    m = [local.mesh(*A), local.mesh(*B)]
    I = np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0], float)
    near, far = I.copy(), I.copy()
    near[9:], far[9:] = [0.02, 0.01, 0.03], [1.8, 0.3, 0.1]
    rc, counts, per_q, bv, leaf, _ = collide_gpu(local, np.array([m], np.int32), I[None],
                                                 near[None], 10**6, capacity=1 << 20)
    full = per_q[0]
    assert rc == 0 and len(full) == counts[0] > 3 * 4096
    held = None
    for cap in (4095, 4096, 4097, 10**6, 100, 10**6):
        pairs, stats = local.collide(m[0], I, m[1], near, cap=cap)
        assert np.array_equal(pairs, full[:cap])
        few = local.collide(m[0], I, m[1], far, cap=cap)[0]
        assert len(few) < 1000
        if cap > len(full):
            assert stats.tolist() == [bv[0], leaf[0]]
        held = held or local.get_engine_param("single_pinned_bytes")
    assert local.get_engine_param("single_pinned_bytes") == held < 4096 * 12 + 1024
    # the geometry of a small answer (pinned) begins that of a large one
    small = local.collide_contact(m[0], I, m[1], near, cap=3000)
    large = local.collide_contact(m[0], I, m[1], near, cap=10**6)
    again = local.collide_contact(m[0], I, m[1], near, cap=10**6)
    assert len(small[0]) == 3000 and len(large[0]) > 4096
    for a, b, c in zip(small[:4], large[:4], again[:4]):
        assert np.array_equal(a, b[:3000]) and np.array_equal(b, c)
    assert local.get_engine_param("single_pinned_bytes") < 4096 * 68 + 1024
    local.close()
