"""Mesh against primitives by whole wavefronts, at the edges of its list and
of its cull: every kind, caps from one to all contacts, uneven trees and poses
that are no rotations, against the oracle; and its other forms -- a lane per
query, stacks in device memory, EPA in the descending lane."""
import numpy as np
import pytest
import torch

import fcl_amd as F
import fclo

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _run(ctx, mesh, rec, pool, qs, tf1, tf2, cap):
    n = len(qs)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a)).to(DEV, d)  # noqa: E731
    counts = torch.zeros(n, dtype=torch.int32, device=DEV)
    prims = torch.full((n * cap,), -1, dtype=torch.int32, device=DEV)
    stats = torch.zeros((n, 2), dtype=torch.int64, device=DEV)
    geo = (torch.zeros((n * cap, 3), dtype=torch.float64, device=DEV),
           torch.zeros((n * cap, 3), dtype=torch.float64, device=DEV),
           torch.zeros(n * cap, dtype=torch.float64, device=DEV))
    s = torch.cuda.current_stream().cuda_stream
    ctx.mesh_shape_collide_batch_async(
        torch.full((n,), mesh, dtype=torch.int32, device=DEV),
        t(np.ascontiguousarray(rec).view(np.uint8), torch.uint8), t(pool, torch.float64),
        t(qs, torch.int32), t(tf1, torch.float64), t(tf2, torch.float64), cap, counts,
        primitives=prims, contact=geo, stats=stats, stream=s)
    ctx.sync(s)
    return (counts.cpu().numpy(), prims.cpu().numpy().reshape(n, cap),
            [g.cpu().numpy().reshape(n, cap, -1) for g in geo], stats.cpu().numpy())


def _fan(n):
    """Triangles that grow by a third each along x: an uneven tree."""
    V, T = [], []
    for i in range(n):
        x = 1.35 ** i * 1e-3
        V += [[x, 0, 0], [x * 1.2, 0.2 * x, 0], [x, 0.1 * x, 0.3 * x]]
        T.append([3 * i, 3 * i + 1, 3 * i + 2])
    return np.array(V), np.array(T, np.int32)


SHAPES = ([F.BOX, F.SPHERE, F.CAPSULE, F.CYLINDER, F.CONVEX],
          [(0.6, 0.4, 0.5), (0.4, 0, 0), (0.2, 0.6, 0), (0.3, 0.5, 0), (0, 0, 0)])


def _check(ctx, V, T, n, cap, shell, scale=1.0):
    rng = np.random.default_rng(n + cap)
    rec, pool = F.shape_table(*SHAPES, [0.4 * rng.standard_normal((9, 3))])
    qs = (np.arange(n) % 5).astype(np.int32)
    tf1, tf2 = F.poses(n, 1, shell[0], shell[1], 0xF0 + n)
    tf1[:, :9] *= scale
    mesh = ctx.mesh(V, T)
    try:
        counts, prims, geo, stats = _run(ctx, mesh, rec, pool, qs, tf1, tf2, cap)
    finally:
        ctx.mesh_destroy(mesh)
    oc, op, og, ost = fclo.mesh_shape_collide_batch([fclo.OracleMesh(V, T)],
                                                    np.zeros(n, np.int32), rec, pool, qs, tf1,
                                                    tf2, cap=cap, enable_contact=True)
    assert np.array_equal(counts, oc) and np.array_equal(stats, ost)
    for q in range(n):
        k = oc[q]
        assert np.array_equal(prims[q, :k], op[q, :k])
        # normals, positions, depths
        assert np.array_equal(np.concatenate([geo[1][q, :k], geo[0][q, :k], geo[2][q, :k]], 1),
                              og[q, :k])
    return oc


@pytest.mark.parametrize("n,cap", [(1, 1), (65, 1), (200, 3), (60, 500)])
def test_all_kinds_and_caps(ctx, n, cap):
    print("case: mesh-shape wavefronts n=%d cap=%d" % (n, cap), flush=True)
    V, T = F.icosphere(9, 0.15, 77)
    oc = _check(ctx, V, T, n, cap, (0.5, 1.6))
    assert n == 1 or (oc > 0).any() and (oc < cap).any()


def test_poses_that_are_no_rotations(ctx):
    print("case: mesh-shape wavefronts, scaled poses", flush=True)
    V, T = F.icosphere(6, 0.15, 78)
    _check(ctx, V, T, 50, 2, (0.5, 2.0), scale=1.4)


@pytest.mark.parametrize("n,levels", [(40, 10), (200, 24)])
def test_long_trees(ctx, n, levels):
    """Trees about twice as deep as even ones."""
    V, T = _fan(n)
    V /= np.abs(V).max()
    assert F.bvh_build(V, T)["depth"] == levels
    print("case: mesh-shape wavefronts, fan of %d" % n, flush=True)
    _check(ctx, V, T, 40, 4, (0.0, 1.2))


FORMS = [{"ordered_lanes": 2}, {"meshshape_list_depth": 0}, {"meshshape_epa_queue": 0}]


@pytest.mark.parametrize("params", FORMS)
@pytest.mark.parametrize("n,cap", [(1, 1), (257, 1), (700, 6), (60, 500)])
def test_other_forms(params, n, cap):
    """A lane per query with its hits queued for EPA; stacks in device memory,
    and EPA in the descending lane."""
    print("case: mesh-shape %s n=%d cap=%d" % (params, n, cap), flush=True)
    local = F.Context(0)
    for k, v in params.items():
        local.set_engine_param(k, v)
    V, T = F.icosphere(9, 0.15, 77)
    oc = _check(local, V, T, n, cap, (0.5, 1.6))
    assert n == 1 or (oc > 0).any() and (oc < cap).any()
    _check(local, V, T, n, cap, (0.5, 2.0), scale=1.4)
    local.close()


@pytest.mark.parametrize("params", FORMS[:2])
def test_other_forms_without_geometry(params):
    local = F.Context(0)
    for k, v in params.items():
        local.set_engine_param(k, v)
    V, T = F.icosphere(7, 0.15, 79)
    rng = np.random.default_rng(4)
    rec, pool = F.shape_table(*SHAPES, [0.4 * rng.standard_normal((9, 3))])
    n = 5000
    print("case: mesh-shape booleans %s" % params, flush=True)
    qs = (np.arange(n) % 5).astype(np.int32)
    tf1, tf2 = F.poses(n, 1, 0.5, 1.8, 0xF3)
    m = local.mesh(V, T)
    counts = torch.zeros(n, dtype=torch.int32, device=DEV)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a)).to(DEV, d)  # noqa: E731
    s = torch.cuda.current_stream().cuda_stream
    local.mesh_shape_collide_batch_async(
        torch.full((n,), m, dtype=torch.int32, device=DEV),
        t(np.ascontiguousarray(rec).view(np.uint8), torch.uint8), t(pool, torch.float64),
        t(qs, torch.int32), t(tf1, torch.float64), t(tf2, torch.float64), 3, counts, stream=s)
    local.sync(s)
    oc = fclo.mesh_shape_collide_batch([fclo.OracleMesh(V, T)], np.zeros(n, np.int32), rec, pool,
                                       qs, tf1, tf2, cap=3)[0]
    assert np.array_equal(counts.cpu().numpy(), oc) and 0 < (oc > 0).mean() < 1
    local.close()


@pytest.mark.parametrize("cap", [1, 4])
@pytest.mark.parametrize("n", [4000, 262144 + 77])
def test_light_and_heavy_meshes_in_one_batch(n, cap):
    """By the rule, with bad ids among them, against wavefronts alone."""
    print("case: mesh-shape light and heavy n=%d cap=%d" % (n, cap), flush=True)
    local = F.Context(0)
    tri = np.array([[0.9, 0, 0], [-0.4, 0.8, 0], [-0.4, -0.8, 0.1]]), np.array([[0, 1, 2]])
    m = np.array([local.mesh(*x) for x in (tri, F.icosphere(2, 0.15, 5), F.icosphere(12, 0.1, 6))],
                 np.int32)
    rng = np.random.default_rng(n)
    rec, pool = F.shape_table(*SHAPES, [0.4 * rng.standard_normal((9, 3))])
    qm, qs = m[rng.integers(0, 3, n)], rng.integers(0, 5, n).astype(np.int32)
    qm[3::997], qs[7::997] = 55, -1
    bad = (qm == 55) | (qs < 0)
    tf1, tf2 = F.poses(n, 1, 0.5, 1.6, 0xF5)
    t = lambda a, d: torch.from_numpy(np.ascontiguousarray(a)).to(DEV, d)  # noqa: E731
    args = [t(qm, torch.int32), t(np.ascontiguousarray(rec).view(np.uint8), torch.uint8),
            t(pool, torch.float64), t(qs, torch.int32), t(tf1, torch.float64),
            t(tf2, torch.float64)]
    s = torch.cuda.current_stream().cuda_stream
    out = []
    for mode in (1, 0):
        local.set_engine_param("ordered_lanes", mode)
        counts = torch.full((n,), -1, dtype=torch.int32, device=DEV)
        prims = torch.full((n * cap,), -1, dtype=torch.int32, device=DEV)
        geo = tuple(torch.zeros((n * cap,) + k, dtype=torch.float64, device=DEV)
                    for k in ((3,), (3,), ()))
        stats = torch.full((n, 2), -1, dtype=torch.int64, device=DEV)
        local.mesh_shape_collide_batch_async(*args, cap, counts, primitives=prims, contact=geo,
                                             stats=stats, stream=s)
        assert local.sync_status(s) == F.N.FCLX_ERR_INVALID_ARGUMENT
        out.append([counts, prims, stats] + list(geo))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    counts = out[0][0].cpu().numpy()
    assert not counts[bad].any() and 0 < (counts > 0).mean() < 1
    local.close()
