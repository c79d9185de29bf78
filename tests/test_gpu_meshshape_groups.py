"""Mesh against primitives by whole wavefronts, at the edges of its list and
of its cull: every kind, caps from one to all contacts, deep meshes on both
sides of the list's depth, and poses that are no rotations, against the
oracle."""
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
    """A mesh whose tree is as deep as it has triangles: sizes that double."""
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
        assert np.array_equal(np.concatenate([geo[1][q, :k], geo[0][q, :k], geo[2][q, :k]], 1)
                              [:, 6], og[q, :k, 6])
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


@pytest.mark.parametrize("n", [40, 200])
def test_long_trees(ctx, n):
    V, T = _fan(n)
    V /= np.abs(V).max()
    print("case: mesh-shape wavefronts, fan of %d" % n, flush=True)
    _check(ctx, V, T, 40, 4, (0.0, 1.2))
