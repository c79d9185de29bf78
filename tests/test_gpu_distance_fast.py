"""FAST distance batches where the FP32 intervals leave least to go by (ties,
touching and flat meshes, far poses), where rounding decides which of several
pairs at one distance is first, and at the edges of how queries are dealt to
wavefronts: bit for bit the PLAIN engine's answers with either kind of bound."""
import numpy as np
import pytest
import torch

import fcl_amd as F
from test_gpu_clearance import _batch

pytestmark = pytest.mark.gpu


def _same(ctx, m, tf1, tf2, label):
    print("case: fast distance %s n=%d" % (label, len(tf1)), flush=True)
    want = _batch(ctx, m, tf1, tf2, F.ENGINE_PLAIN)
    for cull in (1, 0):
        ctx.set_engine_param("dist_fp32_cull", cull)
        try:
            got = _batch(ctx, m, tf1, tf2, F.ENGINE_FAST)
        finally:
            ctx.set_engine_param("dist_fp32_cull", 1)
        for k in range(3):
            assert np.array_equal(got[k], want[k]), (cull, k)


@pytest.mark.parametrize("n", [1, 2, 31, 33, 2049, 4097, 20000])
def test_batch_sizes(ctx, n):
    m = [ctx.mesh(*F.icosphere(5, 0.15, 51), F.RSS), ctx.mesh(*F.icosphere(4, 0.15, 52), F.RSS)]
    tf1, tf2 = F.poses(n, 1, 1.2, 3.5, n)
    _same(ctx, m, tf1, tf2, "sizes")


@pytest.mark.parametrize("scale", [1.0, 1e-3, 1e4])
@pytest.mark.parametrize("ka,kb", [(0, 0), (0, 7), (9, 9)])
def test_scales_and_small_meshes(ctx, ka, kb, scale):
    tri = (np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.2]], float), np.array([[0, 1, 2]], np.int32))
    A, B = [tri if k == 0 else F.icosphere(k, 0.15, 60 + k) for k in (ka, kb)]
    m = [ctx.mesh(A[0] * scale, A[1], F.RSS), ctx.mesh(B[0] * scale, B[1], F.RSS)]
    # (at 1e-3 the reference's own bounds are off by the absolute 1e-7 of its
    # edge tests: which touching pair is first is then the visit order's)
    tf1, tf2 = F.poses(200, 1, 0.5 if scale >= 1 else 2.1, 3.5, 77)
    tf2[::5, 9:] += 50.0  # far apart as well
    tf1[:, 9:] *= scale
    tf2[:, 9:] *= scale
    _same(ctx, m, tf1, tf2, "scale %g" % scale)


def test_flat_meshes(ctx):
    """Two noisy grids nearly face to face: many bounds within an interval."""
    m = [ctx.mesh(*F.heightfield(33, 0.01, s), F.RSS) for s in (3, 4)]
    rng = np.random.default_rng(5)
    tf1 = np.tile(np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0], float), (64, 1))
    tf2 = tf1.copy()
    tf2[:, 9:] = rng.uniform([-0.2, -0.2, 0.0], [0.2, 0.2, 0.3], (64, 3))
    _same(ctx, m, tf1, tf2, "flat")


def test_ties(ctx):
    """Two flat grids face to face: whole rows of triangle pairs at one distance."""
    V, T = F.heightfield(9, 0.0, 1)
    m = [ctx.mesh(V, T, F.RSS), ctx.mesh(V, T, F.RSS)]
    tf1 = np.tile(np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0, 0, 0], float), (5, 1))
    tf2 = tf1.copy()
    tf2[:, 11] = [0.5, 0.25, 1.0, 2.0, 0.0]
    _same(ctx, m, tf1, tf2, "ties")
