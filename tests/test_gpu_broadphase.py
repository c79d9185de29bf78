"""Broadphase pairs on both sides of the tile limit against a numpy restatement:
edges of tiles, dense overlaps, groups, capacities, and odd boxes (inverted,
infinite, NaN), for which the sort-and-sweep's own rule is restated."""
import numpy as np
import pytest
import torch

import fcl_amd as F

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
TILES = 16384


def _boxes(n, seed, size):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (n, 3)) * n ** (1 / 3)
    h = rng.uniform(0.2, 1.0, (n, 3)) * size
    return np.concatenate([c - h, c + h], 1)


def _run(ctx, boxes, cap, groups=None):
    n = len(boxes)
    pairs = torch.full((max(cap, 1), 2), 7, dtype=torch.int32, device=DEV)[:cap]
    num = torch.full((1,), 99, dtype=torch.int64, device=DEV)
    g = None if groups is None else torch.from_numpy(groups.astype(np.int32)).to(DEV)
    s = torch.cuda.current_stream().cuda_stream
    ctx.broadphase_pairs_async(torch.from_numpy(boxes).to(DEV).contiguous(), pairs, num, groups=g,
                               stream=s)
    ctx.sync(s)
    return pairs.cpu().numpy(), int(num.item())


def _overlap(a, b):
    """Not separated on any axis (an unordered bound separates nothing)."""
    with np.errstate(invalid="ignore"):
        return ~((a[:3] > b[..., 3:]) | (b[..., :3] > a[3:])).any(-1)


def _want(boxes, groups=None):
    out = []
    for i in range(len(boxes)):
        hit = _overlap(boxes[i], boxes[i + 1:])
        if groups is not None:
            hit &= groups[i + 1:] != groups[i]
        out += [(i, i + 1 + int(k)) for k in np.flatnonzero(hit)]
    return np.array(out, np.int32).reshape(-1, 2)


@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 1000, 1025])
@pytest.mark.parametrize("grouped", [False, True])
def test_tiles(ctx, n, grouped):
    print("case: broadphase n=%d groups=%d" % (n, grouped), flush=True)
    boxes = _boxes(n, n, 0.8)
    groups = np.arange(n) % 3 if grouped else None
    want = _want(boxes, groups)
    cap = len(want) + 5
    pairs, num = _run(ctx, boxes, cap, groups)
    assert num == len(want) and np.array_equal(pairs[:num], want)
    assert (pairs[num:] == -1).all()
    small, num = _run(ctx, boxes, len(want) // 2, groups)
    assert num == len(want)
    assert set(map(tuple, small.tolist())) <= set(map(tuple, want.tolist()))
    assert _run(ctx, boxes, 0, groups)[1] == len(want)


def test_one_object_and_a_dense_scene(ctx):
    print("case: broadphase dense", flush=True)
    assert _run(ctx, _boxes(1, 1, 1.0), 4)[1] == 0
    boxes = _boxes(300, 2, 30.0)
    want = _want(boxes)
    pairs, num = _run(ctx, boxes, len(want))
    assert num == len(want) > 40000 and np.array_equal(pairs, want)


@pytest.mark.parametrize("grouped", [False, True])
def test_sweep_equals_tiles(ctx, grouped):
    """The same objects with far ones added, so that the batch is on the other
    side of the limit."""
    n = 6000
    print("case: broadphase sweep groups=%d" % grouped, flush=True)
    boxes = _boxes(n, 3, 0.7)
    boxes[17, :3], boxes[17, 3:] = -100, 100  # a box that meets them all
    groups = (np.arange(n) % 2).astype(np.int32) if grouped else None
    few, num = _run(ctx, boxes, 40000, groups)
    far = np.arange(TILES + 1 - n)[:, None] * 3.0 + 1000
    many = np.concatenate([boxes, np.repeat(np.concatenate([far, far + 1], 1), 3, 1)])
    g2 = None if groups is None else np.concatenate([groups, np.zeros(len(far), np.int32)])
    got, num2 = _run(ctx, many, 40000, g2)
    assert len(many) > TILES and num == num2 > n // 2
    assert np.array_equal(few, got)


def _swept(boxes):
    """Sort and sweep restated: bits in ascending order, ties by index."""
    u = boxes[:, 0].copy().view(np.uint64)
    key = np.where(u >> np.uint64(63) != 0, ~u, u | (np.uint64(1) << np.uint64(63)))
    order = np.lexsort((np.arange(len(boxes)), key))
    out = []
    for k, i in enumerate(order):
        for j in order[k + 1:]:
            if boxes[j, 0] > boxes[i, 3]:
                break
            if _overlap(boxes[i], boxes[j]):
                out.append((min(i, j), max(i, j)))
    return np.array(sorted(out), np.int32).reshape(-1, 2)


@pytest.mark.parametrize("seed", range(4))
def test_odd_boxes(ctx, seed):
    print("case: broadphase odd boxes %d" % seed, flush=True)
    rng = np.random.default_rng(seed)
    boxes = _boxes(150, 10 + seed, 0.8)
    for value in (np.nan, -np.nan, np.inf, -np.inf, 0.0, -0.0):
        at = rng.integers(0, 150, 6), rng.integers(0, 6, 6)
        boxes[at] = value
    flip = rng.integers(0, 150, 5)
    boxes[flip, 0], boxes[flip, 3] = boxes[flip, 3], boxes[flip, 0].copy()
    want = _swept(boxes)
    pairs, num = _run(ctx, boxes, len(want))
    assert num == len(want) and np.array_equal(pairs, want)


@pytest.mark.parametrize("n", [64, 65, 700])
def test_unordered_lower_bounds_of_both_signs(ctx, n):
    """Negative NaN sorts first and positive NaN last: a walk from the one
    reaches the other unless an ordered lower x ends it.  Inverted boxes, some
    of them at the largest lower x."""
    print("case: broadphase NaN of both signs, n=%d" % n, flush=True)
    rng = np.random.default_rng(n)
    boxes = _boxes(n, n, 2.0)
    boxes[:, 1:3], boxes[:, 4:] = -1, 1  # the x axis decides
    sign = rng.integers(0, 4, n)
    boxes[sign == 0, 0] = np.nan
    boxes[sign == 1, 0] = -np.nan
    boxes[sign == 3, 3] = rng.choice([np.inf, np.nan, 0.0, -3.0], (sign == 3).sum())
    boxes[sign == 2, 0] = np.where(rng.random((sign == 2).sum()) < 0.2, 9.0, boxes[sign == 2, 0])
    want = _swept(boxes)
    pairs, num = _run(ctx, boxes, len(want) + 3)
    assert num == len(want) and np.array_equal(pairs[:num], want)
    assert len(want) < len(_want(boxes))  # some walks end early
