"""The wavefront form of distance() (kernels_clearance.hip) restated step by
step: distance, pair and test counts are those of the recursion, with bounds
that need not be lower bounds (as merged BVs have them), ties and NaN, and the
list stays inside its bound."""
import math
import random

import pytest

NODE, LEAF, MARK, DONE = 0, 1, 2, 3


class Tree:
    """A synthetic BVTT: bounds and leaf distances by a seeded hash, on a
    coarse grid so that ties are common."""

    def __init__(self, seed, depth, loose, nan):
        self.seed, self.depth, self.loose, self.nan = seed, depth, loose, nan

    def _r(self, node, salt):
        return random.Random("%d/%s/%s" % (self.seed, node, salt)).random()

    def is_leaf(self, node):
        return len(node) >= self.depth or (len(node) > 1 and self._r(node, "l") < 0.1)

    def _low(self, node):
        low = sum(int(c) * (0.5 + self._r(node[:k], "w")) for k, c in enumerate(node))
        return round(8 * (low * 0.5 + self.loose * self._r(node, "b"))) / 8

    def bound(self, node):
        return math.nan if self.nan and self._r(node, "x") < 0.02 else self._low(node)

    def dist(self, node):
        if self.nan and self._r(node, "y") < 0.02:
            return math.nan
        return self._low(node) + round(24 * self._r(node, "t")) / 8


def recursion(tree, seed_dist):
    best, who, bv, leaf = seed_dist, "seed", 0, 0
    stack, node = [], ""
    while True:
        if tree.is_leaf(node):
            leaf += 1
            t = tree.dist(node)
            if best > t:
                best, who = t, node
            node = None
        else:
            a, b = node + "0", node + "1"
            da, db = tree.bound(a), tree.bound(b)
            bv += 2
            near, far = ((b, db), (a, da)) if db < da else ((a, da), (b, db))
            stack.append(far)
            node = near[0] if not near[1] >= best else None
        while node is None and stack:
            n, d = stack.pop()
            if not d >= best:
                node = n
        if node is None:
            return best, who, bv, leaf


def subtree(tree, node, deep, best):
    """The entries a node expanded `deep` levels leaves below itself."""
    out = []
    ch = [(c, tree.bound(c)) for c in (node + "0", node + "1")]
    for c, d in ch[::-1] if ch[1][1] < ch[0][1] else ch:
        if d >= best:
            continue
        if tree.is_leaf(c):
            out.append((LEAF, c, d, None))
        elif deep == 1:
            out.append((NODE, c, d, None))
        else:
            out += [(MARK, c, d, None)] + subtree(tree, c, deep - 1, best)
    return out


def wavefront(tree, best, wave, cap, margin, mistake=None):
    levels = wave.bit_length() - 2
    who, bv, leaf, drop, steps, high = "seed", 0, 0, -1, 0, 1
    root = LEAF if tree.is_leaf("") else NODE
    lst = [(root, "", -math.inf, None)]  # kind, node, bound, distance; top last

    def first(p):
        return next((k for k in range(n) if p(k)), wave)

    while lst:
        steps, old = steps + 1, best
        assert steps < 20000
        n = min(len(lst), wave)
        ent = [list(lst[-1 - k]) for k in range(n)]
        keep = [True] * n
        lev = [len(e[1]) for e in ent]
        if drop >= 0:
            end = first(lambda k: lev[k] <= drop)
            keep = [k >= end for k in range(n)]
            if end < n:
                drop = -1
        over = [e[2] >= best for e in ent]
        keep = [keep[k] and not (over[k] and ent[k][0] != MARK) for k in range(n)]
        top = first(lambda k: keep[k])
        if top < wave and ent[top][0] == MARK and over[top]:
            end = first(lambda k: k > top and lev[k] <= lev[top])
            for k in range(top, min(end, n)):
                keep[k] = False
            if end >= n and mistake != "drop":
                drop = lev[top]
        room = cap - margin - len(lst)
        head = first(lambda k: keep[k])
        nodes = [k for k in range(n) if keep[k] and ent[k][0] == NODE]
        deep = max([d for d in range(1, levels + 1) if len(nodes) <= wave >> (d + 1)], default=1)
        while deep > 1 and (len(nodes) << (deep + 1)) > room:
            deep -= 1
        most = min(room // (2 << deep), wave // (2 << deep))
        expand = [False] * n
        for r, k in enumerate(nodes):
            expand[k] = r < most if most > 0 else k == head
        leaves = [k for k in range(n) if keep[k] and ent[k][0] == LEAF]
        if leaves and (not any(expand) or len(leaves) >= wave // 4 or head in leaves):
            for k in leaves:
                ent[k][0], ent[k][3] = DONE, tree.dist(ent[k][1])
        settled = [keep[k] and ent[k][0] in (MARK, DONE) for k in range(n)]
        stop = first(lambda k: keep[k] and not settled[k])
        low, before, low_who = best, [], who
        lows = []
        for k in range(n):
            before.append(low)
            if settled[k] and k < stop and ent[k][0] == DONE and ent[k][3] < low:
                low = ent[k][3]
            lows.append(low)
        bad = first(lambda k: settled[k] and k < stop and ent[k][2] >= before[k])
        end = min(bad, stop)
        turn = [settled[k] and k < end for k in range(n)]
        bv += 2 * sum(turn[k] and ent[k][0] == MARK for k in range(n))
        done = [k for k in range(n) if turn[k] and ent[k][0] == DONE]
        leaf += len(done)
        if done:
            now = lows[min(end, n) - 1]
            if now < best:
                low_who = next(k for k in done if ent[k][3] == now)
                best, who = now, ent[low_who][1]
        lst = lst[:len(lst) - n]
        out = []
        for k in range(n):
            if not keep[k] or turn[k]:
                continue
            kind, node, d, t = ent[k]
            if not expand[k]:
                out.append((kind, node, d, t))
                continue
            if k == end and not d >= best:
                bv += 2
            else:
                out.append((MARK, node, d, None))
            out += subtree(tree, node, deep, old)
        lst += out[::-1]
        high = max(high, len(lst))
        assert high <= cap
    return (best, who, bv, leaf), high


@pytest.mark.parametrize("wave,cap", [(64, 512), (16, 27), (4, 20)])
@pytest.mark.parametrize("nan", [False, True])
def test_wavefront_is_the_recursion(wave, cap, nan):
    tight = 0
    for seed in range(150):
        rng = random.Random(seed)
        depth = rng.randint(0, 12)
        tree = Tree(seed, depth, rng.choice([0.0, 0.5, 4.0]), nan)
        start = rng.choice([0.0, 1.5, 6.0, math.inf])
        got, high = wavefront(tree, start, wave, cap, depth + 2)
        assert repr(got) == repr(recursion(tree, start))
        tight += high > cap - depth - 2
    assert tight > 0 or cap > 100, "the bound was never in force"


def test_a_planted_mistake_is_seen():
    wrong = 0
    for seed in range(200):
        tree = Tree(seed, 12, 4.0, False)
        wrong += wavefront(tree, 20.0, 16, 60, 14, "drop")[0] != recursion(tree, 20.0)
    assert wrong > 0
