"""The lane-group traversal (device/ordered.h) restated step by step: whatever
a group tests ahead of its turn, the contacts, their order and the test counts
are those of the depth-first recursion, and the list stays inside its bound.

The tree is synthetic: every node pair is disjoint, internal or a leaf by a
seeded hash, leaves hit with 0 to 2 contacts (contact geometry) or one.
"""
import random

import pytest

NODE, LEAF, HIT = 0, 1, 2


class Tree:
    def __init__(self, seed, depth, p_overlap, p_hit, contact):
        self.seed, self.depth, self.contact = seed, depth, contact
        self.p_overlap, self.p_hit = p_overlap, p_hit

    def _r(self, node, salt):
        return random.Random("%d/%s/%s" % (self.seed, node, salt)).random()

    def test(self, node):
        """'no', 'leaf' or the two children of an overlapping pair."""
        if self._r(node, "o") >= self.p_overlap and node != "":
            return "no"
        if len(node) >= self.depth or (len(node) > 2 and self._r(node, "l") < 0.15):
            return "leaf"
        return node + "0", node + "1"

    def hit(self, node):
        """None, or the pair's number of contacts."""
        if self._r(node, "h") >= self.p_hit:
            return None
        return int(3 * self._r(node, "n")) if self.contact else 1


def recursion(tree, cap):
    out, bv, leaf, stack = [], 0, 0, [""]
    while stack and not (out and len(out) >= cap):
        node = stack.pop()
        bv += 1
        t = tree.test(node)
        if t == "leaf":
            leaf += 1
            n = tree.hit(node)
            if n is not None:
                out += [(node, i) for i in range(min(n, cap - len(out)))]
        elif t != "no":
            stack += [t[1], t[0]]
    return out, bv, leaf


class Group:
    """One group's query: the list (top last), totals, the records emitted."""

    def __init__(self, tree, cap, G, list_cap, margin, mistake=None, carry_max=2**31):
        self.carry_max, self.most, self.serial = carry_max, 0, 0
        self.audit_in = carry_max // 128
        self.tree, self.cap, self.G = tree, cap, G
        self.list_cap, self.margin, self.mistake = list_cap, margin, mistake
        self.e, self.acc = [(NODE, "")], [[0, 0]]
        self.count = self.bv = self.leaf = 0
        self.tail = [0, 0]
        self.out, self.steps, self.high, self.ahead = [], 0, 1, 0

    def window(self):
        room = self.list_cap - self.margin - len(self.e)
        n = min(len(self.e), self.G)
        return n if n <= room else max(room, 1)

    def audit(self):
        self.bv += self.acc[-1][0]
        self.leaf += self.acc[-1][1]
        self.acc[-1] = [0, 0]
        many = sum(a[0] for a in self.acc) >= self.carry_max // 2
        self.audit_in = 0 if many else self.carry_max // 128
        self.serial += many
        return many

    def step(self, test_leaves):
        n = self.window()
        self.audit_in -= 1
        if self.audit_in < 0 and self.audit():
            n = 1
        lanes = [(self.e[-1 - k], self.acc[-1 - k]) for k in range(n)]
        base = len(self.e) - n
        nodes = sum(e[0] == NODE for e, _ in lanes)
        if any(e[0] == LEAF for e, _ in lanes) and nodes == 0:
            test_leaves = True
        outs, hits, tests = [], [None] * n, []
        for k, (e, _) in enumerate(lanes):
            o, t = [], (0, 0)
            if e[0] >= HIT:
                o, hits[k] = [e], e[0] - HIT
            elif e[0] == NODE:
                t, r = (1, 0), self.tree.test(e[1])
                o = [] if r == "no" else [(LEAF, e[1])] if r == "leaf" else [(NODE, c) for c in r]
            elif test_leaves:
                t, m = (0, 1), self.tree.hit(e[1])
                if m is not None:
                    o, hits[k] = [(HIT + m, e[1])], m
            else:
                o = [e]
            outs.append(o)
            tests.append(t)
        # ord_settle
        last, committed = n - 1, -1
        if any(h is not None for h in hits):
            before, reach = [], -1
            for k in range(n):
                before.append(sum(h for h in hits[:k] if h))
                if reach < 0 and hits[k] and hits[k] >= self.cap - self.count - before[k]:
                    reach = k
            if reach >= 0:
                last, base = reach, 0
                self.tail = [0, 0]
                outs = [o if k <= last else [] for k, o in enumerate(outs)]
            opened = [k for k in range(n) if outs[k] and hits[k] is None]
            lead = opened[0] if opened else n
            mine = [k for k in range(n) if hits[k] is not None and k < lead and k <= last]
            total = 0
            for k in mine:
                take = min(hits[k], self.cap - self.count - before[k])
                self.out += [(lanes[k][0][1], i) for i in range(take)]
                total = before[k] + take
                committed = k
                outs[k] = []
            self.count += total
        pre, s = [], [0, 0]
        for k in range(n):
            if k <= last:
                s = [s[j] + lanes[k][1][j] + tests[k][j] for j in (0, 1)]
            pre.append(s)
        at = lambda k: pre[k] if k >= 0 else [0, 0]  # noqa: E731
        self.e = self.e[:base]
        new_e, new_acc, prev = [], [], -1
        for k in range(n):
            if not outs[k]:
                continue
            frm = max(prev, committed)
            new_e += outs[k]
            new_acc.append([pre[k][j] - at(frm)[j] for j in (0, 1)])
            new_acc += [[0, 0]] * (len(outs[k]) - 1)
            prev = k
        end = max(prev, committed)
        rest = [pre[n - 1][j] - at(end)[j] for j in (0, 1)]
        if committed >= 0:
            self.bv += pre[committed][0]
            self.leaf += pre[committed][1]
        below = self.acc[:base]
        if base > 0:
            below[-1] = [below[-1][j] + rest[j] for j in (0, 1)]
        elif self.mistake == "tail":  # the tests behind the list's end counted at once
            self.bv += rest[0]
            self.leaf += rest[1]
        else:
            self.tail = [self.tail[j] + rest[j] for j in (0, 1)]
        self.e += new_e[::-1]
        self.acc = below + new_acc[::-1]
        self.most = max([self.most] + [x for a in self.acc for x in a])
        self.high = max(self.high, len(self.e))
        self.steps += 1
        if not self.e or self.count >= self.cap:
            if self.count < self.cap:
                self.bv += self.tail[0]
                self.leaf += self.tail[1]
            return False
        return True

    def run(self, rng):
        while self.step(rng.random() < 0.4):
            assert self.high <= self.list_cap and self.steps < 100000
        return self.out, self.bv, self.leaf


CASES = [(16, 192), (64, 512), (4, 24), (8, 28)]  # the last two: the bound in force


@pytest.mark.parametrize("G,list_cap", CASES)
@pytest.mark.parametrize("contact", [False, True])
def test_group_traversal_is_the_recursion(G, list_cap, contact):
    rng = random.Random(G)
    narrow = ended = 0
    for seed in range(60):
        depth = rng.randint(3, 14)
        tree = Tree(seed, depth, rng.choice([0.55, 0.7, 0.85]), rng.choice([0.0, 0.05, 0.4]),
                    contact)
        for cap in (1, 2, 7, 10**6):
            want = recursion(tree, cap)
            g = Group(tree, cap, G, list_cap, depth + 3)
            assert g.run(rng) == want
            narrow += g.high > list_cap - depth - 3
            ended += len(want[0]) == cap
    assert ended > 20 and (narrow > 0 or list_cap > 100)


@pytest.mark.parametrize("carry_max", [1, 40, 300])
def test_no_entry_carries_more_than_its_bits(carry_max):
    """A list near its carry limit goes one node at a time: same answers and
    counts, and no entry carries more than the limit and one step's tests."""
    rng = random.Random(carry_max)
    G, free, held = 64, 0, 0
    for seed in range(25):
        tree = Tree(seed, rng.randint(6, 13), 0.85, rng.choice([0.0, 0.05]), False)
        for cap in (1, 7, 10**6):
            want = recursion(tree, cap)
            g = Group(tree, cap, G, 512, 16, carry_max=carry_max)
            assert g.run(rng) == want and g.most <= carry_max + G
            u = Group(tree, cap, G, 512, 16)
            assert u.run(rng) == want
            free, held = max(free, u.most), held + (g.serial > 0)
    assert free > carry_max + G and held > 5


def test_a_planted_mistake_is_seen():
    rng = random.Random(3)
    wrong = 0
    for seed in range(40):
        tree = Tree(seed, 10, 0.7, 0.1, False)
        wrong += Group(tree, 1, 16, 192, 13, mistake="tail").run(rng) != recursion(tree, 1)
    assert wrong > 0
