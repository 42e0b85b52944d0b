"""The records that the kernels walk closest hits with (RB_LAYOUT_MI355X_WALK),
checked on the CPU, in exact arithmetic, against the binary records they stand for:
* a record's children are binary ones of its subtree, every leaf with triangles
  appears once, links go to later records, in turn;
* the origin is the children's smallest corner, a plane with step 0 lies at it, and
  every other plane outside its child's box by 2^-20 of the children's extent -- what
  makes a ray pass the box whenever it passes the binary one;
* a slot without a child links the zero triangle behind a box no ray passes;
* the stack entries that a ray can need are three per level, below the kernels' 96;
* behind the records, each reference's box holds its leaf's; the triangles are the
  binary walk's with their ids."""
from fractions import Fraction

import numpy as np
import pytest

from conftest import random_triangles


def _grid(k):
    """A flat square of k x k quads and one upright triangle."""
    g = np.linspace(-3, 3, k + 1, dtype=np.float32)
    a, b = np.meshgrid(g, g, indexing="ij")
    v = np.stack([a, b, np.zeros_like(a)], -1).reshape(-1, 3)
    i, j = (x.ravel() for x in np.meshgrid(np.arange(k), np.arange(k), indexing="ij"))
    q = i * (k + 1) + j
    idx = np.concatenate([np.stack([q, q + k + 1, q + k + 2], -1), np.stack([q, q + k + 2, q + 1], -1)])
    v = np.concatenate([v, np.array([[0, 0, 1], [1, 0, 1], [0, 0, 2]], np.float32)])
    return v, np.concatenate([idx, [[len(v) - 3, len(v) - 2, len(v) - 1]]]).astype(np.uint32)


def _nested(n, levels, ratio, shift):
    """Clusters of n triangles, each smaller by the ratio: a deep tree."""
    v, idx = random_triangles(n, seed=9, spread=1.0, size=0.3)
    v = np.concatenate([(v + shift) * np.float32(ratio) ** k for k in range(levels)]).astype(np.float32)
    return v, np.arange(len(v), dtype=np.uint32).reshape(-1, 3)


def _scaled(n, seed, scale):
    v, idx = random_triangles(n, seed=seed)
    return (v * np.float32(scale)).astype(np.float32), idx


CASES = {"random": lambda: _scaled(3000, 5, 1.0), "large": lambda: _scaled(1500, 6, 1e4),
         "small": lambda: _scaled(1500, 7, 1e-3), "huge": lambda: _scaled(1000, 8, 1e30),
         "endless": lambda: _scaled(500, 10, 1e32), "flat": lambda: _grid(17), "deep": lambda: _nested(24, 60, 0.5, 2),
         "deeper": lambda: _nested(200, 50, 0.3, 2),
         "one": lambda: _scaled(1, 11, 1.0), "three": lambda: _scaled(3, 12, 1.0)}


def _binary_children(nodes, rec):
    r, f = nodes[rec], nodes[rec].view(np.float32)
    for c in range(2):
        w = [f[4 * c], f[4 * c + 1], f[4 * c + 2], f[4 * c + 3], f[8 + 2 * c], f[9 + 2 * c]]
        # an inverted pair of planes is the box between them
        yield ([min(w[2 * a], w[2 * a + 1]) for a in range(3)], [max(w[2 * a], w[2 * a + 1]) for a in range(3)],
               int(np.int32(r[12 + c])))


def _empty(link):
    return link < 0 and (~link & 31) == 0


def _leaves_of_binary(nodes):
    """The leaves in depth-first order, and each record's range of them."""
    leaves, spans = [], {}

    def walk(rec):
        first = len(leaves)
        for lo, hi, link in _binary_children(nodes, rec):
            if link >= 0:
                walk(link)
            elif not _empty(link):
                leaves.append((link, lo, hi))
        spans[rec] = (first, len(leaves))

    walk(0)
    return leaves, spans


def _depth(nodes, rec=0):
    return max([1 + _depth(nodes, link) for _, _, link in _binary_children(nodes, rec) if link >= 0], default=0)


def test_a_tree_too_deep_keeps_the_binary_walk(rbm):
    from renderbox2_amd import _lib as L
    b = rbm.BVH(_nested(500, 30, 0.2, 0))
    assert _depth(b.export(L.RB_LAYOUT_MI355X)[0].reshape(-1, 16)) >= 62  # 32 levels of three entries
    with pytest.raises(rbm.RbError, match="too deep"):
        b.export(L.RB_LAYOUT_MI355X_WALK)


@pytest.mark.parametrize("case", CASES)
def test_walk_records(rbm, case):
    from renderbox2_amd import _lib as L
    b = rbm.BVH(CASES[case]())
    bn, bt, bx = b.export(L.RB_LAYOUT_MI355X)
    wn, wt, wx = b.export(L.RB_LAYOUT_MI355X_WALK)
    nodes, n_refs = bn.reshape(-1, 16), len(bx)
    assert np.array_equal(wx[:n_refs], bx) and len(wx) == n_refs + 1
    entries = int(wx[n_refs])
    tris = wt.reshape(-1, 16)
    assert len(tris) == n_refs + 1 and not tris[n_refs].any() and not tris[:, 13:].any()
    assert np.array_equal(tris[:n_refs, :12], bt.reshape(-1, 12)[:n_refs]) and np.array_equal(tris[:n_refs, 12], bx)
    n = (len(wn) - 8 * (n_refs + 1)) // 16
    recs, boxes = wn[:16 * n].reshape(-1, 16), wn[16 * n:].view(np.float32).reshape(-1, 8)
    assert n >= 1 and len(boxes) == n_refs + 1

    leaves, spans = _leaves_of_binary(nodes)
    at = {leaf[0]: k for k, leaf in enumerate(leaves)}
    assert len(at) == len(leaves)
    none = ~(n_refs << 5 | 1)
    links = recs[:, 12:16].astype(np.int32)
    # numbering, then each record's range of leaves from the last one up
    order = [int(x) for row in links for x in row if x >= 0]
    assert order == list(range(1, n))
    span, level = [None] * n, [0] * n
    for w in range(n):
        for x in links[w]:
            if x >= 0:
                level[x] = level[w] + 1
    for w in reversed(range(n)):
        ranges = [span[x] if x >= 0 else (at[int(x)], at[int(x)] + 1) for x in links[w] if x != none]
        assert all(p[1] == q[0] for p, q in zip(ranges, ranges[1:]))  # contiguous: none twice, none left out
        span[w] = (ranges[0][0], ranges[-1][1])
    assert span[0] == (0, len(leaves))
    assert entries == 3 * (max(level) + 1) and entries < 96
    if case == "deeper":  # by surface area too many levels: every inner child replaced by its own two
        assert max(level) == _depth(nodes) // 2

    stands_for = [0] * n
    endless = 0
    for w in range(n):
        # the children under the binary record it stands for: leaves as they are, inner ones where a record has their range
        left = [int(x) for x in links[w] if x != none]
        found = []

        def cut(rec):
            for lo, hi, link in _binary_children(nodes, rec):
                if _empty(link):
                    continue
                if link < 0:
                    assert left[len(found)] == link
                    found.append((lo, hi))
                elif len(found) < len(left) and left[len(found)] >= 0 and span[left[len(found)]] == spans[link]:
                    stands_for[left[len(found)]] = link
                    found.append((lo, hi))
                else:
                    cut(link)

        cut(stands_for[w])
        assert len(found) == len(left)
        f = recs[w].view(np.float32)
        for c in range(4):
            if c >= len(left):
                assert links[w][c] == none
        for a in range(3):
            q = [[(int(recs[w][6 + 2 * a + e]) >> (8 * c)) & 0xFF for e in range(2)] for c in range(4)]
            assert all(x == [255, 0] for x in q[len(left):])
            p, s = f[a], f[3 + a]
            assert p == min(lo[a] for lo, _ in found)
            extent = Fraction(float(max(hi[a] for _, hi in found))) - Fraction(float(p))
            if np.isinf(s):  # an axis too long for steps, which the walk leaves out
                assert extent >= Fraction(2) ** 102 and all(x == [0, 0] for x in q[:len(left)])
                endless += 1
                continue
            # (the exporter's own margin is rounded to a double)
            step, margin = Fraction(float(s)) / 2 ** 24, extent / 2 ** 20 * (1 - Fraction(1, 2 ** 30))
            for (lo, hi), (ql, qh) in zip(found, q):
                l, h = Fraction(float(lo[a])) - Fraction(float(p)), Fraction(float(hi[a])) - Fraction(float(p))
                assert ql <= qh
                assert l >= 0 if ql == 0 else ql * step <= l - margin
                assert qh == 0 if h == 0 else qh * step >= h + margin
    assert (endless > 0) == (case in ("huge", "endless"))
    for link, lo, hi in leaves:
        first, count = ~link >> 5, ~link & 31
        for r in range(first, first + count):
            box = boxes[r]
            assert all(box[2 * a] <= lo[a] and box[2 * a + 1] >= hi[a] for a in range(3)) and not box[6:].any()
