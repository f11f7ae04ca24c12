"""The broad phase's lists of node pairs where they can go wrong, against every
pair of boxes tested on the host: trees of one leaf, of one node and just past
it (32 leaves), at and past the start level (2^16 leaves) and a step further
(2^19), of unequal depths; boxes without bounds; and lists that overflow, so
that the tree is walked, and then are long enough."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


def boxes(g, n, size):
    # multiples of 2^-20: exact in single precision, so the raw pairs are these
    lo = g.integers(0, 1 << 20, (n, 3))
    return np.hstack([lo, lo + g.integers(0, size + 1, (n, 3))]) / (1 << 20)


def overlaps(a, b):
    out = []
    for i in range(0, len(a), 64):
        p, q = a[i:i + 64, None], b[None]
        s, c = np.nonzero(((p[..., :3] <= q[..., 3:]) & (p[..., 3:] >= q[..., :3])).all(-1))
        out.append(np.stack([s + i, c], 1))
    return np.concatenate(out)


def same(got, want):
    got = got[np.lexsort((got[:, 1], got[:, 0]))]
    want = want[np.lexsort((want[:, 1], want[:, 0]))]
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("ns,nc", [(1, 1), (1, 33), (31, 32), (32, 33), (33, 65), (257, 8193), (65536, 5), (7, 65537),
                                   (65537, 600), (1, 524289), (300, 600000)])
def test_tree_sizes(ctx, ns, nc):
    g = np.random.default_rng(ns + nc)
    size = (1 << 20) // 3 if ns * nc < 1 << 20 else 1 << 15
    a, b = boxes(g, ns, size), boxes(g, nc, size)
    same(ctx.broad_phase(a, b), overlaps(a, b))


@pytest.mark.parametrize("ns,nc", [(3, 5), (33, 70000)])
def test_boxes_without_bounds(ctx, ns, nc):
    g = np.random.default_rng(ns)
    a, b = boxes(g, ns, 1 << 12), boxes(g, nc, 1 << 12)
    big = np.finfo(np.float32).max
    a[ns // 2] = [-big, -big, -big, big, big, big]
    b[nc // 3, :2], b[nc // 3, 3:5] = -big, big
    same(ctx.broad_phase(a, b), overlaps(a, b))


def test_overflowing_lists(ctx):
    """Crossed rods: most node pairs overlap, few rods do."""
    n = 65536
    g = np.random.default_rng(5)
    y, x = g.integers(0, 1 << 20, n), g.integers(0, 1 << 20, n)
    za, zb = g.integers(0, 1 << 20, n), g.integers(0, 1 << 20, n)
    one = np.full(n, 1 << 20)
    a = np.stack([0 * one, y, za, one, y, za], 1) / (1 << 20)
    b = np.stack([x, 0 * one, zb, x, one, zb], 1) / (1 << 20)
    order = np.argsort(zb, kind="stable")
    lo, hi = np.searchsorted(zb[order], za, "left"), np.searchsorted(zb[order], za, "right")
    want = np.stack([np.repeat(np.arange(n), hi - lo),
                     np.concatenate([order[p:q] for p, q in zip(lo, hi)])], 1)
    for _ in range(2): # walked, then with lists of the length that was needed
        same(ctx.broad_phase(a, b), want)
