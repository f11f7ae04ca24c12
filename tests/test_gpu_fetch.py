"""Results fetched through the pinned stage or past it, and candidate pairs
sorted either way: few pairs, pairs few among the faces, many pairs a face, and
lists of more than the stage's 2^20 bytes; the same results from two threads."""
import threading

import numpy as np
import pytest

import meshes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("ns,nc,side", [(50, 50, 0.05), (3000, 100, 0.03), (400, 400, 0.3), (700, 900, 0.9)])
def test_pairs_in_order(ctx, ns, nc, side):
    g = np.random.default_rng(ns)
    def boxes(n):
        lo = g.integers(0, 1 << 16, (n, 3)) / (1 << 16)
        return np.hstack([lo, lo + side])
    a, b = boxes(ns), boxes(nc)
    s, c = np.nonzero(((a[:, None, :3] <= b[None, :, 3:]) & (a[:, None, 3:] >= b[None, :, :3])).all(-1))
    np.testing.assert_array_equal(ctx.broad_phase(a, b), np.stack([s, c], 1))  # nonzero lists them in order


def test_two_threads(ctx):
    R = ctx.dispatch(*meshes.icosphere_pair(4))
    want = R.registry()
    got, bad = [], []

    def work():
        try:
            for _ in range(20):
                got.append(R.registry())
        except Exception as e:  # noqa: BLE001
            bad.append(e)

    t = [threading.Thread(target=work) for _ in range(2)]
    for x in t:
        x.start()
    for x in t:
        x.join()
    assert not bad and len(got) == 40
    for r in got:
        for x, y in zip(r, want):
            assert np.array_equal(x, y)
