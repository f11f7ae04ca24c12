"""A dispatch that a fresh context has to run again for many reasons, one hiding
the next: coordinates so far from the origin that the broad phase goes to
shifted ones, node-pair lists and an edge bucket that overflow, then lists of
pairs, of tests and of registry entries that are too short.  It must end with
the outputs of the same dispatch on the walk, and so must the next one, whose
lists are long enough."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pair():
    from test_gpu_edge_buckets import crowded
    g = np.random.default_rng(9)
    V, F, _ = crowded(4000)  # disjoint triangles whose edges hash to one bucket
    V = np.floor(g.random(V.shape) * 127)
    T = np.asarray(F).reshape(-1, 3)
    n = len(T)
    a = np.floor(g.random((n, 2)) * 40)  # large ones, each in a plane of whole z
    size = 50 + np.floor(g.random(n) * 36)
    z = 1 + np.floor(g.random(n) * 125)
    flip = np.where(g.random(n) < 0.5, 1.0, 0.0)
    V[T[:, 0]] = np.stack([a[:, 0] + flip * size, a[:, 1] + flip * size, z], 1)
    V[T[:, 1]] = np.stack([a[:, 0] + size, a[:, 1], z], 1)
    V[T[:, 2]] = np.stack([a[:, 0], a[:, 1] + size, z], 1)
    m = 170000  # small ones through the planes
    c = np.floor(g.random((m, 3)) * 125)
    W = np.repeat(c, 3, 0).reshape(m, 3, 3)
    W[:, 1] += [1, 0, 2]
    W[:, 2] += [0, 1, 2]
    return (V + 2.0 ** 52, F, None), (W.reshape(-1, 3) + 2.0 ** 52, np.arange(3 * m, dtype=np.uint32), None)


def test_every_reason_in_one_dispatch():
    from mcut_amd import frontend
    p = pair()
    c = frontend.Context(0)
    try:
        c.set_tuning(wave_leaves=16)
        W = c.dispatch(*p)
        want = W.status, W.counts, W.registry()
    finally:
        c.close()
    print(want[1], flush=True)
    assert want[1]["pairs"] > 4 * 174000 and want[1]["registry"] > 1 << 18
    c = frontend.Context(0)
    try:
        for _ in range(2):
            R = c.dispatch(*p)
            assert R.status == want[0] and R.counts == want[1]
            for x, y in zip(R.registry(), want[2]):
                assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
    finally:
        c.close()
