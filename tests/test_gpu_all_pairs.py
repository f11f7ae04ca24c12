"""Meshes of few faces, whose pairs of face boxes are all tested: against the
oracle and against the trees (a forced launch shape), on both sides of the
limit of 2^26 pairs, at tile edges (256 source faces, 32 cut faces), with
polygons, and with the autotuner, which needs the trees."""
import numpy as np
import pytest

import meshes
from mcut_amd import meshgen as mg
from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


def strips(n, m):
    """n and m triangles across each other, vertices of their own."""
    def strip(k, axis):
        t = np.linspace(-1, 1, k) if k > 1 else np.zeros(1)
        V = np.zeros((k, 3, 3))
        V[:, :, axis] = t[:, None] + [0.0, 1.3 / k, 0.6 / k]
        V[:, :, 1 - axis] = [-1.1, -1.2, 1.05]
        V[:, :, 2] = np.array([-0.3, 0.11, 0.35]) + 0.01 * (np.arange(k) % 5)[:, None] * (1 + axis)
        return V.reshape(-1, 3), np.arange(3 * k, dtype=np.uint32), None
    return strip(n, 0), strip(m, 1)


@pytest.mark.parametrize("n,m", [(1, 1), (255, 31), (256, 32), (257, 33), (1, 700), (700, 1), (513, 97)])
def test_tiles(ctx, n, m):
    compare(ctx, *strips(n, m))


def test_polygons(ctx):
    compare(ctx, mg.tessellated_box((0, 0, 0), 1.0, 20, rotation=mg.random_rotation(3), triangulate=False),
            mg.tessellated_box((0.4, 0.3, 0.2), 0.9, 7, rotation=mg.random_rotation(4), triangulate=False))


@pytest.mark.parametrize("faces", [(1 << 26) // 80, (1 << 26) // 80 + 160])
def test_limit(ctx, faces):
    # an icosphere of 80 faces against a strip on either side of 2^26 pairs
    V, F, _ = mg.grid_patch(int(np.sqrt(faces / 2)), 1.0)
    F = np.asarray(F).ravel()[:3 * faces]
    s = meshes.icosphere_pair(1)[0]
    src = (np.asarray(V) * [2.0, 2.0, 1.0] + [0.013, 0.011, 0.0071], F, None)
    R = ctx.dispatch(src, s)
    ctx.set_tuning(wave_leaves=16)
    try:
        W = ctx.dispatch(src, s)
        assert W.status == R.status and W.counts == R.counts and R.counts["raw_pairs"] > 0
        for x, y in zip(R.registry(), W.registry()):
            assert np.array_equal(x, y)
    finally:
        ctx.set_tuning()


def test_autotune_makes_trees():
    from mcut_amd import frontend
    c = frontend.Context(0)
    try:
        src, cut = meshes.icosphere_pair(3)
        R = c.dispatch(src, cut)
        t = c.autotune()
        assert t["candidates"] == 36 and 0 < t["traversal_ms"] <= t["default_traversal_ms"]
        W = c.dispatch(src, cut)
        assert W.counts == R.counts
        for x, y in zip(R.registry(), W.registry()):
            assert np.array_equal(x, y)
    finally:
        c.close()
