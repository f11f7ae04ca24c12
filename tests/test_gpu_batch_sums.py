"""Coordinate sums of a batch, three coordinates of a mesh in one wave: vertex
counts around its steps (a row of 16 lanes, a wave of 64, their multiples) and
meshes of very different lengths in one batch.  A sum in any other order moves
the shift, and with it the bits of the points, off those of the plain dispatch
(which the oracle holds)."""
import numpy as np
import pytest

from mcut_amd import meshgen as mg

pytestmark = pytest.mark.gpu


def box(nv, seed, centre):
    """A rotated box of 12 triangles (8 vertices) behind nv - 8 unused vertices."""
    V, F, _ = mg.tessellated_box(centre, 1.0, 1, rotation=mg.random_rotation(seed), triangulate=True)
    V = np.asarray(V)
    pad = 0.3 * np.random.default_rng(seed).random((nv - len(V), 3)) + np.array(centre)
    return np.vstack([pad, V]), (np.asarray(F) + nv - len(V)).astype(np.uint32), None


@pytest.mark.parametrize("counts", [
    [(8, 9), (15, 16), (17, 31), (32, 33), (47, 48), (49, 63)],
    [(63, 64), (64, 65), (65, 127), (128, 129), (191, 192), (193, 8)],
    [(8, 20011), (20011, 8), (1023, 1024), (1025, 4097), (4096, 4095), (8, 8)],
])
def test_batch_sums_match_plain(counts):
    from mcut_amd import frontend
    pairs = [(box(a, 10 + i, (0.0, 0.0, 0.0)), box(b, 50 + i, (0.45, 0.3, 0.2))) for i, (a, b) in enumerate(counts)]
    ctx, plain = frontend.Context(0), frontend.Context(0)
    try:
        B = ctx.dispatch_batch(pairs)
        for i, (s, c) in enumerate(pairs):
            R = plain.dispatch(s, c)
            assert B.status[i] == R.status and R.counts["registry"] > 0
            for x, y in zip(B.pair_registry(i), R.registry()):
                assert np.array_equal(x, y), counts[i]
    finally:
        ctx.close()
        plain.close()
