"""Meshes past the sizes at which the edge numbering and the coordinate sums
change: more than 2^23 corners (wide counters of the buckets' scatter) and more
than 2^21 vertices (values after a failed check in a kernel of their own),
against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [2796202, 2796203])
def test_strip_past_2_23_corners(ctx, n):
    from test_gpu_edge_buckets import blade, strip
    from test_gpu_parity import compare
    src, cut = strip(n), blade(0.01 * n)
    compare(ctx, src, cut, detail=False)
    v0, v1, f0, f1 = ctx.dispatch(src, cut).edges()
    assert v0.size == 2 * n + 1 + 33  # the strip's edges and the sheet's
    assert int((f1 < 0).sum()) == n + 2 + 12


@pytest.mark.parametrize("name", ["uniform", "absorbed"])
@pytest.mark.parametrize("n", [(1 << 21) - 4096, 1 << 21, (1 << 21) + 1, (1 << 21) + 70001])
@pytest.mark.parametrize("swap", [False, True])
def test_centres(ctx, name, n, swap):
    from oracle import oracle as om
    from test_sum_chunks import VALUES
    g = np.random.default_rng(n)
    F = np.arange(3, dtype=np.uint32)
    V = np.stack([VALUES[name](g, n) for _ in range(3)], 1), F, None
    W = np.stack([VALUES["uniform"](g, 5001) for _ in range(3)], 1) + 0.01, F, None
    pair = (W, V) if swap else (V, W)
    R = ctx.dispatch(*pair)
    O = om.frontend(*pair, detail=False)
    assert np.array_equal(R.com.view(np.uint64), np.asarray(O["com"]).view(np.uint64))
    assert np.array_equal(R.t.view(np.uint64), np.asarray(O["t"]).view(np.uint64))
