"""What a dispatch does before its streams part, at the edges of its branches,
against the oracle: polygon meshes whose face offsets one block scans (a tile
of 4,096 faces, several, the last size and the first the general scan takes),
one mesh of polygons and one of triangles either way round, leaf keys of 16 and
22 bits (up to and past 2^15 leaves), a chain of 4,096 vertices and one past it
beside a short one, and every face list fault."""
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


def quads(n):
    return mg.tessellated_box((0, 0, 0), 1.0, n, rotation=mg.random_rotation(3), triangulate=False)


def cube(triangulate=False):
    return mg.tessellated_box((0.4, 0.3, 0.2), 0.9, 1, rotation=mg.random_rotation(4), triangulate=triangulate)


@pytest.mark.parametrize("n", [1, 26, 27, 104, 105])
def test_polygon_offsets(ctx, n):
    compare(ctx, quads(n), cube(), detail=n < 30)


def test_polygons_and_triangles(ctx):
    compare(ctx, quads(9), cube(True))
    compare(ctx, cube(True), quads(9))


@pytest.mark.parametrize("a,b", [(90, 90), (90, 91), (91, 91)])
def test_leaf_keys(ctx, a, b):
    # 16,200 or 16,562 triangles each: 32,400, 32,762 and 33,124 leaves of trees
    A, F, _ = mg.grid_patch(a, 1.0)
    B, G, _ = mg.grid_patch(b, 1.0)
    B = (np.asarray(B) @ mg.random_rotation(8).T) + [0.013, 0.017, 0.019]
    compare(ctx, (np.asarray(A), F, None), (B, G, None), detail=False)


@pytest.mark.parametrize("nv", [4096, 4097])
def test_sums_at_the_serial_limit(ctx, nv):
    V, F, _ = cube(True)
    V, F = np.asarray(V), np.asarray(F)
    g = np.random.default_rng(nv)
    pad = V[0] + 0.01 * g.random((nv - V.shape[0], 3)) # vertices that no face uses
    big, small = (np.vstack([V, pad]), F, None), quads(3)
    compare(ctx, big, small)
    compare(ctx, small, big)


@pytest.mark.parametrize("polygon", [False, True])
@pytest.mark.parametrize("fault", ["index", "repeat"])
@pytest.mark.parametrize("side", [0, 1])
def test_face_list_faults(ctx, polygon, fault, side):
    from mcut_amd import frontend
    pair = [quads(3) if polygon else cube(True), quads(2) if polygon else cube(True)]
    V, F, S = pair[side]
    F = np.array(F, np.uint32)
    F[-1] = V.shape[0] if fault == "index" else F[-2]
    pair[side] = (V, F, S)
    with pytest.raises(frontend.McgpuError) as e:
        ctx.dispatch(*pair)
    assert e.value.code == -1
