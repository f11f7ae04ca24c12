"""The edge numbering by LDS buckets where it can go wrong, against the oracle:
meshes of one bucket and the first ones of several (4,096 corners), a ragged
scatter tile, wide scatter tiles (more than 2^19 corners), tiles of ranks, open
borders, polygon corners, and a soup built so that one bucket overflows, which
the hash tables then number."""
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


def strip(n):
    """An open fan-free strip of n triangles across the z = 0 plane."""
    i = np.arange(n + 2)
    V = np.stack([0.01 * i, np.where(i % 2, 0.3, -0.2) + 0.001 * (i % 7), np.where(i % 3, 0.11, -0.13)], 1)
    j = np.arange(n)
    F = np.where((j % 2)[:, None], np.stack([j + 1, j, j + 2], 1), np.stack([j, j + 1, j + 2], 1))
    return V, F.astype(np.uint32).ravel(), None


def blade(length):
    """A sheet through the strip, near its plane of symmetry."""
    G, F, _ = mg.grid_patch(3, 1.0)
    return G * [length, 1.0, 1.0] + [0.45 * length, 0.01, 0.003], F, None


@pytest.mark.parametrize("n", [1, 2, 1365, 1366, 2731, 5462, 174763, 699051])
def test_strip_sizes(ctx, n):
    # 1365 triangles: 4,095 corners, one bucket; 1366: 4,098, four; 174,763: past
    # 2^19 corners (8 a thread in the scatter); 699,051: past 2^21 (16 a thread)
    compare(ctx, strip(n), blade(0.01 * n), detail=n < 10000)
    R = ctx.dispatch(strip(n), blade(0.01 * n))
    v0, v1, f0, f1 = R.edges()
    assert v0.size == 2 * n + 1 + 33  # the strip's edges and the sheet's
    assert int((f1 < 0).sum()) == n + 2 + 12


@pytest.mark.parametrize("n,m", [(4, 5), (19, 30), (60, 24)])
def test_polygon_corners(ctx, n, m):
    box = mg.tessellated_box((0, 0, 0), 1.0, n, rotation=mg.random_rotation(3), triangulate=False)
    cut = mg.tessellated_box((0.4, 0.3, 0.2), 0.9, m, rotation=mg.random_rotation(4), triangulate=False)
    compare(ctx, box, cut)


def _bucket(group, vbits, bb):
    """The bucket of the edges within one group of eight vertices (topo_word)."""
    gb = 2 * (vbits - 3)
    mask = (1 << gb) - 1
    h = ((group << (vbits - 3)) | group) & mask
    h = (h * 0x9e3779b97f4a7c15) & mask
    h ^= h >> (gb // 2)
    h = (h * 0xd6e8feb86659fd93) & mask
    h ^= h >> (gb // 2)
    return h >> (gb - bb)


def crowded(triangles=1500, vbits=17):
    """Disjoint triangles whose edges all hash to one bucket of four or eight."""
    k = 3 * triangles
    bb = 0
    while (2048 << bb) < k:
        bb += 1
    pick = [g for g in range(1 << (vbits - 3)) if _bucket(g, vbits, bb) == 1][:triangles // 2]
    assert len(pick) * 2 == triangles and k > 4096
    g = np.random.default_rng(1)
    V = np.zeros((1 << vbits, 3))
    V[:, 0] = np.arange(1 << vbits) * 1e-5
    V[:, 1:] = g.random((1 << vbits, 2)) - 0.5
    F = np.concatenate([[8 * p, 8 * p + 1, 8 * p + 2, 8 * p + 3, 8 * p + 4, 8 * p + 5] for p in pick])
    return V, F.astype(np.uint32), None


def test_overflowing_bucket_falls_back_to_the_tables(ctx):
    src = crowded()
    G, F, _ = mg.grid_patch(4, 3.0)
    cut = (np.stack([G[:, 0] + 0.6, G[:, 2] + 0.01 + 0.02 * G[:, 1], G[:, 1]], 1), F, None)
    R, O = compare(ctx, src, cut)
    compare(ctx, *meshes.icosphere_pair(4))  # the next dispatch numbers its edges by buckets again
    compare(ctx, cut, src)


def fans(rings, hub):
    """A closed double fan over each ring of vertices: two hubs a ring, every
    other vertex on four faces."""
    V, F = [], []
    base = 0
    for r in rings:
        t = np.linspace(0, 2 * np.pi, r, endpoint=False)
        ring = np.stack([np.cos(t), np.sin(t), 0 * t], 1) + [0, 0, 3.0 * len(V)]
        ends = np.array([[0, 0, -1.0], [0, 0, 1.0]]) + [0, 0, 3.0 * len(V)]
        i = np.arange(r)
        if hub == "first":
            V.append(np.vstack([ends, ring]))
            lo, hi, o = base, base + 1, base + 2
        else:
            V.append(np.vstack([ring, ends]))
            lo, hi, o = base + r, base + r + 1, base
        F.append(np.stack([o + i, o + (i + 1) % r, 0 * i + hi], 1))
        F.append(np.stack([o + (i + 1) % r, o + i, 0 * i + lo], 1))
        base += r + 2
    return np.vstack(V), np.concatenate(F).astype(np.uint32).ravel(), None


@pytest.mark.parametrize("hub", ["first", "last"])
@pytest.mark.parametrize("rings", [[100000], [3000] * 40, [700] * 200])
def test_vertices_of_many_faces(ctx, rings, hub):
    # past 2^19 corners the buckets are vertex ranges unless one holds too much:
    # a hub of 100,000 or 3,000 faces does (hashed buckets), of 700 does not
    src = fans(rings, hub)
    cut = blade(1.0)
    compare(ctx, src, cut, detail=False)
    R = ctx.dispatch(src, cut)
    v0, v1, f0, f1 = R.edges()
    assert v0.size == 3 * sum(rings) + 33 and int((f1 < 0).sum()) == 12


@pytest.mark.parametrize("index", [0, 1, 2])
@pytest.mark.parametrize("value", ["nv", "max"])
def test_refused_lists_of_large_meshes(ctx, index, value):
    # an index past the vertices, in meshes whose buckets are vertex ranges:
    # refused, alone and in a batch, and the context goes on
    from mcut_amd import frontend
    V, F, _ = strip(174763)
    bad = F.copy()
    bad[3 * 1000 + index] = V.shape[0] if value == "nv" else 0xffffffff
    with pytest.raises(frontend.McgpuError) as e:
        ctx.dispatch((V, bad, None), blade(1.0))
    assert e.value.code == -1
    with pytest.raises(frontend.McgpuError) as e:
        ctx.dispatch_batch([((V, F, None), blade(1.0)), ((V, bad, None), blade(1.0))])
    assert e.value.code == -1
    assert ctx.dispatch((V, F, None), blade(1.0)).counts["edges"] == 2 * 174763 + 1 + 33
