"""Which face of an edge emits its edge-face test: the rule for the broad
phase's own pairs and the one for pairs kept while the cut mesh moves (also
further than the cut boxes were widened by), each against the hash of the given
pairs, on triangles and polygons, on closed and open meshes."""
import numpy as np
import pytest

import meshes
from mcut_amd import meshgen as mg
from test_narrow import soup_inputs

pytestmark = pytest.mark.gpu


def polygons():
    return (mg.tessellated_box((0, 0, 0), 1.0, 7, rotation=mg.random_rotation(3), triangulate=False),
            mg.tessellated_box((0.4, 0.3, 0.2), 0.9, 5, rotation=mg.random_rotation(4), triangulate=False))


def sheet():
    G, F, _ = mg.grid_patch(9, 3.0)
    V, T, _ = meshes.icosphere_pair(3)[0]
    return (V, T, None), (G + [0.01, 0.02, 0.003], F, None)


@pytest.mark.parametrize("pair", [meshes.config1_rotated(), meshes.icosphere_pair(3), polygons(), sheet()],
                         ids=["box", "icosphere", "polygons", "sheet"])
@pytest.mark.parametrize("move", [0.0, 1e-7, 0.05])
def test_rules_agree(pair, move):
    from mcut_amd import frontend
    src, cut = pair
    Vs = np.asarray(src[0]).reshape(-1, 3).shape[0]
    Vc = np.asarray(cut[0]).reshape(-1, 3).shape[0]
    a, b = frontend.Context(0), frontend.Context(0)
    try:
        R = a.dispatch(src, cut, flags=1 << 15)
        s2, c2, sb, cb, pairs = soup_inputs(R, src, cut)
        if move:
            R = a.redispatch_perturbed(np.array([move, -0.6 * move, 0.3 * move]), 1, Vs + Vc)
            c2 = (R.ps_vertices()[Vs:],) + tuple(c2[1:])
        N = b.dispatch_narrow(s2, c2, sb, cb, pairs, flags=1 << 15, enforcement_count=1 if move else 0)
        assert N.status == R.status and N.counts["pairs"] == R.counts["pairs"]
        assert N.counts["tests"] == R.counts["tests"] > 0
        for x, y in zip(N.registry(), R.registry()):
            assert np.array_equal(x, y)
    finally:
        a.close()
        b.close()
