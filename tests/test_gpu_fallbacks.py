"""The ways that a dispatch takes when a buffer of the usual one overflows are
the ones taken: what the library reports of each run (MCGPU_DEBUG) shows the
overflow, the run after it on the other way, and later dispatches on the usual
one again, or past an overflow that their longer lists no longer have."""
import re

import numpy as np
import pytest

import meshes
from mcut_amd import meshgen as mg

pytestmark = pytest.mark.gpu


@pytest.fixture
def runs(monkeypatch, capfd):
    from mcut_amd import frontend
    monkeypatch.setenv("MCGPU_DEBUG", "1")
    c = frontend.Context(0)

    def go(*pair):
        """The dispatch's runs: (node lists overflowed, bucket overflowed, walked, hash tables, shifted)."""
        capfd.readouterr()
        c.dispatch(*pair)
        lines = [ln for ln in capfd.readouterr().err.splitlines() if ln.startswith("[mcgpu]")]
        return [tuple(int(x) for x in re.search(r"ov_nodes=(\d) ov_topo=(\d) walk=(\d) hash=(\d) shifted=(\d)", ln).groups())
                for ln in lines]
    yield go
    c.close()


def test_edge_bucket(runs):
    from test_gpu_edge_buckets import crowded
    G, F, _ = mg.grid_patch(4, 3.0)
    cut = (np.stack([G[:, 0] + 0.6, G[:, 2] + 0.01 + 0.02 * G[:, 1], G[:, 1]], 1), F, None)
    for _ in range(2):  # the buckets are tried anew
        assert runs(crowded(), cut) == [(0, 1, 0, 0, 0), (0, 0, 0, 1, 0)]
        assert runs(*meshes.icosphere_pair(4)) == [(0, 0, 0, 0, 0)]


def test_every_way(runs):
    from test_gpu_reruns import pair
    p = pair()
    got = runs(*p)
    assert got[0] == (0, 1, 0, 0, 0)        # the bucket, and coordinates too far from the origin
    assert got[1] == (1, 0, 0, 1, 1)        # the lists of node pairs
    assert set(got[2:]) == {(0, 0, 1, 1, 1)} and len(got) <= 8
    # longer lists of node pairs, the buckets tried anew
    assert runs(*p) == [(0, 1, 0, 0, 0), (0, 0, 0, 1, 1)]
