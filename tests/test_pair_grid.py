"""The grid of the broad phase's first launch (k_pairs_start) for a mesh of few
faces against one of millions, whichever of them is the source, and of a batch's
raw boxes (k_batch_bbox) for one large mesh among thousands of small ones.

CPU: the launch sizes (mcut_amd/csrc/pairgrid.hpp, compiled for the host)
against the device's limits, and the blocks' cover of the pairs.

GPU: a box of 12 faces against a sheet of 2.2 M, in both orders, against the
walk of the trees; and such a batch, whose large pair must equal the pair alone."""
import os
import subprocess

import numpy as np
import pytest

from mcut_amd import meshgen as mg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed")
def test_launches_fit_the_device(tmp_path):
    exe = tmp_path / "pairgrid_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "--offload-arch=gfx950", "--offload-host-only",
                    "-I", os.path.join(ROOT, "mcut_amd", "csrc"), os.path.join(ROOT, "tests", "support", "pairgrid_check.cpp"),
                    "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.split()[-2:] == ["bad", "0"], out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("box_first", [True, False])
def test_few_faces_against_millions(box_first):
    from mcut_amd import frontend
    V, F, _ = mg.grid_patch(1050, 3.0)  # 2,205,000 faces: more than 65,535 tiles of 32
    sheet = (V + [0.0113, 0.0071, 0.0137], np.asarray(F).ravel(), None)
    B, Fb, _ = mg.tessellated_box((0.0, 0.0, 0.0), 1.0, 1, rotation=mg.random_rotation(5))
    box = (B, Fb, None)
    pair = (box, sheet) if box_first else (sheet, box)
    c = frontend.Context(0)
    try:
        R = c.dispatch(*pair)
        got = (R.status, R.counts, *R.registry())
        assert R.counts["registry"] > 0
        c.set_tuning(wave_leaves=16)
        W = c.dispatch(*pair)
        assert (W.status, W.counts) == got[:2]
        for x, y in zip(got[2:], W.registry()):
            assert np.array_equal(x.view(np.uint8), y.view(np.uint8))
    finally:
        c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("at", [0, 2300, 4199])
def test_one_large_mesh_among_thousands(at):
    from mcut_amd import frontend
    # 66,049 vertices: 17 tiles of 4,096, a block takes three
    V, F, _ = mg.grid_patch(256, 3.0)
    sheet = (V + [0.0113, 0.0071, 0.0137], np.asarray(F).ravel(), None)
    B, Fb, _ = mg.tessellated_box((0.0, 0.0, 0.0), 1.0, 3, rotation=mg.random_rotation(5))
    G, Fg, _ = mg.grid_patch(2, 3.0)
    small = (B, Fb, None), (G + [0.0113, 0.0071, 0.0137], np.asarray(Fg).ravel(), None)
    large = (B, Fb, None), sheet
    c = frontend.Context(0)
    try:
        want = [[np.array(x) for x in c.dispatch(*p).registry()] for p in (small, large)]
        assert len(want[1][0]) > 0
        R = c.dispatch_batch([large if i == at else small for i in range(4200)])
        for i in (0, at, at - 1 if at else 1, 4199):
            for x, y in zip(R.pair_registry(i), want[i == at]):
                assert np.array_equal(np.ascontiguousarray(x).view(np.uint8), y.view(np.uint8)), i
    finally:
        c.close()
