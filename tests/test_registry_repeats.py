"""Registries in which an (edge, face) comes more than once: a caller's list of
pairs may name a pair twice (mcgpu_dispatch_narrow).

CPU: the places that the registry's sort counts for its entries
(mcut_amd/csrc/regrank.hpp, compiled for the host) against a stable sort, with
keys that repeat, within a group of 16, across runs and across tiles of 4,096.

GPU: a list with every pair repeated has each entry of the list's own
registry that often, in the same order."""
import os
import subprocess

import numpy as np
import pytest

import meshes
from mcut_amd import meshgen as mg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed")
def test_places_of_repeated_keys(tmp_path):
    exe = tmp_path / "regrank_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "--offload-arch=gfx950", "--offload-host-only",
                    "-I", os.path.join(ROOT, "mcut_amd", "csrc"), os.path.join(ROOT, "tests", "support", "regrank_check.cpp"),
                    "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.split()[-2:] == ["bad", "0"], out.stdout


def soup(src, cut):
    """The meshes in their own coordinates and their face boxes."""
    out = []
    for V, F, _ in (src, cut):
        T = V[np.asarray(F).reshape(-1, 3)]
        out.append(np.hstack([T.min(1), T.max(1)]))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("times", [2, 9])
@pytest.mark.parametrize("level,cells", [(2, 3), (3, 12), (5, 40)])
def test_repeated_pairs(level, cells, times):
    # registries of one group, of runs, and (level 5, nine times) of several tiles
    from mcut_amd import frontend
    src = meshes.icosphere_pair(level)[0]
    G, F, _ = mg.grid_patch(cells, 3.0)
    cut = (G + [0.01, 0.02, 0.013] + 0.02 * np.sin(3 * G[:, :1]) * [0, 0, 1], F, None)
    sb, cb = soup(src, cut)
    ctx = frontend.Context(0)
    try:
        pairs = ctx.broad_phase(sb, cb)
        R = ctx.dispatch_narrow(src, cut, sb, cb, pairs)
        e, g, p = R.registry()
        status = R.status
        print(level, len(pairs), len(e), flush=True)
        assert len(e) > 0
        again = np.concatenate([pairs] * times)
        again = again[np.random.default_rng(level).permutation(len(again))]
        R = ctx.dispatch_narrow(src, cut, sb, cb, np.ascontiguousarray(again))
        e2, g2, p2 = R.registry()
        assert R.status == status and len(e2) == times * len(e)
        assert np.array_equal(e2, np.repeat(e, times)) and np.array_equal(g2, np.repeat(g, times))
        assert np.array_equal(p2.view(np.uint64), np.repeat(p, times, axis=0).view(np.uint64))
    finally:
        ctx.close()
