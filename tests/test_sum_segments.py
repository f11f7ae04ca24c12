"""Coordinate sums from segments that move with their start
(mcut_amd/csrc/sumseg.hpp, k_sum_items .. k_sum_rest) against the left-to-right
sum, bit for bit.

CPU: the header's own walk, composition and adds, compiled for the host, on
values that hover about zero, cancel to noise, lie on grids, tie, span scales,
leave the double range, with predictions pushed off by up to 0.37; every result
must be the sequential one, and the usual inputs must need no replay.

GPU: the centre of vertex arrays at the sizes where the kernels change (one
serial chain up to 4,096 values, tiles of 4,096, chunks of 64, more than 16,384
adds), against the oracle."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is needed")
def test_segments_reproduce_the_sequential_sum(tmp_path):
    exe = tmp_path / "sumseg_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-ffp-contract=off", "--offload-arch=gfx950", "--offload-host-only",
                    "-I", os.path.join(ROOT, "mcut_amd", "csrc"), os.path.join(ROOT, "tests", "support", "sumseg_check.cpp"),
                    "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0 and out.stdout.split()[-2:] == ["bad", "0"], out.stdout
    rows = {ln.split()[0]: dict(p.split("=") for p in ln.split()[1:5]) for ln in out.stdout.splitlines() if " n=60000 " in ln}
    for name in ("hover", "normal", "positive", "offset", "rings", "grid", "gridz", "ties", "scales", "zeros", "walk"):
        assert rows[name]["replayed"] == "0", (name, rows[name])
    assert int(rows["positive"]["l1"]) < 60000 / 32 and int(rows["hover"]["l1"]) < 60000 / 16


VALUES = {
    "uniform": lambda g, n: g.uniform(-1, 1, (n, 3)),
    "positive": lambda g, n: g.uniform(0.2, 1.2, (n, 3)),
    "thirds": lambda g, n: np.stack([(np.arange(n) % 31 - 15.0) / 30.0] * 3, 1) + [0.0, 0.1, 1.0 / 3],
    "rings": lambda g, n: np.stack([np.sin(2 * np.pi * (np.arange(n) % 64) / 64) * (1 + np.arange(n) // 64 % 16)] * 3, 1),
    "steps": lambda g, n: g.normal(size=(n, 3)) * 2.0 ** g.integers(-30, 30, (n, 3)),
    "ties": lambda g, n: np.round(g.uniform(-1, 1, (n, 3)) * 2 ** 30) / 2 ** 30 + 2.0 ** 21,
}


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4096, 4097, 8192, 8193, 12351, 70001])
@pytest.mark.parametrize("name", list(VALUES))
def test_centre_bits_at_the_kernels_edges(ctx, name, n):
    from oracle import oracle as om
    g = np.random.default_rng(n)
    V = np.ascontiguousarray(VALUES[name](g, n))
    W = np.ascontiguousarray(VALUES[name](g, 1 + n // 3) + 0.01)
    F = np.arange(3, dtype=np.uint32)
    R = ctx.dispatch((V, F, None), (W, F, None))
    O = om.frontend((V, F, None), (W, F, None), detail=False)
    assert np.array_equal(R.com.view(np.uint64), np.asarray(O["com"]).view(np.uint64))
    assert np.array_equal(R.t.view(np.uint64), np.asarray(O["t"]).view(np.uint64))
