"""The exact orient3d sign (mcut_amd/csrc/geom.hpp, compiled for the host with
the address and undefined-behaviour checks) against integer determinants: its
arrays hold the longest expansions, those of coordinates whose differences all
have a tail and scales far apart, and no sign is wrong, zeros included."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from mcut_amd import exact

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def cases(g, n):
    out = []
    # every difference with a tail: magnitudes from 2^-40 to 2^40 mixed
    out.append(g.uniform(-1, 1, (n, 4, 3)) * 2.0 ** g.integers(-40, 41, (n, 4, 3)))
    # nearly coplanar: the fourth point from the plane of the others, moved in its last place
    T = g.uniform(-1, 1, (n, 4, 3))
    w = g.uniform(-1, 1, (n, 2, 1))
    T[:, 3] = T[:, 0] + w[:, 0] * (T[:, 1] - T[:, 0]) + w[:, 1] * (T[:, 2] - T[:, 0])
    out.append(np.nextafter(T, T + g.integers(-1, 2, T.shape)))
    # coplanar exactly, on a grid, and a repeated point
    G = g.integers(-50, 51, (n, 4, 3)).astype(float)
    G[:, :, 2] = 3 * G[:, :, 0] - 2 * G[:, :, 1] + 7
    out.append(G)
    D = g.uniform(-1, 1, (n, 4, 3))
    D[:, 3] = D[:, 0]
    out.append(D)
    return np.concatenate(out)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is needed")
def test_signs(tmp_path):
    exe = tmp_path / "orient_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "tests", "support", "hostinc"),
                    "-I", os.path.join(ROOT, "mcut_amd", "csrc"), os.path.join(ROOT, "tests", "support", "orient_check.cpp"),
                    "-o", str(exe)], check=True, capture_output=True)
    P = cases(np.random.default_rng(4), 400)
    P.tofile(tmp_path / "p")
    out = subprocess.run([str(exe), str(tmp_path / "p")], capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    got = np.array(out.stdout.split(), int)
    X, _ = exact._scaled_ints(P)
    want = np.array([(v > 0) - (v < 0) for v in exact._det3(X[:, 0], X[:, 1], X[:, 2], X[:, 3])])
    assert len(got) == len(P) and (want == 0).sum() >= 800 and (want != 0).sum() >= 600
    assert np.array_equal(got, want)
