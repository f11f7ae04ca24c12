"""The coordinate sums as the kernels take them, on inputs that need every part.

CPU: a host replica of the kernels over mcut_amd/csrc/sumseg.hpp gives the
left-to-right sum, bit for bit, with no chunk's adds past its place; the
inputs that absorb small values (so that every prediction after them is off)
reach the values taken one by one, and those about a power of two the most adds.

GPU: the same inputs' centres against the oracle, and the device memory that
the sums hold."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from mcut_amd import meshgen as mg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


def absorbed(g, n):
    """Values far below the last place of the sum before them, which then cancels."""
    x = g.uniform(0.5, 1.5, n)
    x[0] = 2.0 ** 60
    x[n // 3] = -2.0 ** 60
    return x


def edges(g, n):
    """From a power of two up by a tie and back onto it, inexactly, in turn: a
    segment of five adds and a step for every two values."""
    x = np.tile([3.0, -3.6], n // 2 + 1)[:n]
    x[1:] = x[:-1].copy()
    x[0] = 2.0 ** 53
    return x


VALUES = {
    "uniform": lambda g, n: g.uniform(-1, 1, n),
    "positive": lambda g, n: g.uniform(0.2, 1.2, n),
    "absorbed": absorbed,
    "edges": edges,
    "scales": lambda g, n: g.normal(size=n) * 2.0 ** g.integers(-30, 30, n),
    "ties": lambda g, n: np.round(g.uniform(-1, 1, n) * 2 ** 30) / 2 ** 30 + 2.0 ** 21,
}
SIZES = [4097, 8192, 8255, 12351, 70001]


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc is needed")
    d = tmp_path_factory.mktemp("sumchunk")
    exe = d / "sumchunk_check"
    subprocess.run([HIPCC, "-std=c++17", "-O2", "-ffp-contract=off", "--offload-arch=gfx950", "--offload-host-only",
                    "-I", os.path.join(ROOT, "mcut_amd", "csrc"), os.path.join(ROOT, "tests", "support", "sumchunk_check.cpp"),
                    "-o", str(exe)], check=True, capture_output=True)

    def run(x):
        np.ascontiguousarray(x).tofile(d / "x")
        out = subprocess.run([str(exe), str(d / "x")], capture_output=True, text=True)
        assert out.returncode == 0, out.stdout
        return {k: int(v) for k, v in (p.split("=") for p in out.stdout.split()[:-1])}
    return run


@pytest.mark.parametrize("name", list(VALUES))
@pytest.mark.parametrize("n", SIZES)
def test_replica(check, name, n):
    r = check(VALUES[name](np.random.default_rng(n), n))
    print(name, r)
    if name in ("absorbed", "edges"):
        assert r["replayed"] > 0
    if name == "edges":
        assert r["most"] == 192
    if name in ("uniform", "positive", "ties"):
        assert r["replayed"] == 0


def meshes(name, n):
    g = np.random.default_rng(n)
    V = np.stack([VALUES[name](g, n) for _ in range(3)], 1)
    W = np.stack([VALUES[name](g, 1 + n // 3) for _ in range(3)], 1)
    F = np.arange(3, dtype=np.uint32)
    return (V, F, None), (W, F, None)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(VALUES))
@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("swap", [False, True])
def test_centres(name, n, swap):
    from mcut_amd import frontend
    from oracle import oracle as om
    pair = meshes(name, n)
    pair = pair[::-1] if swap else pair
    c = frontend.Context(0)
    try:
        R = c.dispatch(*pair)
        O = om.frontend(*pair, detail=False)
        assert np.array_equal(R.com.view(np.uint64), np.asarray(O["com"]).view(np.uint64))
        assert np.array_equal(R.t.view(np.uint64), np.asarray(O["t"]).view(np.uint64))
    finally:
        c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,most", [("dispatch", 1800), ("given pairs", 1000)])
def test_device_memory(kind, most):
    """What a larger pair adds to a context's buffers, in bytes a vertex: a sheet
    of 251,001 vertices against a small box (one mesh's sums are long), and
    given pairs, which take no sums."""
    from mcut_amd import frontend
    c = frontend.Context(0)
    hip = C.CDLL("libamdhip64.so.7")

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    def spheres(n):
        V, F, _ = mg.geodesic_sphere(n)
        return (V, F, None), (V @ mg.rotation_from_uniforms(0.3, 0.5, 0.7).T + [0.5, 0.0, 0.0], F, None)

    def boxes(m):
        T = m[0][np.asarray(m[1]).reshape(-1, 3)]
        return np.hstack([T.min(1), T.max(1)])

    try:
        def narrow(pair):
            b = boxes(pair[0]), boxes(pair[1])
            pairs = c.broad_phase(*b)
            at = free()
            c.dispatch_narrow(*pair, *b, pairs)
            return at
        small = spheres(40)
        c.dispatch(*small)  # what the kernels hold besides buffers
        narrow(small)
        if kind == "dispatch":
            V, F, _ = mg.grid_patch(500, 3.0)
            B, Fb, _ = mg.tessellated_box((0, 0, 0), 1.0, 8, rotation=mg.random_rotation(5))
            pair = (V + [0.0113, 0.0071, 0.0137], np.asarray(F).ravel(), None), (B, Fb, None)
            at = free()
            c.dispatch(*pair)
        else:
            pair = spheres(128)
            at = narrow(pair)
        held = (at - free()) / (len(pair[0][0]) + len(pair[1][0]))
        print(kind, "%.0f bytes a vertex" % held, flush=True)
        assert 0 < held < most
    finally:
        c.close()
