"""Batches on the device whose last pair starts with a face of no corners or of
fewer than three, which only the kernels see: refused, and the context goes
on.  The pair's first corner then lies at the end of the corner arrays."""
import ctypes as C

import numpy as np
import pytest

from mcut_amd import meshgen as mg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [0, 1, 2])
@pytest.mark.parametrize("side", [0, 1])
def test_faces_of_too_few_corners(side, size):
    from mcut_amd import frontend
    ctx = frontend.Context(0)
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library loaded
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    keep = []

    def up(a):
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), max(a.nbytes, 4)) == 0
        assert hip.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0
        keep.append(p)
        return p.value

    def part(k, m, bad):
        """A part of two pairs: a box of quads each, or the second one's only face too small."""
        V, F, S = mg.tessellated_box((0.4 * k, 0.3 * k, 0.2 * k), 1.0, m, rotation=mg.random_rotation(3 + k), triangulate=False)
        F, S = np.asarray(F, np.uint32).ravel(), np.asarray(S, np.uint32)
        F2, S2 = (np.arange(size, dtype=np.uint32), np.array([size], np.uint32)) if bad else (F, S)
        VV, FF, SS = np.vstack([V, V]), np.concatenate([F, F2]), np.concatenate([S, S2])
        mesh = frontend.device_mesh(up(VV), up(FF), up(SS), len(VV), len(SS))
        return mesh, np.array([0, len(V), len(VV)], np.uint32), np.array([0, len(S), len(SS)], np.uint32)

    try:
        def dispatch(bad):
            a, av, af = part(0, 4, bad and side == 0)
            b, bv, bf = part(1, 3, bad and side == 1)
            return ctx.dispatch_batch_device(2, a, b, [av, af, bv, bf])
        with pytest.raises(frontend.McgpuError) as e:
            dispatch(True)
        assert e.value.code == -1
        R = dispatch(False)
        assert list(R.status) == [0, 0] and R.info.num_registry > 0
    finally:
        ctx.close()
        for p in keep:
            hip.hipFree(p)
