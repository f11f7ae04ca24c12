"""The thread's last HIP error and the small copies: a getter returns its result
whatever error another library left there, and an error that a launch of the
call left is reported by the call (here one left before it stands in for it)."""
import ctypes as C

import numpy as np
import pytest

import meshes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from mcut_amd import frontend
    c = frontend.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def leave_error(ctx):
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library loaded

    def leave():
        assert hip.hipSetDevice(4096) != 0 and hip.hipPeekAtLastError() != 0
    yield leave
    hip.hipGetLastError()


def test_getters_return_their_results(ctx, leave_error):
    src, cut = meshes.icosphere_pair(3)
    R = ctx.dispatch(src, cut)
    want = R.registry(), R.pairs()
    B = ctx.dispatch_batch([(src, cut)])
    first = B.pair_registry(0)
    leave_error()
    for x, y in zip(B.pair_registry(0), first):
        assert np.array_equal(x, y)
    C.CDLL("libamdhip64.so.7").hipGetLastError()
    R = ctx.dispatch(src, cut)
    leave_error()
    for x, y in zip(R.registry(), want[0]):
        assert np.array_equal(x, y)
    assert np.array_equal(R.pairs(), want[1])
    C.CDLL("libamdhip64.so.7").hipGetLastError()


def test_errors_of_a_call_are_reported(ctx, leave_error):
    from mcut_amd import frontend
    src, cut = meshes.icosphere_pair(3)
    nv = len(src[0]) + len(cut[0])
    ctx.dispatch(src, cut)
    leave_error()
    with pytest.raises(frontend.McgpuError) as e:
        ctx.redispatch_perturbed([1e-6, 0.0, 0.0], 0, nv)
    assert e.value.code == -2
    R = ctx.dispatch(src, cut)  # the error is spent
    assert R.status == 0 and ctx.redispatch_perturbed([1e-6, 0.0, 0.0], 0, nv).status == 0
