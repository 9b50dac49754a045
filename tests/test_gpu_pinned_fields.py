"""The mixed form's FP32 fields in pinned and in ordinary host memory.

Large fields are converted on the device where that is the shorter way, which for
ordinary memory, whose every byte is copied once more on the host, it is not
(uploads beyond 1,048,576 values apart).  Both ways round once and give back what
is stored.  Which way a field goes is checked on the host (no GPU: the fake HIP
runtime).
"""
import ctypes

import numpy as np
import pytest

import fake_hip
import lulesh_amd as la
from hip_buffers import HipBuffers

# s: p is converted on the device for (pinned up, down, ordinary up, down)
WAYS = {46: (False, False, False, False), 50: (False, True, False, False), 54: (True, True, False, False),
        102: (True, True, True, False)}  # 97,336, 125,000, 157,464 and 1,061,208 values


def _ways(fake, la, s, ensemble):
    import ctypes
    dp = ctypes.POINTER(ctypes.c_double)
    lib, p = la.gpu_lib(), la.FIELDS.index("p")
    if ensemble:
        owner = la.Ensemble([s], [1.0], [1], [1], precision=la.MIXED)
        up, down = (lambda a, f=f: f(owner.dev, 0, p, a) for f in (lib.lgpu_ensemble_upload, lib.lgpu_ensemble_download))
    else:
        owner = la.SedovDevice(s, precision=la.MIXED)
        up, down = (lambda a, f=f: f(owner.ptr, p, a) for f in (lib.lgpu_upload, lib.lgpu_download))
    ways = []
    for array in (fake.pinned(8 * s ** 3), (ctypes.c_double * s ** 3)()):
        for call in (up, down):
            fake.launches()
            la.check(call(ctypes.cast(array, dp)))
            ways.append(any("k_convert" in k for k in fake.launches()))
    return ways


@pytest.mark.parametrize("ensemble", [False, True])
@pytest.mark.parametrize("s", sorted(WAYS))
def test_fields_go_the_shorter_way(s, ensemble):
    assert tuple(fake_hip.run(_ways, s, ensemble)) == WAYS[s]


@pytest.mark.gpu
@pytest.mark.parametrize("s", sorted(WAYS))
def test_pinned_and_ordinary_memory_hold_the_same(s):
    n, dp = s ** 3, ctypes.POINTER(ctypes.c_double)
    lib, p = la.gpu_lib(), la.FIELDS.index("p")
    hip, ptr = HipBuffers().hip, ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(ptr), ctypes.c_size_t(8 * n), 0) == 0
    pinned = np.ctypeslib.as_array(ctypes.cast(ptr, dp), (n,))
    r = np.random.RandomState(s)
    values = r.standard_normal(n) * 10.0 ** r.uniform(-44, 37, n)  # FP32 subnormals among them
    values[:6] = [0.0, -0.0, np.inf, -np.inf, 1 + 2.0 ** -24, 1 + 3 * 2.0 ** -24]
    want = values.astype(np.float32).astype(np.float64)
    ctx = la.SedovDevice(s, precision=la.MIXED)
    others = {f: ctx.download(f) for f in ("x", "e", "v")}
    for up_pinned in (True, False):
        pinned[:] = values
        la.check(lib.lgpu_upload(ctx.ptr, p, ctypes.cast(ptr, dp) if up_pinned else values.ctypes.data_as(dp)))
        pinned[:] = np.nan
        la.check(lib.lgpu_download(ctx.ptr, p, ctypes.cast(ptr, dp)))
        for got in (pinned, ctx.download("p")):
            assert np.array_equal(got.view(np.int64), want.view(np.int64)), up_pinned
        ctx.upload("p", np.zeros(n))
    for f, v in others.items():
        assert np.array_equal(ctx.download(f), v), f
    ctx.close()
    assert hip.hipHostFree(ptr) == 0
