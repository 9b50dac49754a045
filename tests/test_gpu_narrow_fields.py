"""The mixed form's FP32 fields through the FP64 calls of the ABI.

Up to 98,304 values are converted on the host, more of them on the device:
both round to nearest and give back what is stored.
"""
import ctypes

import numpy as np
import pytest

import lulesh_amd as la

pytestmark = pytest.mark.gpu


def _values(n, seed):
    r = np.random.RandomState(seed)
    v = r.standard_normal(n) * 10.0 ** r.uniform(-44, 38, n)  # FP32 subnormals and overflow among them
    v[:8] = [0.0, -0.0, np.inf, -np.inf, np.nan, 1 + 2.0 ** -24, 1 + 3 * 2.0 ** -24, 3.4028235677973366e38]
    return v


def _stored(v):
    with np.errstate(over="ignore"):
        return v.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("flags", [0, la.native.FLAG_GENERIC])
@pytest.mark.parametrize("s", [5, 46, 47])  # 97,336 and 103,823 elements
def test_fields_come_back_rounded_once(s, flags):
    ctx = la.SedovDevice(s, precision=la.MIXED, flags=flags)
    others = {f: ctx.download(f) for f in ("x", "zd", "e", "v", "volo", "nodalMass")}
    fields = {f: _values(s ** 3, i) for i, f in enumerate(("p", "q", "ss", "delv_zeta"))}
    for f, v in fields.items():
        ctx.upload(f, v)
    for f, v in fields.items():
        got, want = ctx.download(f), _stored(v)
        assert np.array_equal(got, want, equal_nan=True), f
        assert np.array_equal(np.signbit(got[:2]), np.signbit(want[:2])), f
    for f, v in others.items():
        assert np.array_equal(ctx.download(f), v), f


def test_ensemble_members_between_cycles():
    """A member's fields are moved through scratch that no member holds."""
    sizes = [47, 6, 48]
    ens = la.Ensemble(sizes, [1.0, 1.5, 0.7], [1, 1, 2], [1, 2, 1], precision=la.MIXED)
    assert ens.run(5)[0] == 0
    lib = la.gpu_lib()

    def download(m, f):
        n = (sizes[m] + 1) ** 3 if f in la.native.NODE_FIELDS else sizes[m] ** 3
        out = np.empty(n)
        la.check(lib.lgpu_ensemble_download(ens.dev, m, la.FIELDS.index(f),
                                            out.ctypes.data_as(ctypes.POINTER(ctypes.c_double))))
        return out

    before = [{f: download(m, f) for f in ("x", "yd", "p", "q", "e")} for m in range(3)]
    new = _values(sizes[2] ** 3, 9)
    ens.upload(2, "q", new)
    assert np.array_equal(download(2, "q"), _stored(new), equal_nan=True)
    ens.upload(2, "q", before[2]["q"])
    for m in range(3):
        for f, v in before[m].items():
            assert np.array_equal(download(m, f), v), (m, f)
