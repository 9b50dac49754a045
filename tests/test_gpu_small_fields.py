"""Small fields travel by a kernel through pinned memory: the same bits as the
copies of larger fields, after the stream's earlier work.
"""
import ctypes

import numpy as np
import pytest

import lulesh_amd as la

pytestmark = pytest.mark.gpu


def _bits(n, seed):
    v = np.random.RandomState(seed).randint(0, 2 ** 63, n, dtype=np.int64)  # NaNs and subnormals among them
    return v.view(np.float64)


# one value, whole and part waves of 128, beyond 2,048, of which single problems copy FP64 otherwise
@pytest.mark.parametrize("s", [1, 4, 7, 11, 12, 13])
def test_every_bit_comes_back(s):
    ctx = la.SedovDevice(s)
    names = ["x", "zd", "e", "v", "ss", "delv_xi"]
    fields = {f: _bits((s + 1) ** 3 if f in la.native.NODE_FIELDS else s ** 3, i) for i, f in enumerate(names)}
    for f, v in fields.items():
        ctx.upload(f, v)
    for f, v in fields.items():
        assert np.array_equal(ctx.download(f).view(np.int64), v.view(np.int64)), f
    ctx.close()


def test_copies_follow_enqueued_cycles():
    """A download right after cycles that are only enqueued, and an upload
    that the next cycles read, against a context that waits in between."""
    got = []
    for wait in (False, True):
        ctx = la.SedovDevice(11)
        ctx.run(5)
        e = ctx.download("e")
        for k in range(3):
            assert ctx.lagrange_nodal(1e-6) == 0 and ctx.lagrange_elements(1e-6) == 0
            if wait:
                assert ctx.time_constraints()[0] == 0
            e = ctx.download("e")
            e[k] *= 1.5
            ctx.upload("e", e)
        assert ctx.lagrange_nodal(1e-6) == 0 and ctx.lagrange_elements(1e-6) == 0
        got.append([ctx.download(f) for f in ("x", "e", "p", "q")])
        ctx.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", [la.FP64, la.MIXED])
def test_members_keep_apart(precision):
    sizes = [5, 3, 12, 13]  # odd offsets; nodes of the third and both of the last are large
    ens = la.Ensemble(sizes, [1.0] * 4, [1] * 4, [1] * 4, precision=precision)
    lib, dp = la.gpu_lib(), ctypes.POINTER(ctypes.c_double)
    fields = {(m, f): np.random.RandomState(9 * m + i).standard_normal((s + 1) ** 3 if f == "x" else s ** 3)
              .astype(np.float32).astype(np.float64)
              for m, s in enumerate(sizes) for i, f in enumerate(("x", "e", "p", "ss"))}
    for (m, f), v in fields.items():
        ens.upload(m, f, v)
    for (m, f), v in fields.items():
        out = np.empty(v.size)
        la.check(lib.lgpu_ensemble_download(ens.dev, m, la.FIELDS.index(f), out.ctypes.data_as(dp)))
        assert np.array_equal(out, v), (m, f)
    ens.close()
