"""Ensembles whose fields travel both ways: those of small members by the copy
kernel, waited for by its counts, and those of a large one by hipMemcpy.  Every
value arrives where it belongs, whichever way the field before it went.  That the
members go by both ways is checked on the host (no GPU: the fake HIP runtime).
"""
import ctypes

import numpy as np
import pytest

import fake_hip
import lulesh_amd as la

SIZES = [5, 3, 4, 6, 26]  # the last one's nodes and elements are above the limit of 16,384 values
FIELDS = ["x", "e", "p", "ss"]


def _ways(fake, la, sizes, fields, precision):
    import numpy as np
    n = len(sizes)
    ens = la.Ensemble(sizes, [1.0] * n, [1] * n, [1] * n, precision=precision)
    ways = []
    for m, s in enumerate(sizes):
        for f in fields:
            fake.launches()
            before = fake.copies()
            ens.upload(m, f, np.ones((s + 1) ** 3 if f == "x" else s ** 3))
            ways.append([m, any("k_small" in k for k in fake.launches()), fake.copies() > before])
    return ways


@pytest.mark.parametrize("precision", [la.FP64, la.MIXED])
def test_members_go_by_both_ways(precision):
    for m, by_kernel, by_memcpy in fake_hip.run(_ways, SIZES, FIELDS, precision):
        assert (by_kernel, by_memcpy) == ((False, True) if SIZES[m] == 26 else (True, False)), m


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [la.FP64, la.MIXED])
def test_fields_of_both_ways_keep_apart(precision):
    n = len(SIZES)
    ens = la.Ensemble(SIZES, [1.0] * n, [1] * n, [1] * n, precision=precision)
    lib, dp = la.gpu_lib(), ctypes.POINTER(ctypes.c_double)
    rng = np.random.RandomState(3)

    def download(m, f):
        out = np.empty((SIZES[m] + 1) ** 3 if f == "x" else SIZES[m] ** 3)
        la.check(lib.lgpu_ensemble_download(ens.dev, m, la.FIELDS.index(f), out.ctypes.data_as(dp)))
        return out

    assert ens.run(3)[0] == 0
    now = {(m, f): download(m, f) for m in range(n) for f in FIELDS}
    # small and large members in turn, uploads and downloads among one another
    for step in range(120):
        m = n - 1 if step % 3 == 1 else rng.randint(n)
        f = FIELDS[rng.randint(len(FIELDS))]
        now[m, f] = rng.standard_normal(now[m, f].size).astype(np.float32).astype(np.float64)
        ens.upload(m, f, now[m, f])
        m, f = (rng.randint(n) if step % 3 == 1 else n - 1), FIELDS[rng.randint(len(FIELDS))]
        assert np.array_equal(download(m, f), now[m, f]), (step, m, f)
    for (m, f), v in now.items():
        assert np.array_equal(download(m, f), v), (m, f)
    ens.close()
