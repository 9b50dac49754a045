"""lgpu_time_constraints_noalloc around the list length up to which one
workgroup takes it in one launch: the same bits as the formulas in FP64 on the
host, which round as the device does.
"""
import numpy as np
import pytest
import torch

import lulesh_amd as la

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("listed", [False, True])
@pytest.mark.parametrize("n", [0, 1, 63, 1024, 1025, 3072, 3073, 8192])
def test_short_lists(n, listed):
    r = np.random.RandomState(n + 1)
    total = 9000
    ss, area = r.uniform(0.1, 3.0, total) * 1e3, r.uniform(1e-3, 1.0, total)
    vdov = r.standard_normal(total) * 10.0 ** r.uniform(-2, 3, total)
    vdov[r.random_sample(total) < 0.3] = 0.0
    elems = r.permutation(total)[:n].astype(np.int32) if listed else np.arange(n)
    qqc, dvovmax = 2.0, 0.1
    s, v, a = ss[elems], vdov[elems], area[elems]
    root = s * s
    root = np.where(v < 0.0, root + 64.0 * qqc * qqc * a * a * v * v, root)
    moving = v != 0.0
    want = [min([1.0e20, *(a / np.sqrt(root))[moving]]), min([1.0e20, *(dvovmax / (np.abs(v) + 1.0e-20))[moving]])]
    dev = [torch.from_numpy(x).cuda() for x in (ss, vdov, area)]
    ids = torch.from_numpy(np.ascontiguousarray(elems, np.int32)).cuda() if listed else None
    out = torch.full((2,), -1.0, dtype=torch.float64, device="cuda")
    la.check(la.gpu_lib().lgpu_time_constraints_noalloc(
        *(x.data_ptr() for x in dev), ids.data_ptr() if listed and n else None, n, qqc, dvovmax, out.data_ptr(),
        torch.cuda.current_stream().cuda_stream))
    assert out.cpu().tolist() == want
