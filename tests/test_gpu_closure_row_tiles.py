"""Training rows where their tiles end: every stencil feature equals the centre feature of the neighbour's own row.

A row's slot s of either input is the value at the stencil point s, clamped into the range, and that point's own row
holds the same value in its centre slot, rounded to bf16 from the same FP32 value: equal bit for bit.  (The centre
slots themselves are checked against the domain's arrays in test_gpu_closure.py.)  Ranges of 10, 63 and 65 columns:
one short tile, one that ends with column 64, one that starts a second tile; rows off a 16-byte boundary.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,shift", [(12, 0), (65, 0), (67, 1)])
def test_stencil_slots_are_the_neighbours_centres(gpu, nx, shift):
    import torch

    from wrfdc.cases import make_case
    from wrfdc.closure import NFEAT, NTARGET, ClosureNorm, row_count
    from wrfdc.device import Domain

    print(f"[closure] rows of {nx}x13x7, {shift} elements off alignment", flush=True)
    case = make_case(nx, 13, 7, nmoist=1, hill_height=300.0)
    dom = Domain(case.config, gpu)
    dom.upload(case.arrays)
    n = row_count(dom.config)
    flat = torch.full((n * NFEAT + 8,), 7.0, dtype=torch.bfloat16, device=gpu)
    T = torch.zeros((n, NTARGET), dtype=torch.float32, device=gpu)
    nm = ClosureNorm(-7.0, 0.5, 1e-4, 1e-4, 1.25, 100.0).as_struct()
    rc = dom.lib.wrfdc_closure_rows(dom.ctx, ctypes.byref(nm), ctypes.c_void_p(flat.data_ptr() + 2 * shift),
                                    ctypes.c_void_p(T.data_ptr()))
    assert rc == 0
    dom.synchronize()
    assert (flat[:shift] == 7.0).all() and (flat[shift + n * NFEAT:] == 7.0).all()
    X = flat[shift:shift + n * NFEAT].float().cpu().numpy().reshape(11, 7, nx - 2, 2, 32)
    dom.close()
    j, k, i = np.meshgrid(np.arange(11), np.arange(7), np.arange(nx - 2), indexing="ij")
    for s in range(27):
        jj, kk, ii = np.clip(j + s // 9 - 1, 0, 10), np.clip(k + s // 3 % 3 - 1, 0, 6), np.clip(i + s % 3 - 1, 0, nx - 3)
        assert np.array_equal(X[..., s], X[jj, kk, ii, :, 13]), s
    assert (X[..., 0, 27] == 1.25).all() and (X[..., 1, 27] == 0.0).all() and (X[..., 28:] == 0.0).all()
