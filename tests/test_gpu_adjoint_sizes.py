"""The adjoint transport at the sizes where its gather can go wrong.

12x12x6 (the smallest domain: no point has only 5th-order faces around it), 65x13x8 (a second tile of one column,
tiles of both kinds) and 40x36x12.  A window of whole steps runs the stages of the one-stage entry point with the
same arithmetic: equal bit for bit.  <M x, y> = <x, M^T y> in FP64 sums of the FP32 results: each result carries a few
ulp (6e-8) per stage, and the two sums of n products of random sign differ by less than 1e-5 of the larger norm
product / sqrt(n) bound used in test_gpu_adjoint.py, here taken relative to |Mx| |y|.
"""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,nsteps", [((12, 12, 6), 1), ((65, 13, 8), 2), ((40, 36, 12), 3)])
def test_window_is_the_stages_and_the_transpose(gpu, shape, nsteps):
    import torch

    from wrfdc.adjoint import Trajectory, Transport
    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    print(f"[adjoint] {shape}, {nsteps} steps", flush=True)
    case = make_case(*shape, nmoist=1, nscalar=0, hill_height=300.0)
    dom = Domain(case.config, gpu)
    dom.upload(case.arrays)
    tr = Transport(Trajectory(dom, nsteps))
    rng = np.random.default_rng(31)
    x, y = (torch.tensor(rng.standard_normal(case.arrays["t_2"].shape).astype(np.float32), device=gpu) for _ in range(2))
    got = tr.adjoint(y)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    qbar = y
    for n in reversed(range(nsteps)):
        acc, b2, b1 = (torch.zeros_like(y) for _ in range(3))
        for rk, out, into in ((3, qbar, b2), (2, b2, b1), (1, b1, acc)):
            rc = dom.lib.wrfdc_transport_stage_adjoint(dom.ctx, rk, tr.traj.stage_ptrs(n, rk), p(out), p(acc), p(into))
            assert rc == 0
        qbar = acc
    assert torch.equal(got, qbar)
    mx, aty = tr.forward(x).double(), got.double()
    lhs, rhs = float((mx * y.double()).sum()), float((x.double() * aty).sum())
    assert abs(lhs - rhs) <= 1e-6 * float(mx.norm() * y.double().norm()), (lhs, rhs)
    ring = torch.ones(y.shape, dtype=torch.bool, device=gpu)
    ring[:shape[1], :shape[2], :shape[0]] = False
    assert (got[ring] == 0).all() and (mx[ring] == 0).all()
    dom.close()
