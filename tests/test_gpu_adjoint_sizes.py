"""The adjoint transport at the sizes where its gather can go wrong.

12x12x6 (the smallest domain: no point has only 5th-order faces around it), 65x13x8 (a second tile of one column,
tiles of both kinds) and 40x36x12.  A window of whole steps runs the stages of the one-stage entry point with the
same arithmetic: equal bit for bit.  <M x, y> = <x, M^T y> in FP64 sums of the FP32 results: each result carries a few
ulp (6e-8) per stage, and the two sums of n products of random sign differ by less than 1e-5 of the larger norm
product / sqrt(n) bound used in test_gpu_adjoint.py, here taken relative to |Mx| |y|.

A non-finite adjoint value or mass flux reaches the points whose value some flux at its cell or face reads, and no
other: the reads of a face by its order (second at faces 2 and e-1, fifth on [4, e-3], third between).
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


def _reads(f, e):
    """Cells that the flux through face f of a row of e-1 cells reads."""
    if f < 2 or f > e - 1:
        return set()
    lo, hi = (3, 2) if 4 <= f <= e - 3 else (1, 0) if f in (2, e - 1) else (2, 1)
    return set(range(f - lo, f + hi + 1))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("axis", ["x", "y"])
def test_non_finite_values_stay_with_the_fluxes_that_read_them(gpu, axis, bad):
    import torch

    from wrfdc.adjoint import Trajectory
    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    nx, ny, nz = (16, 14, 6) if axis == "x" else (14, 16, 6)
    print(f"[adjoint] {bad} along {axis} of {nx}x{ny}x{nz}", flush=True)
    case = make_case(nx, ny, nz, nmoist=1, nscalar=0, hill_height=300.0)
    dom = Domain(case.config, gpu)
    dom.upload(case.arrays)
    traj = Trajectory(dom, 1)
    flux = traj.stages[1][0 if axis == "x" else 1]
    rng = np.random.default_rng(6)
    y = torch.tensor(rng.standard_normal(case.arrays["t_2"].shape).astype(np.float32), device=gpu)
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    e, k, mid = 17, 3, 7  # faces 2 .. e-1; the row's level and its place across (1-based, an inner point)

    def at(c):
        return (mid - 1, k - 1, c - 1) if axis == "x" else (c - 1, k - 1, mid - 1)

    def spread(qbar_out):
        old, into = torch.zeros_like(y), torch.zeros_like(y)
        assert dom.lib.wrfdc_transport_stage_adjoint(dom.ctx, 2, traj.stage_ptrs(0, 2), p(qbar_out), p(old), p(into)) == 0
        a = into.isfinite().cpu().numpy()
        return {c for c in range(1, e) if not a[at(c)]}

    assert spread(y) == set()
    for c in range(2, e - 1):  # cells with a tendency
        q = y.clone()
        q[at(c)] = bad
        assert spread(q) == _reads(c, e) | _reads(c + 1, e) | {c}, c
    for f in range(2, e):
        was = flux[at(f)].clone()
        flux[at(f)] = bad
        assert spread(y) == _reads(f, e), f
        flux[at(f)] = was
    dom.close()
