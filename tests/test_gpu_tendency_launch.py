"""The five RK tendencies in one launch and in five: one step against the oracle on both sides of the line (5 * 2^17
elements of a 3-D field, jde * kde * pitch: 80 and 81 rows of 64 levels at a pitch of 128) and of 2^20, with boundary
tendencies that the ring takes.  Tolerance of the one-step parity tests: relative L2 1e-5 per field."""

import numpy as np
import pytest

from parity import REL_L2_STEP, STEP_DIAGNOSTICS, compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(12, 12, 6), (127, 79, 63), (127, 80, 63), (127, 127, 63), (127, 128, 63)])
def test_step_matches_oracle(gpu, nx, ny, nz):
    from oracle import Oracle
    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    print(f"[tendencies] {nx}x{ny}x{nz}", flush=True)
    case = make_case(nx, ny, nz, nmoist=1, hill_height=300.0)
    rng = np.random.default_rng(8)
    for v in ("u", "v", "t", "ph", "qv", "mu"):
        for e in ("xs", "xe", "ys", "ye"):
            a = case.arrays[f"{v}_bt{e}"]
            a[:] = (1e-3 * rng.standard_normal(a.shape)).astype(np.float32)
    dom = Domain(case.config, gpu)
    dom.upload(case.arrays)
    dom.step(1, 5.0)
    o = Oracle(case.config, case.arrays)
    o.step(1, 5.0)
    bad = compare(dom.download(), o.arrays, tol=REL_L2_STEP, skip=STEP_DIAGNOSTICS)
    o.close()
    dom.close()
    assert not bad, bad
