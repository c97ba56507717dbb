"""The column kernel's two block shapes against the oracle: one step on domains on either side of the line.

Up to 256 blocks of 64 columns (ceil((nx + 1) / 64) * (ny + 1)) a block has 16 waves, beyond it 8.  Level counts on
both sides of an instantiation's range for 16 waves (32, 33, 64, 65, 96, 97 w levels).  Tolerance of the one-step
parity tests: relative L2 1e-5 per field.
"""

import pytest

from parity import REL_L2_STEP, STEP_DIAGNOSTICS, compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(14, 12, 31), (14, 12, 32), (12, 13, 63), (12, 13, 64), (12, 12, 95), (13, 12, 96),
                                      (64, 127, 6), (64, 128, 6)])
def test_step_matches_oracle(gpu, nx, ny, nz):
    from oracle import Oracle
    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    print(f"[column] {nx}x{ny}x{nz}", flush=True)
    case = make_case(nx, ny, nz, nmoist=2, hydrometeors=True, hill_height=300.0)
    dom = Domain(case.config, gpu)
    dom.upload(case.arrays)
    dom.step(1, 0.0)
    o = Oracle(case.config, case.arrays)
    o.step(1, 0.0)
    bad = compare(dom.download(), o.arrays, tol=REL_L2_STEP, skip=STEP_DIAGNOSTICS)
    o.close()
    dom.close()
    assert not bad, bad
