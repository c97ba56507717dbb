"""Species dealt over blocks of their own on small domains: one step against the oracle with one species a block,
several a block with a shorter last share, and all in one block, for both transport variants.  Tolerance of the
one-step parity tests: relative L2 1e-5 per field."""

from dataclasses import replace

import pytest

from parity import REL_L2_STEP, STEP_DIAGNOSTICS, compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pd", [False, True])
@pytest.mark.parametrize("nx,ny,nz,nmoist,nscalar", [(12, 12, 6, 1, 0), (30, 30, 30, 6, 1), (70, 33, 30, 7, 0), (130, 60, 40, 3, 2)])
def test_step_matches_oracle(gpu, nx, ny, nz, nmoist, nscalar, pd):
    from oracle import Oracle
    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    print(f"[species shares] {nx}x{ny}x{nz} {nmoist}+{nscalar} pd={pd}", flush=True)
    case = make_case(nx, ny, nz, nmoist=nmoist, nscalar=nscalar, hill_height=300.0)
    config = replace(case.config, pd_moist=int(pd), pd_scalar=int(pd))
    dom = Domain(config, gpu)
    dom.upload(case.arrays)
    dom.step(1, 5.0)
    o = Oracle(config, case.arrays)
    o.step(1, 5.0)
    bad = compare(dom.download(), o.arrays, tol=REL_L2_STEP, skip=STEP_DIAGNOSTICS)
    o.close()
    dom.close()
    assert not bad, bad
