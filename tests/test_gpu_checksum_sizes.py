"""Checksums at the sizes where the column walk can go wrong, against NumPy in FP64.

One short tile, a tile that ends on column 64 and one that goes past it, runs of one level; then enough columns for
runs of 2 for the state and 3 for the species, of 5 and 9, and of 16 with one level left over.  The sums are FP64 of
the same FP32 values: the order of at most 1e6 terms and a few roundings per term give 1e-12 relative.  A non-finite pressure must show in the energy and nowhere else, a non-finite wind in the count.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _numpy(case):
    cfg, A = case.config, {k: v.astype(np.float64) for k, v in case.arrays.items()}
    nx, ny, nz = cfg.nx, cfg.ny, cfg.nz
    f = {n: float(np.float32(getattr(cfg, n))) for n in ("dx", "dy", "g", "r_d", "cpovcv", "t0", "p0")}

    def at(n, dj=0, dk=0, di=0):
        return A[n][dj:ny + dj, dk:nz + dk, di:nx + di]

    mt = (A["mu_2"] + A["mub"])[:ny, None, :nx]
    c1, c2, dnw = (A[n][:nz][None, :, None] for n in ("c1h", "c2h", "dnw"))
    dm = (c1 * mt + c2) * -dnw * f["dx"] * f["dy"] / f["g"] / (A["msftx"] * A["msfty"])[:ny, None, :nx]
    kin = (at("u_2") + at("u_2", di=1)) ** 2 + (at("v_2") + at("v_2", dj=1)) ** 2 + (at("w_2") + at("w_2", dk=1)) ** 2
    temp = (f["t0"] + at("t_2")) * ((at("p") + at("pb")) / f["p0"]) ** (1.0 - 1.0 / f["cpovcv"])
    phi = 0.5 * (at("ph_2") + at("phb") + at("ph_2", dk=1) + at("phb", dk=1))
    energy = (dm * (0.125 * kin + f["r_d"] / (f["cpovcv"] - 1.0) * temp + phi)).sum()
    return [mt.sum(), at("t_2").sum(), A["moist"][:, :ny, :nz, :nx].sum(), 0.0, dm.sum(), energy]


@pytest.mark.parametrize("nx,ny,nz", [(12, 12, 6), (64, 13, 16), (65, 12, 17), (65, 130, 17), (129, 330, 18), (12, 640, 97)])
def test_sums_match_numpy(gpu, nx, ny, nz):
    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    print(f"[checksums] {nx}x{ny}x{nz}", flush=True)
    case = make_case(nx, ny, nz, nmoist=2, hydrometeors=True)
    case.arrays["msftx"][:] = 1.05
    case.arrays["w_2"][:] += 0.25
    dom = Domain(case.config, gpu)
    dom.upload(case.arrays)
    np.testing.assert_allclose(dom.checksums(), _numpy(case), rtol=1e-12)
    dom.buffers["p"][ny - 1, nz - 1, nx - 1] = float("inf")
    assert dom.checksums()[5] == np.inf and dom.checksums()[3] == 0
    dom.buffers["p"][ny - 1, nz - 1, nx - 1] = -3e5
    assert np.isnan(dom.checksums()[5])
    dom.buffers["u_2"][0, 0, 0] = float("nan")
    with pytest.raises(FloatingPointError):
        dom.checksums()
    dom.close()
