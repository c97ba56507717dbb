"""Reference-layout transfers turned on the device, against to_registry / from_registry: equal bit for bit.

Every field kind at odd sizes; arrays larger than a transfer chunk (the 7-slot moist stack of 150x90x33 is 13 MB,
the chunk 8 MB); arrays that are not contiguous or not float32, and shapes the host rules accept by broadcasting.
"""

import numpy as np
import pytest

from wrfdc.fields import FIELD_SPECS

pytestmark = pytest.mark.gpu


def _domain(gpu, nx, ny, nz, nmoist, nscalar):
    from dataclasses import replace

    from wrfdc.cases import make_case
    from wrfdc.device import Domain

    cfg = make_case(12, 12, 6, nmoist=nmoist, nscalar=nscalar).config
    dom = Domain(replace(cfg, nx=nx, ny=ny, nz=nz, ip=(nx + 16) // 16 * 16), gpu)
    return dom, dom.dims


@pytest.mark.parametrize("shape", [(13, 17, 7, 3, 2), (31, 12, 6, 1, 0), (150, 90, 33, 6, 1)])
def test_both_ways_match_the_host_conversion(gpu, shape):
    from wrfdc.step_em import from_registry, get_reference, put_reference, reference_shape, to_registry

    print(f"[layout] {shape}", flush=True)
    dom, d = _domain(gpu, *shape)
    rng = np.random.default_rng(4)
    refs = {n: rng.standard_normal(reference_shape(n, d)).astype(np.float32) for n, _ in FIELD_SPECS}
    for t in dom.buffers.values():
        t.fill_(-7.0)  # the pad columns must be cleared too
    put_reference(dom, d, refs)
    got = dom.download()
    for name, _ in FIELD_SPECS:
        np.testing.assert_array_equal(got[name], to_registry(name, refs[name], d), err_msg=name)
    back = get_reference(dom, d, [n for n, _ in FIELD_SPECS])
    for name, _ in FIELD_SPECS:
        np.testing.assert_array_equal(back[name], from_registry(name, got[name], d), err_msg=name)
    dom.close()


def test_other_types_strides_and_shapes(gpu):
    from wrfdc.step_em import put_reference, reference_shape, to_registry

    dom, d = _domain(gpu, 13, 17, 7, 2, 0)
    rng = np.random.default_rng(5)
    u = rng.standard_normal(reference_shape("u_2", d))  # float64
    v = np.asfortranarray(rng.standard_normal(reference_shape("v_2", d)).astype(np.float32))
    refs = {"u_2": u, "v_2": v, "t_2": np.float32(rng.standard_normal((1, d.kde, 1))), "znu": np.arange(2.0 * d.kde),
            "mu_2": rng.integers(0, 9, reference_shape("mu_2", d)),
            "moist": rng.standard_normal((d.ide, d.kde, d.jde, 5)).astype(np.float32)}
    put_reference(dom, d, refs)
    got = dom.download(list(refs))
    for name, a in refs.items():
        np.testing.assert_array_equal(got[name], to_registry(name, a, d), err_msg=name)
    with pytest.raises(ValueError):
        put_reference(dom, d, {"w_2": np.zeros((3, 4, 5), np.float32)})
    dom.close()
