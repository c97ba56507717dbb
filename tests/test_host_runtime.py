"""The host side of libwrfdc on the CPU (host/host_checks.hip).

The library's source is compiled for the host alone and run over a HIP runtime written for the purpose, which can make
a chosen call fail: what the library uploads, waits for, allocates and destroys, also where a call of the runtime
fails.  No kernel runs.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.environ.get("HIPCC", os.path.join(ROCM, "bin", "hipcc"))
CHECKS = ["context_upload", "phi_tendency_blocks", "transfer_call_failures", "transfer_short_memory", "transfer_allocation_failures", "ensemble_lifecycle", "ensemble_create_failures",
          "ensemble_destroy_failures"]

pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not found")


def _build(d, *defines):
    obj, exe = str(d / "host_checks.o"), str(d / "host_checks")
    subprocess.run([HIPCC, "--offload-host-only", "--offload-arch=gfx950", "-O1", "-std=c++17", "-ffp-contract=off", *defines, "-c",
                    os.path.join(HERE, "host", "host_checks.hip"), "-o", obj], check=True, capture_output=True)
    # (the device code's image, which the host code registers, is not there)
    subprocess.run([os.path.join(ROCM, "llvm", "bin", "clang++"), obj, "-lpthread",
                    "-Wl,--unresolved-symbols=ignore-in-object-files", "-o", exe], check=True, capture_output=True)
    return exe


@pytest.fixture(scope="module")
def checks(tmp_path_factory):
    return _build(tmp_path_factory.mktemp("host"))


def _run(exe, name):
    res = subprocess.run([exe, name], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr


@pytest.mark.parametrize("name", CHECKS)
def test_host_side(checks, name):
    _run(checks, name)


@pytest.mark.parametrize("rows", [2, 8])
def test_other_face_rows(tmp_path, rows):
    _run(_build(tmp_path, f"-DWRFDC_FACE_ROWS={rows}"), "phi_tendency_blocks")
