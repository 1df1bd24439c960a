"""The C ABI's host side (page pool, metadata patches, launch order) on the
CPU: bsattn_capi.cpp linked with a stub HIP runtime and stub launchers
(tests/capi_host), so that a launch can be made to fail."""
from __future__ import annotations

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CAPI = os.path.join(HERE, "..", "mlx-swift-lm_amd", "csrc", "bsattn_capi.cpp")
ROCM = os.environ.get("ROCM", "/opt/rocm")


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    d = tmp_path_factory.mktemp("capi_host")
    out = []
    for src in (CAPI, os.path.join(HERE, "capi_host", "stubs.cpp")):
        out.append(str(d / (os.path.basename(src) + ".o")))
        subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", "-c", src, "-o",
                        out[-1]], check=True)
    return out


@pytest.mark.parametrize("program", ["failed_launch", "prefill_workspace"])
def test_capi_host(objects, tmp_path, program):
    exe = str(tmp_path / program)
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                    os.path.join(HERE, "capi_host", program + ".cpp"), *objects, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
