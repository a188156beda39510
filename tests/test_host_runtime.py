"""Host code of libcismgpu.so without a device: the library is loaded by a
program that stands in for the HIP runtime on host memory and launches no
kernels (tests/native).  Allocation and copy failures, and the route that a
call takes, can be looked at this way."""
import os
import subprocess

import pytest

from cism_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="session")
def host_checks(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("native") / "host_checks")
    subprocess.run(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-o", exe,
                    os.path.join(ROOT, "tests", "native", "host_checks.cpp"), "-ldl", "-lpthread"], check=True)
    return exe


CHECKS = ["reassembly_out_of_memory", "reassembly_failed_copy", "zero_store_no_ice", "zero_store_outflow",
          "one_product_per_solve", "level_shares_thin", "level_shares_deep", "level_shares_small",
          "large_copies", "large_copies_no_heap", "large_copies_no_pinned"]


@pytest.mark.parametrize("check", CHECKS)
def test_host(host_checks, check):
    if not os.path.exists(build.LIB):
        build.build()
    env = {k: v for k, v in os.environ.items() if not k.startswith("CISMGPU_")}
    r = subprocess.run([host_checks, build.LIB, check], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"{r.returncode}\n{r.stdout}{r.stderr}"
