"""The library's host side without a GPU (tests/host/host_checks.cpp): what it
decides, allocates, keeps and launches, with the HIP runtime stood in for."""
import os
import subprocess

import pytest

from omega_playground_amd import build as b

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "host_checks")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__",
           "-I", os.path.join(os.path.dirname(os.path.dirname(b.HIPCC)), "include"), "-I", b.CSRC,
           os.path.join(HERE, "host", "host_checks.cpp"), "-o", exe, "-rdynamic",
           "-L", b.HERE, "-lomega_swe", "-Wl,--unresolved-symbols=ignore-all", "-Wl,-rpath," + b.HERE]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    return exe


@pytest.mark.parametrize("what", ["tall", "rebuild", "keep_stepper", "keep_ensemble", "block_order",
                                  "tuned_cells", "reports", "tuning", "few_launches",
                                  "side_by_side", "one_model", "vjp_rows"])
def test_host_side(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and f"{what} ok" in r.stdout, r.stdout + r.stderr
