"""The host layer's large blocking calls (panels of rows, helper threads) without a GPU: rk_core.cpp, rk_w4a8.cpp and
rk_quant_matmul.cpp compiled with host_calls_cpu.cpp, which takes the place of the HIP side."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rknpu2_matmul_open_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host_calls") / "host_calls"
    sources = [os.path.join(CSRC, f) for f in ("rk_core.cpp", "rk_w4a8.cpp", "rk_quant_matmul.cpp")]
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-rdynamic", "-I" + CSRC, "-I" + os.path.join(ROOT, "include"), "-o", str(exe),
                           os.path.join(ROOT, "tests", "host_calls_cpu.cpp")] + sources +
                          ["-Wl,--unresolved-symbols=ignore-all,-z,lazy", "-lpthread", "-ldl"])  # (what no checked call reaches)
    return str(exe)


@pytest.mark.parametrize("check", ["rejected_before", "own_work_only", "out_of_memory", "helpers", "panelled"])
def test_blocking_calls(program, check):
    done = subprocess.run([program, check], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert done.returncode == 0, done.stdout
