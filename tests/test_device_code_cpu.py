"""What the compiler made of the large-tile GEMM's kernels, read back from the built library: costs that no result shows
and that come and go with small changes of the source or of the compiler."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from rknpu2_matmul_open_amd import build

TOOLS = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    """The library's device code objects, one per source file."""
    dump = os.path.join(TOOLS, "llvm-objdump")
    if not os.path.exists(dump) or not os.path.exists(build.LIB):
        pytest.skip("needs the built library and llvm-objdump")
    where = tmp_path_factory.mktemp("code")
    lib = shutil.copy(build.LIB, where)
    subprocess.run([dump, "--offloading", lib], check=True, stdout=subprocess.DEVNULL, cwd=where)
    return sorted(glob.glob(lib + ".*gfx950"))


@pytest.fixture(scope="module")
def gemm_kernels(code_objects):
    """Mangled name -> instructions of every kernel of rk_kernels_gemm.hip."""
    for obj in code_objects:
        notes = subprocess.run([os.path.join(TOOLS, "llvm-readelf"), "--notes", obj], check=True, capture_output=True, text=True).stdout
        if "gemm_wk_kernel" in notes:
            text = subprocess.run([os.path.join(TOOLS, "llvm-objdump"), "-d", "--no-show-raw-insn", obj], check=True, capture_output=True, text=True).stdout
            parts = re.split(r"^[0-9a-f]+ <(\w+)>:\n", text, flags=re.M)
            return dict(zip(parts[1::2], parts[2::2]))
    raise AssertionError("no code object holds gemm_wk_kernel")


def test_k_halves_meet_without_a_select_per_accumulator(gemm_kernels):
    """Which rows a wave hands over depends on its k-half, a branch.  Made one piece of code by the compiler, with vector
    selects of every accumulator, it cost a tile of 128 x 256 close to a microsecond."""
    checked = 0
    for name, text in gemm_kernels.items():
        m = re.search(r"gemm_wk_kernelILi(\d)ELb[01]ELi\dELi(\d)ELb0E", name)
        if m:
            accumulators = 16 * int(m.group(1)) * int(m.group(2))
            assert text.count("v_cndmask") < accumulators / 2, name
            checked += 1
    assert checked >= 20


def test_the_reduce_launch_has_a_parts_loads_in_flight_together(gemm_kernels):
    """A wave adds up to 32 rows x 64 columns of each part of K: eight loads per 32 rows, none of which waits for another."""
    checked = 0
    for name, text in gemm_kernels.items():
        m = re.search(r"gemm_wk_reduce_kernelILi(\d)E", name)
        if m:
            up_to_wait = text[text.index("global_load_dwordx4"):].split("vmcnt")[0]
            assert up_to_wait.count("global_load_dwordx4") == 4 * min(int(m.group(1)), 2), name
            checked += 1
    assert checked >= 15


def test_no_large_tile_kernel_keeps_registers_in_memory(code_objects):
    """Registers spilled to scratch memory are loads and stores that wait among those of the loop's own."""
    checked = 0
    for obj in code_objects:
        notes = subprocess.run([os.path.join(TOOLS, "llvm-readelf"), "--notes", obj], check=True, capture_output=True, text=True).stdout
        for entry in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\w+)", entry).group(1)
            if "gemm_wk_" in name:
                assert int(re.search(r"\.private_segment_fixed_size: (\d+)", entry).group(1)) == 0, name
                checked += 1
    assert checked >= 39
