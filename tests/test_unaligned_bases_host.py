"""What a plan runs where an operand's base is not aligned for its tile, and the workspace recommended for it."""
import os
import subprocess

import pytest

import cases
from hiptensor_amd import _lib
from hiptensor_amd import workloads as wl

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_best_staged_tile_stands_in(tmp_path):
    """tests/cpp/unaligned_bases.cpp: every direct-load choice of a list of problems, with the kernels looked up at addresses
    off its alignment."""
    src, out = os.path.join(ROOT, "tests", "cpp", "unaligned_bases.cpp"), tmp_path / "unaligned_bases"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"), "-isystem", "/opt/rocm/include",
                    "-D__HIP_PLATFORM_AMD__", src, "-o", str(out), "-L" + os.path.dirname(_lib.LIB_PATH), "-lhiptensor_amd",
                    "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)], check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1].startswith("ok"), (r.stdout[-2000:], r.stderr)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_recommended_workspace_covers_operands_declared_off_the_tiles_alignment(host_handle, dtype):
    """160 x 768 x 1152 runs a direct-load tile in one pass; operands declared at 2 bytes run staged tiles in slices."""
    w = wl.make_workload(dtype, cases.COMPUTE[dtype], [0, 20], [10, 20], [0, 10], {0: 160, 10: 768, 20: 1152}, 1.5, None, name=f"declared_{dtype}")
    sizes = {}
    for align in (16, 4, 2):
        c = wl.Contraction(host_handle, w, align=align)
        sizes[align] = c.workspace_bytes, c.info["workspace_bytes"], c.info["kernel_name"]
        c.close()
    assert sizes[16] == sizes[4] and "direct" in sizes[16][2] and sizes[16][0] == sizes[16][1], sizes
    assert sizes[2][1:] == sizes[16][1:] and sizes[2][0] % (160 * 768 * 4) == 0 and sizes[2][0] >= 2 * 160 * 768 * 4, sizes
