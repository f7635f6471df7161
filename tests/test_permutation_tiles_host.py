"""The address arithmetic of the plain permutation tiles with 16-byte vectors at any element, walked on the CPU, and the
rules that choose them."""
import os
import subprocess

import pytest

from hiptensor_amd import _lib
from hiptensor_amd import workloads as wl

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tiles_of_vectors_at_any_element(tmp_path):
    src, out = os.path.join(ROOT, "tests", "cpp", "tile_bounds.cpp"), tmp_path / "tile_bounds"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"), "-isystem", "/opt/rocm/include",
                    "-D__HIP_PLATFORM_AMD__", src, "-o", str(out), "-L" + os.path.dirname(_lib.LIB_PATH), "-lhiptensor_amd",
                    "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)], check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1].startswith("ok"), (r.stdout[-2000:], r.stderr)


@pytest.mark.parametrize("dtype,lens,perm,name", [
    ("f16", [1943, 205, 637], [2, 1, 0], "permute_tiled_f16_256x128_r8_w8_loose"),
    ("f16", [324, 350, 368], [1, 2, 0], "permute_tiled_f16_32x512_r2_w8"),  # pairs keep their own vectors
    ("f32", [946, 579, 437], [2, 1, 0], "permute_tiled_f32_64x64_r4_w4_loose"),
    ("f32", [164, 329, 609], [1, 0, 2], "permute_tiled_f32_64x64_r4_w1"),  # read whole
    ("f32", [512, 64, 128, 64], [2, 0, 3, 1], "permute_tiled_f32_128x128_r4_w4"),
    ("f32", [5128, 880], [1, 0], "permute_tiled_f32_64x64_r4_w4"),  # 64 KiB tiles would be 287
    ("f16", [692, 464], [1, 0], "permute_grouped_f16_32x64_r2_w8"),
    ("f32", [238, 117], [1, 0], "permute_gather_f32"),
    ("f16", [19, 25, 23, 8, 29], [1, 0, 4, 2, 3], "permute_gather_f16"),  # blocks transposed in place
    ("f32", [21311, 57], [1, 0], "permute_tiled_f32_64x64_r4_w4_loose"),
])
def test_choice(host_handle, dtype, lens, perm, name):
    p = wl.Permutation(host_handle, wl.permutation(dtype, lens, perm))
    got = p.info(0, 0)["kernel_name"]
    p.close()
    assert got == name


def test_tiles_that_share_lines_go_to_one_die(tmp_path):
    """tests/cpp/tile_order.cpp: matrices and blocks transposed in place, and others, with the tile order of their plan."""
    src, out = os.path.join(ROOT, "tests", "cpp", "tile_order.cpp"), tmp_path / "tile_order"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "include"), "-isystem", "/opt/rocm/include",
                    "-D__HIP_PLATFORM_AMD__", src, "-o", str(out), "-L" + os.path.dirname(_lib.LIB_PATH), "-lhiptensor_amd",
                    "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)], check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1].startswith("ok"), (r.stdout[-2000:], r.stderr)
