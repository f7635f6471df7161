"""Host-side behaviour of hiptensorPermutation that needs no device: argument checks in the
reference's order (library/src/permutation/hiptensor_permutation.cpp:77-155, 173-189), mode
fusion and kernel choice of the planner."""
import ctypes as C
import os
import subprocess

import pytest

import perm_cases
from hiptensor_amd import _lib, api
from hiptensor_amd import workloads as wl


def _descs(h, lens, perm, dtype=api.HIP_R_32F, dtypeB=None):
    modes = list(range(100, 100 + len(lens)))
    dA = api.check(api.hiptensorInitTensorDescriptor(h, lens, None, dtype), "dA")
    dB = api.check(api.hiptensorInitTensorDescriptor(h, [lens[p] for p in perm], None, dtype if dtypeB is None else dtypeB), "dB")
    return dA, modes, dB, [modes[p] for p in perm]


def test_null_arguments_are_not_initialized(host_handle):
    dA, mA, dB, mB = _descs(host_handle, [4, 5], [1, 0])
    one = C.c_float(1.0)
    good = [host_handle, one, 256, dA, mA, 512, dB, mB]
    for i in range(len(good)):
        args = list(good)
        args[i] = None
        st = api.hiptensorPermutation(*args, api.HIP_R_32F, None)
        assert st == api.HIPTENSOR_STATUS_NOT_INITIALIZED, i


def test_type_checks_in_reference_order(host_handle):
    one = C.c_float(1.0)
    # data type other than f16 / f32: NOT_SUPPORTED, before the A/B mismatch check
    dA, mA, dB, mB = _descs(host_handle, [4, 5], [1, 0], api.HIP_R_64F, api.HIP_R_32F)
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB, mB, api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_NOT_SUPPORTED
    dA, mA, dB, mB = _descs(host_handle, [4, 5], [1, 0], api.HIP_R_16BF)
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB, mB, api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_NOT_SUPPORTED
    # A and B of different types: INVALID_VALUE
    dA, mA, dB, mB = _descs(host_handle, [4, 5], [1, 0], api.HIP_R_32F, api.HIP_R_16F)
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB, mB, api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_INVALID_VALUE
    # scalar type other than f16 / f32: NOT_SUPPORTED
    dA, mA, dB, mB = _descs(host_handle, [4, 5], [1, 0])
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB, mB, api.HIP_R_64F, None) == api.HIPTENSOR_STATUS_NOT_SUPPORTED


@pytest.mark.parametrize("lens", [[7], [2, 2, 2, 2, 2, 2, 2]])
def test_ranks_without_an_instance_report_internal_error(host_handle, lens):
    dA, mA, dB, mB = _descs(host_handle, lens, list(range(len(lens))))
    st = api.hiptensorPermutation(host_handle, C.c_float(1.0), 256, dA, mA, 512, dB, mB, api.HIP_R_32F, None)
    assert st == api.HIPTENSOR_STATUS_INTERNAL_ERROR


def test_inconsistent_modes_or_lengths_are_invalid(host_handle):
    one = C.c_float(1.0)
    dA, mA, dB, mB = _descs(host_handle, [4, 5, 6], [2, 0, 1])
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB, [mB[0], mB[1], 999], api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_INVALID_VALUE
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB, [mB[0], mB[0], mB[2]], api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_INVALID_VALUE
    # lengths of B not those of A's modes
    dB2 = api.check(api.hiptensorInitTensorDescriptor(host_handle, [6, 4, 7], None, api.HIP_R_32F), "dB2")
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB2, mB, api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_INVALID_VALUE
    # different rank
    dB3 = api.check(api.hiptensorInitTensorDescriptor(host_handle, [6, 4], None, api.HIP_R_32F), "dB3")
    assert api.hiptensorPermutation(host_handle, one, 256, dA, mA, 512, dB3, mB[:2], api.HIP_R_32F, None) == api.HIPTENSOR_STATUS_INVALID_VALUE


def test_too_many_elements_not_supported(host_handle):
    dA, mA, dB, mB = _descs(host_handle, [1 << 16, 1 << 15], [1, 0])
    assert api.permutationInfo(dA, mA, dB, mB)[0] == api.HIPTENSOR_STATUS_NOT_SUPPORTED


def test_a_handle_without_device_refuses_to_execute(host_handle):
    dA, mA, dB, mB = _descs(host_handle, [4, 5], [1, 0])
    st = api.hiptensorPermutation(host_handle, C.c_float(1.0), 256, dA, mA, 512, dB, mB, api.HIP_R_32F, None)
    assert st == api.HIPTENSOR_STATUS_ARCH_MISMATCH


def _info(h, dtype, lens, perm, A=0, B=0):
    p = wl.Permutation(h, wl.permutation(dtype, lens, perm))
    out = p.info(A, B)
    p.close()
    return out


def test_fusion_and_kernel_choice(host_handle):
    h = host_handle
    # identity order: everything fuses, vector copy
    i = _info(h, "f32", [64, 64, 64], [0, 1, 2])
    assert (i["fused_rank"], i["kernel"], i["vec_r"], i["extent"]) == (1, api.PERM_COPY, 4, [64 ** 3])
    # extent-1 modes vanish, neighbours that stay neighbours fuse
    i = _info(h, "f32", [8, 1, 16, 32, 64], [3, 4, 0, 1, 2])
    assert i["fused_rank"] == 2 and i["extent"] == [8 * 16, 32 * 64] and i["b_stride"] == [32 * 64, 1]
    assert i["kernel"] == api.PERM_TILED and (i["mode_i"], i["mode_j"]) == (0, 1) and (i["vec_r"], i["vec_w"]) == (4, 4)
    # the sample program's shape: 33 is odd, so loads are scalar; stores run along 34 * 35
    i = _info(h, "f32", [33, 32, 34, 35], [2, 3, 1, 0])
    assert i["kernel"] == api.PERM_GROUPED and i["extent"] == [33, 32, 34 * 35] and (i["vec_r"], i["vec_w"]) == (1, 2)
    assert i["kernel_name"] == "permute_grouped_f32_33x64_r1_w2"  # a small tensor: tiles shrunk until 512 workgroups
    # shared fastest mode
    i = _info(h, "f16", [512, 24, 96], [0, 2, 1])
    assert i["kernel"] == api.PERM_ROWS and i["vec_r"] == i["vec_w"] == 8 and i["mode_j"] == 2
    # ... a short one (interleaved channels): tiles of it times chunks of A's and B's next modes
    i = _info(h, "f32", [4, 512, 512, 8], [0, 2, 1, 3])
    assert i["kernel"] == api.PERM_SHARED and i["kernel_name"] == "permute_shared_f32_4x32x32_v4"
    # short fastest mode, tiny tensors: one thread per element
    assert _info(h, "f32", [3, 5, 7, 9, 11], [0, 4, 2, 3, 1])["kernel"] == api.PERM_GATHER
    assert _info(h, "f32", [5, 2, 3, 4], [3, 2, 1, 0])["kernel"] == api.PERM_GATHER
    # a short tile mode whose partner follows it in memory: strips
    i = _info(h, "f32", [512, 512, 3, 16], [2, 0, 1, 3])
    assert i["kernel"] == api.PERM_STRIP and i["tile"] == 0 and i["extent"][:2] == [512 * 512, 3] and (i["vec_r"], i["vec_w"]) == (4, 4)
    i = _info(h, "f16", [3, 512, 512, 16], [1, 2, 0, 3])
    assert i["kernel"] == api.PERM_STRIP and i["tile"] == 1 and (i["vec_r"], i["vec_w"]) == (8, 8)
    # ... when the partner is elsewhere in memory, grouped tiles take B's next mode along instead
    i = _info(h, "f32", [512, 3, 512, 16], [1, 3, 0, 2])
    assert i["kernel"] == api.PERM_GROUPED and i["kernel_name"] == "permute_grouped_f32_128x48_r4_w1"
    # many short modes: rows span A's two fastest modes, columns B's two fastest
    i = _info(h, "f32", [16] * 6, [5, 4, 3, 2, 1, 0])
    assert i["kernel"] == api.PERM_GROUPED and i["kernel_name"] == "permute_grouped_f32_112x112_r4_w4"
    assert _info(h, "f16", [16] * 6, [5, 4, 3, 2, 1, 0])["kernel_name"] == "permute_grouped_f16_128x128_r8_w8"
    # all extents one
    i = _info(h, "f16", [1, 1, 1], [2, 0, 1])
    assert (i["fused_rank"], i["kernel"], i["extent"]) == (1, api.PERM_COPY, [1])
    # a zero extent: nothing to launch
    assert _info(h, "f32", [4, 0, 3], [2, 0, 1])["empty"] == 1


def test_vector_width_follows_pointer_alignment(host_handle):
    h = host_handle
    assert _info(h, "f32", [256, 192], [1, 0], A=0x1000, B=0x2000)["vec_r"] == 4
    i = _info(h, "f32", [256, 192], [1, 0], A=0x1008, B=0x2004)
    assert (i["vec_r"], i["vec_w"]) == (2, 1)
    i = _info(h, "f16", [256, 192], [1, 0], A=0x1004, B=0x2010)
    assert (i["vec_r"], i["vec_w"]) == (2, 8)
    assert _info(h, "f16", [64, 64, 64], [0, 1, 2], A=0x1008, B=0x2000)["vec_r"] == 4


@pytest.mark.parametrize("dtype,lens,perm,name", [
    # pairs of f16 on large tensors: the extents' own vectors (16-byte ones at any element are up to 1.5x slower there)
    ("f16", [138, 16, 70, 18, 82], [2, 1, 4, 0, 3], "permute_grouped_f16_128x70_r2_w2"),
    ("f16", [72, 52, 312, 36], [3, 2, 0, 1], "permute_grouped_f16_128x108_r8_w2"),
    ("f16", [100, 16, 12, 48, 16, 8], [3, 5, 2, 0, 4, 1], "permute_grouped_f16_100x96_r2_w8"),
    ("f16", [638, 52, 95, 51], [3, 2, 1, 0], "permute_grouped_f16_128x102_r2_w1"),
    # ... smaller tensors, single elements and f32: 16-byte vectors at any element
    ("f16", [154, 68, 562], [1, 0, 2], "permute_grouped_f16_128x68_r8_w8_loose"),
    ("f16", [21, 25, 23, 57, 25], [4, 2, 1, 3, 0], "permute_grouped_f16_126x125_r8_w8_loose"),
    ("f16", [7, 32, 32, 32, 16, 8], [5, 4, 1, 3, 2, 0], "permute_grouped_f16_126x128_r8_w8_loose"),
    ("f16", [19, 11, 13, 33, 12, 23], [4, 2, 0, 3, 5, 1], "permute_grouped_f16_114x120_r8_w8_loose"),
    ("f32", [154, 252, 240, 26], [3, 1, 2, 0], "permute_grouped_f32_128x104_r4_w4_loose"),
])
def test_vectors_at_any_element_where_they_gain(host_handle, dtype, lens, perm, name):
    assert _info(host_handle, dtype, lens, perm)["kernel_name"] == name


@pytest.mark.parametrize("dtype,lens,perm,name", [
    # a few MB: one vector per thread, so that there are workgroups enough (32.8.16.40: 160 and not 40)
    ("f32", [32, 8, 16, 40], [0, 3, 2, 1], "permute_runs_f32_32_v4x1"),
    ("f32", [55, 50, 16, 9], [0, 2, 1, 3], "permute_runs_f32_55_v4x1"),
    ("f16", [41, 326, 156], [0, 2, 1], "permute_runs_f16_41_v8x1"),
    # the line: 2^20 vectors
    ("f32", [64, 256, 255], [0, 2, 1], "permute_runs_f32_64_v4x1"),
    ("f32", [63, 256, 261], [0, 2, 1], "permute_runs_f32_63_v4x4"),
    ("f16", [127, 256, 258], [0, 2, 1], "permute_runs_f16_127_v8x1"),
    ("f16", [127, 256, 259], [0, 2, 1], "permute_runs_f16_127_v8x4"),
])
def test_linear_kernel_spreads_small_tensors(host_handle, dtype, lens, perm, name):
    p = wl.Permutation(host_handle, wl.permutation(dtype, lens, perm))
    with _Runs():
        assert p.info()["kernel_name"] == name
    p.close()


@pytest.mark.parametrize("dtype,lens,perm,name", [
    # the runs of a shared fastest mode that square tiles cut: linear on mid-sized tensors ...
    ("f32", [128, 128, 512], [0, 2, 1], "permute_runs_f32_128_v4x4"),
    ("f16", [256, 128, 2048], [0, 2, 1], "permute_runs_f16_256_v8x4"),
    # ... and on the largest, if the next runs lie near in A
    ("f32", [128, 64, 128, 200], [0, 2, 1, 3], "permute_runs_f32_128_v4x4"),
    ("f16", [256, 64, 128, 256], [0, 2, 1, 3], "permute_runs_f16_256_v8x4"),
    # ... and on any where the run is no whole number of 128-byte lines
    ("f32", [1140, 228, 824], [0, 2, 1], "permute_runs_f32_1140_v4x4"),
    ("f32", [396, 13, 21, 15, 63], [0, 4, 3, 2, 1], "permute_runs_f32_396_v4x4"),
    ("f16", [1032, 191, 1182], [0, 2, 1], "permute_runs_f16_1032_v8x4"),
    ("f32", [132, 134, 300, 42], [0, 3, 2, 1], "permute_runs_f32_132_v4x4"),
    # tiles where the linear walk loses locality
    ("f32", [192, 128, 2730], [0, 2, 1], "permute_rows_f32_64x64_r4_w4"),
    ("f32", [128, 32, 16, 2048], [0, 3, 2, 1], "permute_rows_f32_64x64_r4_w4"),
    ("f32", [128, 16, 1024, 64], [0, 3, 2, 1], "permute_rows_f32_64x64_r4_w4"),
    ("f16", [256, 32, 16, 2048], [0, 3, 2, 1], "permute_rows_f16_128x128_r8_w8"),
    ("f16", [256, 32, 1024, 32], [0, 3, 2, 1], "permute_rows_f16_512x32_r8_w8"),
    # half of a long tile inside: linear on smaller tensors
    ("f32", [128, 8, 16, 64], [0, 2, 1, 3], "permute_runs_f32_128_v4x1"),
    ("f32", [128, 128, 16, 1024], [0, 2, 1, 3], "permute_rows_f32_256x16_r4_w4"),
    ("f16", [256, 16, 512, 32], [0, 3, 2, 1], "permute_runs_f16_256_v8x4"),
])
def test_linear_kernel_or_row_tiles(host_handle, dtype, lens, perm, name):
    assert _info(host_handle, dtype, lens, perm)["kernel_name"] == name


class _Runs:
    """The linear kernel wherever the layout admits it, for the duration of a block."""

    def __enter__(self):
        os.environ["HIPTENSOR_AMD_PERMUTE"] = "runs"

    def __exit__(self, *a):
        del os.environ["HIPTENSOR_AMD_PERMUTE"]


def test_every_validation_case_plans(host_handle):
    for rank in (2, 3, 4, 5, 6):
        for w in perm_cases.validation(rank, thin=36):
            p = wl.Permutation(host_handle, w)
            i = p.info()
            p.close()
            assert i["kernel_name"], w["name"]


def test_vectors_at_any_element_stay_inside(tmp_path):
    """tests/cpp/perm_bounds.cpp: every load and store of the kernels that move 16-byte vectors at any element, walked on
    the host with the planner's own choices and the kernels' own address functions (kernels/perm_addr.hpp)."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, out = os.path.join(root, "tests", "cpp", "perm_bounds.cpp"), tmp_path / "perm_bounds"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(root, "include"), src, "-o", str(out),
                    "-L" + os.path.dirname(_lib.LIB_PATH), "-lhiptensor_amd", "-Wl,-rpath," + os.path.dirname(_lib.LIB_PATH)],
                   check=True, capture_output=True)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().splitlines()[-1] == "ok", (r.stdout[-2000:], r.stderr)
