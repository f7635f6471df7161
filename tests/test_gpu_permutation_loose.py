"""GPU parity of the grouped permutation tiles with 16-byte vectors at any element: odd extents on both sides, tiles at the edges whose
runs are shorter than a vector (down to one element) or a little longer, row and column chunks that do not divide their modes,
bases off their alignment."""
import pytest

import gpu_util
import perm_cases
from hiptensor_amd import workloads as wl
from test_gpu_permutation import _Override, _same

pytestmark = pytest.mark.gpu

# 129 = 128 + 1, 131 = 128 + 3, 137 = 128 + 9: the second tile's run is 1, 3 or 9 elements
SHAPES = [
    ([129, 150, 131], [2, 1, 0]), ([131, 129, 200], [1, 0, 2]), ([137, 171, 129], [2, 1, 0]), ([67, 305, 129], [2, 1, 0]),
    ([21, 25, 23, 31, 25], [4, 2, 1, 3, 0]), ([19, 7, 49, 9, 57], [3, 4, 2, 1, 0]), ([65, 513, 129], [1, 2, 0]),
    ([13, 11, 7, 9, 15, 35], [4, 2, 3, 0, 5, 1]),
]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("shift", [(0, 0), (1, 3)])
def test_loose_tiles(gpu_handle, oracle_mod, dtype, shift):
    used = 0
    with _Override("grouped"):
        for n, (lens, perm) in enumerate(SHAPES):
            w = wl.permutation(dtype, lens, perm, 1.7, dtype, *perm_cases.OPS[n % 4])
            A = wl.permutation_input(w)
            print(f"[case] {dtype} {lens} {perm} shift {shift}", flush=True)
            got, info = gpu_util.run_gpu_permutation(gpu_handle, w, A, a_shift=shift[0], b_shift=shift[1], return_info=True)
            used += info["kernel_name"].endswith("_loose")
            assert _same(got, oracle_mod.permute(w, A)), (lens, perm, shift, info["kernel_name"])
    assert used == len(SHAPES)


# (a side of 1 or 3 elements, several tiles along either mode, a batch mode)
TILE_SHAPES = [([129, 150, 3], [1, 0, 2]), ([131, 5, 129], [2, 1, 0]), ([257, 515], [1, 0]), ([40, 300, 7], [1, 2, 0]), ([300, 41], [1, 0]),
               ([70, 2, 513], [2, 0, 1]), ([19, 25, 8], [1, 0, 2]), ([515, 33, 5], [1, 2, 0]), ([1025, 17, 2], [1, 0, 2])]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("tile", [0, 1, 2, 3])
def test_plain_tiles_at_any_element(gpu_handle, oracle_mod, dtype, tile):
    for group in (0, 16):
        with _Override(f"loose,{tile},8,{group}"):
            for n, (lens, perm) in enumerate(TILE_SHAPES):
                for shift in ((0, 0), (1, 3)):
                    w = wl.permutation(dtype, lens, perm, 1.7, dtype, *perm_cases.OPS[n % 4])
                    A = wl.permutation_input(w)
                    print(f"[case] {dtype} {lens} {perm} tile {tile} group {group} shift {shift}", flush=True)
                    got, info = gpu_util.run_gpu_permutation(gpu_handle, w, A, a_shift=shift[0], b_shift=shift[1], return_info=True)
                    assert info["kernel_name"].startswith("permute_tiled") and info["kernel_name"].endswith("_loose"), info["kernel_name"]
                    assert _same(got, oracle_mod.permute(w, A)), (lens, perm, shift, info["kernel_name"])


@pytest.mark.parametrize("dtype,lens,perm", [("f16", [411, 163, 157], [2, 1, 0]), ("f32", [946, 57, 237], [2, 1, 0]), ("f32", [205, 33, 279, 9], [2, 1, 0, 3]),
                                             ("f32", [23, 20, 14, 13, 18, 11], [3, 2, 5, 0, 4, 1]), ("f16", [52, 41, 77, 103], [1, 0, 3, 2]),
                                             ("f32", [7, 501, 77, 97], [0, 2, 1, 3]), ("f32", [77, 207, 1099], [1, 2, 0])])
def test_runs_that_share_lines(gpu_handle, oracle_mod, dtype, lens, perm):
    """Large tensors whose runs of B start anywhere: neighbouring tiles on one die, ordinary stores."""
    w = wl.permutation(dtype, lens, perm, 1.7, dtype)
    A = wl.permutation_input(w)
    print(f"[case] {dtype} {lens} {perm}", flush=True)
    got, info = gpu_util.run_gpu_permutation(gpu_handle, w, A, return_info=True)
    assert _same(got, oracle_mod.permute(w, A)), info["kernel_name"]
