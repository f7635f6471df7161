"""GPU parity of the linear permutation (a shared fastest mode, B written in 16-byte vectors): runs of exactly a vector, of a vector
and a few elements more, long odd ones; vectors that span two runs, at the front and at the end of A among them; element counts that are no multiple of
the vector; bases off their alignment; both forms of the element operation."""
import pytest

import gpu_util
import perm_cases
from hiptensor_amd import workloads as wl
from test_gpu_permutation import _Override, _same

pytestmark = pytest.mark.gpu

# (extents, order): B's second run is A's last, A's first, a middle one; rank 2 to 6; more than one workgroup of vectors
SHAPES = [
    ([4, 2, 3], [0, 2, 1]), ([8, 3, 2], [0, 2, 1]), ([9, 2, 2], [0, 2, 1]), ([11, 7, 5], [0, 2, 1]), ([15, 2, 3, 4], [0, 3, 2, 1]),
    ([17, 3, 5, 2, 4], [0, 4, 2, 3, 1]), ([30, 7, 11, 7, 3, 5], [0, 4, 2, 3, 1, 5]), ([41, 61, 13], [0, 2, 1]),
    ([229, 6, 5, 7], [0, 3, 2, 1]), ([1659, 20, 3, 2], [0, 2, 3, 1]), ([64, 33, 9], [0, 2, 1]), ([4099, 2, 3], [0, 2, 1]),
]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("shift", [(0, 0), (1, 0), (0, 3), (3, 1)])
def test_runs(gpu_handle, oracle_mod, dtype, shift):
    used = 0
    with _Override("runs"):
        for n, (lens, perm) in enumerate(SHAPES):
            w = wl.permutation(dtype, lens, perm, 1.7, dtype, *perm_cases.OPS[n % 4])
            A = wl.permutation_input(w)
            print(f"[case] {dtype} {lens} {perm} shift {shift}", flush=True)
            got, info = gpu_util.run_gpu_permutation(gpu_handle, w, A, a_shift=shift[0], b_shift=shift[1], return_info=True)
            used += info["kernel_name"].startswith("permute_runs")
            assert _same(got, oracle_mod.permute(w, A)), (lens, perm, shift, info["kernel_name"])
    assert used == sum(lens[0] * wl.ELEM_BYTES[dtype] >= 16 for lens, _ in SHAPES)


@pytest.mark.parametrize("dtype,lens", [("f32", [63, 256, 261]), ("f16", [127, 256, 259])])
@pytest.mark.parametrize("shift", [(0, 0), (1, 3)])
def test_four_vectors_a_thread(gpu_handle, oracle_mod, dtype, lens, shift):
    """Just over the line from which a thread moves four vectors; the last workgroup holds few."""
    w = wl.permutation(dtype, lens, [0, 2, 1], 1.7, dtype, *perm_cases.OPS[0])
    A = wl.permutation_input(w)
    print(f"[case] {dtype} {lens} shift {shift}", flush=True)
    with _Override("runs"):
        got, info = gpu_util.run_gpu_permutation(gpu_handle, w, A, a_shift=shift[0], b_shift=shift[1], return_info=True)
    assert info["kernel_name"].endswith("x4"), info["kernel_name"]
    assert _same(got, oracle_mod.permute(w, A))


@pytest.mark.parametrize("dtype,lens,perm", [("f32", [30, 7, 61, 7, 7, 13], [0, 4, 2, 3, 1, 5]), ("f16", [229, 60, 25, 4], [0, 3, 2, 1]),
                                             ("f32", [128, 32, 48, 24], [0, 2, 1, 3])])
def test_default_choice(gpu_handle, oracle_mod, dtype, lens, perm):
    w = wl.permutation(dtype, lens, perm, -0.75, dtype, *perm_cases.OPS[0])
    A = wl.permutation_input(w)
    got, info = gpu_util.run_gpu_permutation(gpu_handle, w, A, return_info=True)
    assert info["kernel_name"].startswith("permute_runs"), info["kernel_name"]
    assert _same(got, oracle_mod.permute(w, A))
