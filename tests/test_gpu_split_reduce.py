"""GPU parity of the split-K reduction at the sizes where it changes form: outputs that are no multiple of the 16 bytes a
thread owns where there are many (the last vector is loaded from inside the slice and moved to the front), rows of D
that end inside a vector, few and many slices (dealt to one or to several threads per output), C / D offsets computed or from
tables, with and without C."""
import os

import pytest

import cases
import gpu_util
from hiptensor_amd import api
from hiptensor_amd import workloads as wl

pytestmark = pytest.mark.gpu

# a small tile of the class per gather: 16-byte vectors, scalars
TILES = {"f16": (2, 4), "bf16": (2, 4), "f32": (1,), "f64": (1,), "c32": (1,), "c64": (1,)}
# (M modes, N modes): 1, 3, 63, 8 710 and 526 275 outputs (the last: 16 bytes of outputs a thread)
OUTPUTS = [((1,), (1,)), ((1,), (3,)), ((7,), (9,)), ((13, 10), (67,)), ((29, 25), (726,))]


def _run(handle, w, inp, split, d_alias_c=False):
    """On the first of the class's small tiles that takes the layout."""
    for tile in TILES[w["dtype"]]:
        os.environ["HIPTENSOR_AMD_FORCE_KERNEL"] = f"{tile},{split}"
        print(f"[case] {w['name']} tile={tile} split={split} beta={w['beta']}", flush=True)
        try:
            return gpu_util.run_gpu(handle, w, inp, pref=api.HIPTENSOR_WORKSPACE_MAX, d_alias_c=d_alias_c,
                                    return_info=True)
        except api.HiptensorError as e:
            assert e.status == api.HIPTENSOR_STATUS_EXECUTION_FAILED and tile != TILES[w["dtype"]][-1], e
        finally:
            os.environ.pop("HIPTENSOR_AMD_FORCE_KERNEL", None)


@pytest.mark.parametrize("dtype", list(TILES))
@pytest.mark.parametrize("m,n", OUTPUTS)
def test_reduction_forms(gpu_handle, oracle_mod, dtype, m, n):
    a, b = (1.1 + 0.4j, 0.6 - 0.3j) if dtype.startswith("c") else (1.5, 0.75)
    big = n[0] > 700
    for k, splits in ((130, (2,)) if big else (4160, (2, 16, 32, 64)),):
        for beta, table in ((None, False), (b, True)):
            modes = list(range(len(m))), list(range(10, 10 + len(n)))
            ext = {**dict(zip(modes[0], m)), **dict(zip(modes[1], n)), 20: k}
            d = modes[0] + modes[1]
            if table:
                d = d[::-1]  # columns fastest, and rows of two modes in another order than A's: offsets from tables
            w = wl.make_workload(dtype, cases.COMPUTE[dtype], modes[0] + [20], modes[1] + [20], d, ext, a, beta,
                                 name=f"reduce_{dtype}_{'x'.join(map(str, m))}_{'x'.join(map(str, n))}_{k}")
            inp = wl.host_inputs(w)
            exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
            for split in splits:
                got, info = _run(gpu_handle, w, inp, split)
                assert info["split_k"] == split
                cases.assert_parity(w, cases.logical_view(w, got), exp, f"{info['kernel_name']} split {split}")


# largest K tile of the tiles above
K_TILE = {"f16": 64, "bf16": 64, "f32": 16, "f64": 16, "c32": 8, "c64": 8}


def _one(handle, oracle_mod, dtype, m, n, k_tiles, split, beta, table=False, alias=False, compute=None):
    k = k_tiles * (64 if compute == api.HIPTENSOR_COMPUTE_16F else K_TILE[dtype])
    a = 1.1 + 0.4j if dtype.startswith("c") else 1.5
    b = None if not beta else 0.6 - 0.3j if dtype.startswith("c") else 0.75
    modes = list(range(len(m))), list(range(10, 10 + len(n)))
    ext = {**dict(zip(modes[0], m)), **dict(zip(modes[1], n)), 20: k}
    d = modes[0] + modes[1]
    w = wl.make_workload(dtype, compute or cases.COMPUTE[dtype], modes[0] + [20], modes[1] + [20], d[::-1] if table else d, ext, a, b,
                         name=f"reduce_{dtype}_{'x'.join(map(str, m))}_{'x'.join(map(str, n))}_{k}")
    inp = wl.host_inputs(w)
    exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
    got, info = _run(handle, w, inp, split, d_alias_c=alias)
    assert info["split_k"] == split
    tiles = k // info["tile_k"]
    slices = -(-tiles // -(-tiles // split))  # none of them empty
    assert slices > 8 and slices % 4 != 0, info
    cases.assert_parity(w, cases.logical_view(w, got), exp, f"{info['kernel_name']} split {split}")


@pytest.mark.parametrize("dtype", list(TILES))
@pytest.mark.parametrize("m,n,table", [((7,), (9,), False), ((16, 16), (16, 16), False), ((16, 17), (241,), True), ((400,), (331,), False)])
def test_many_slices(gpu_handle, oracle_mod, dtype, m, n, table):
    """A hundred K tiles in 32 and 64 slices asked for: 25 and 50 slices of four and two tiles, so that the threads of a
    workgroup get unequal numbers of them, and a thread has whole batches of loads and a rest."""
    for split in (32, 64):
        for beta in (False, True):
            _one(gpu_handle, oracle_mod, dtype, m, n, 100, split, beta, table)


@pytest.mark.parametrize("dtype", list(TILES))
@pytest.mark.parametrize("m,n", [((725,), (725,)), ((29, 25), (726,)), ((29, 25), (11, 66)), ((1100,), (500,))])
def test_large_outputs(gpu_handle, oracle_mod, dtype, m, n):
    """16 bytes of outputs a thread and eleven slices (two batches of four and a rest); 1, 2, 2 and 0 outputs left behind the
    last whole vector; D apart from C and in its place, computed offsets and ones from tables (rows along D and across it)."""
    for beta, table, alias in ((False, False, False), (True, False, True), (True, True, True)):
        _one(gpu_handle, oracle_mod, dtype, m, n, 22, 16, beta, table, alias)


@pytest.mark.parametrize("dtype,compute", [("f64", api.HIPTENSOR_COMPUTE_32F), ("f32", api.HIPTENSOR_COMPUTE_16F)])
def test_large_outputs_computed_narrower(gpu_handle, oracle_mod, dtype, compute):
    """The partials' type is not the tensors' (f64 data: four f32 sums make 32 bytes of D)."""
    for m, n, alias in (((725,), (725,), False), ((29, 25), (726,), True)):
        _one(gpu_handle, oracle_mod, dtype, m, n, 22, 16, alias, False, alias, compute)


@pytest.mark.parametrize("dtype", list(TILES))
@pytest.mark.parametrize("m,n", [((1,), (3,)), ((70,), (130,)), ((200,), (14, 10))])
def test_slices_shared_out_between_dies(gpu_handle, oracle_mod, dtype, m, n):
    """Two hundred K tiles in 29 and 50 slices of 1 to 12 (35 for complex f64) output tiles: workgroups are then dealt to
    the dies slice by slice, in shares that do not end where a slice does."""
    for split in (32, 64):
        _one(gpu_handle, oracle_mod, dtype, m, n, 200, split, split == 32)
