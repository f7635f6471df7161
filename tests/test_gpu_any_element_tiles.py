"""GPU parity of the f32, f64 and complex f32 tiles that are loaded straight into LDS from any element, where they can go wrong:
every kind of K tail (none; ending at, and inside, a vector), fewer K tiles than the ring has stages or waves, and more, rows and
columns that end inside a tile (moved back where they are the operand's runs), leading dimensions off the vectors' length, in
place and split."""
import os

import pytest

import cases
import gpu_util
from hiptensor_amd import api
from hiptensor_amd import workloads as wl

pytestmark = pytest.mark.gpu

TILES = {4: 64, 5: 32}
BK = {"f32": 16, "f64": 8, "c32": 8}
VEC = {"f32": 4, "f64": 2, "c32": 2}
# (A, B) stored with the free (r) or the contracted (k) modes fastest
LAYOUTS = ["kk", "rr", "rk", "kr"]


def workload(dtype, layout, m, n, k, beta, pad=0):
    """D is contiguous along B's free mode: A holds the rows and B the columns of the tile; `pad`: elements behind A's and
    B's fastest mode."""
    a, b = ([0, 20] if layout[0] == "r" else [20, 0]), ([10, 20] if layout[1] == "r" else [20, 10])
    ext = {0: m, 10: n, 20: k}
    strides = lambda o: {o[0]: 1, o[1]: ext[o[0]] + pad}
    sa, sb = strides(a), strides(b)
    return wl.make_workload(dtype, cases.COMPUTE[dtype], a, b, [10, 0], ext, 1.5, beta, strideA=[sa[x] for x in a],
                            strideB=[sb[x] for x in b], name=f"any_{dtype}_{layout}_{m}x{n}x{k}_pad{pad}")


def run(handle, w, inp, tile, split=1, **kw):
    os.environ["HIPTENSOR_AMD_FORCE_KERNEL"] = f"{tile},{split}"
    print(f"[case] {w['name']} tile {tile} split {split}", flush=True)
    try:
        return gpu_util.run_gpu(handle, w, inp, pref=api.HIPTENSOR_WORKSPACE_MAX, return_info=True, **kw)
    except api.HiptensorError as e:
        assert e.status == api.HIPTENSOR_STATUS_EXECUTION_FAILED, e
        return None, None
    finally:
        os.environ.pop("HIPTENSOR_AMD_FORCE_KERNEL", None)


def check(handle, oracle_mod, w, tile, split=1, **kw):
    inp = wl.host_inputs(w)
    exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
    got, info = run(handle, w, inp, tile, split, **kw)
    if got is None:
        return False
    assert "_any_x" in info["kernel_name"], info["kernel_name"]
    cases.assert_parity(w, cases.logical_view(w, got), exp, f"{info['kernel_name']} split {info['split_k']}")
    return True


@pytest.mark.parametrize("dtype", list(BK))
@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("layout", LAYOUTS)
def test_k_tails_and_short_rings(gpu_handle, oracle_mod, dtype, tile, layout):
    bk = BK[dtype]
    for k in (bk, bk + 1, bk + 2, 2 * bk - 1, 2 * bk, 3 * bk + 3, 4 * bk + 1, 5 * bk - 2, 9 * bk, 9 * bk + 5):
        assert check(gpu_handle, oracle_mod, workload(dtype, layout, 68, 100, k, 0.75), tile)
    assert check(gpu_handle, oracle_mod, workload(dtype, layout, 68, 100, 6 * bk + 1, None, pad=1), tile)
    assert not check(gpu_handle, oracle_mod, workload(dtype, layout, 68, 100, bk - 1, None), tile)


@pytest.mark.parametrize("dtype", list(BK))
@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("layout", LAYOUTS)
def test_ragged_rows_and_columns(gpu_handle, oracle_mod, dtype, tile, layout):
    b = TILES[tile]
    for m, n in ((b, b), (65, 65), (127, 67), (69, 191), (4 * b, 2 * b)): # (ragged runs of fewer than 64 rows are gathered by elements)
        w = workload(dtype, layout, m, n, 77, 0.75)
        assert check(gpu_handle, oracle_mod, w, tile, d_alias_c=True), w["name"]


@pytest.mark.parametrize("dtype", list(BK))
@pytest.mark.parametrize("tile", list(TILES))
def test_splits(gpu_handle, oracle_mod, dtype, tile):
    """Slices with and without the tile that K ends in, of one tile and of several."""
    for layout in LAYOUTS:
        for k, split in ((83, 2), (83, 4), (517, 4), (11221, 8)):
            assert check(gpu_handle, oracle_mod, workload(dtype, layout, 67, 97, k, 0.75), tile, split)
