"""GPU parity of the 16-bit tiles of 64 and 128 rows whose operand tiles are loaded straight into LDS, where they can go wrong:
every kind of K tail (whole tiles only; ending at, and inside, a vector), fewer K tiles than the ring has stages and more,
rows and columns that end inside a tile (moved back where they are the operand's runs), vectors at 4-byte addresses, an operand
base off its alignment, in place and split."""
import os

import pytest

import cases
import gpu_util
from hiptensor_amd import api
from hiptensor_amd import workloads as wl

pytestmark = pytest.mark.gpu

TILES = {13: (64, 64), 14: (128, 64), 15: (64, 128)}
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
                            strideB=[sb[x] for x in b], name=f"mid_{dtype}_{layout}_{m}x{n}x{k}_pad{pad}")


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
    assert f"{TILES[tile][0]}x{TILES[tile][1]}x64" in info["kernel_name"] and "direct_ring" in info["kernel_name"], info["kernel_name"]
    cases.assert_parity(w, cases.logical_view(w, got), exp, f"{info['kernel_name']} split {info['split_k']}")
    return True


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("layout", LAYOUTS)
def test_k_tails_and_short_rings(gpu_handle, oracle_mod, dtype, tile, layout):
    for k in (64, 65, 66, 72, 104, 126, 128, 192, 256, 318, 320, 390, 640):
        assert check(gpu_handle, oracle_mod, workload(dtype, layout, 136, 200, k, 0.75), tile) == ("k" not in layout or k % 2 == 0)
    assert check(gpu_handle, oracle_mod, workload(dtype, layout, 136, 200, 134, None, pad=2), tile)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("layout", LAYOUTS)
def test_ragged_rows_and_columns(gpu_handle, oracle_mod, dtype, tile, layout):
    bp, bq = TILES[tile]
    for m, n in ((bp, bq), (bp + 2, bq + 2), (2 * bp - 2, bq + 6), (bp + 10, 3 * bq - 2), (16, 2 * bq + 8), (bp + 8, 24), (8, 8)):
        w = workload(dtype, layout, m, n, 200, 0.75)
        assert check(gpu_handle, oracle_mod, w, tile, d_alias_c=True), w["name"]
    # odd rows: only where they are not an operand's runs
    assert check(gpu_handle, oracle_mod, workload(dtype, layout, bp + 3, 2 * bq, 200, None), tile) == (layout[0] == "k")
    assert check(gpu_handle, oracle_mod, workload(dtype, layout, 2 * bp, bq + 5, 200, 0.75), tile, d_alias_c=True) == (layout[1] == "k")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", list(TILES))
def test_splits(gpu_handle, oracle_mod, dtype, tile):
    """Slices with and without the tile that K ends in, of one tile and of several; 8 slices of 160 tiles are shared out between
    the dies slice by slice."""
    for layout in LAYOUTS:
        for k, split in ((330, 2), (330, 4), (1030, 4), (11222, 8)):
            assert check(gpu_handle, oracle_mod, workload(dtype, layout, 130, 194, k, 0.75), tile, split)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_operand_bases(gpu_handle, oracle_mod, dtype):
    """Bases 4 bytes off a 16-byte boundary run the direct loads, 2 bytes off the tile staged through registers: the same
    contraction either way."""
    import torch

    for layout in LAYOUTS:
        w = workload(dtype, layout, 136, 200, 330, None)
        inp = wl.host_inputs(w)
        exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
        os.environ["HIPTENSOR_AMD_FORCE_KERNEL"] = "13,1"
        try:
            c = wl.Contraction(gpu_handle, w, align=2)
        finally:
            os.environ.pop("HIPTENSOR_AMD_FORCE_KERNEL", None)
        for shift in (0, 2, 1, 3):
            A, B = (torch.zeros(inp[t].size + 8, dtype=torch.int16, device="cuda") for t in "AB")
            A[shift:shift + inp["A"].size] = gpu_util.to_device(inp["A"]).view(torch.int16)
            B[shift:shift + inp["B"].size] = gpu_util.to_device(inp["B"]).view(torch.int16)
            D = gpu_util.to_device(wl.nan_buffer(dtype, inp["spanD"]))
            print(f"[case] {w['name']} shift {shift}", flush=True)
            st = c.run(A.data_ptr() + 2 * shift, B.data_ptr() + 2 * shift, None, D.data_ptr(), None, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            api.check(st, w["name"])
            cases.assert_parity(w, cases.logical_view(w, D.cpu().numpy().view(wl.NP_STORE[dtype])), exp, f"shift {shift}")
        c.close()
