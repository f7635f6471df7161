"""GPU parity of the tiles loaded straight into LDS where the tests of each kernel do not reach: slices shared out between the
dies on every one of them, rows and columns of several modes (offsets from tables, C / D addressed through tables), and
infinities and NaN on both sides of the K tail's end."""
import numpy as np
import pytest

import cases
import gpu_util
import test_gpu_any_element_tiles as any_tiles
import test_gpu_mid_tiles as mid_tiles
from hiptensor_amd import api
from hiptensor_amd import workloads as wl

pytestmark = pytest.mark.gpu

LAYOUTS = mid_tiles.LAYOUTS


# (dtype, direct tile ids, K: 160 K tiles and more, with a short one at the end, rows, columns)
SLICED = [("f16", (9, 10, 11, 12), 10256, 264, 520), ("bf16", (9, 10, 11, 12), 10256, 264, 520), ("f32", (2, 3), 2564, 68, 164),
          ("f64", (2, 3), 2564, 68, 164), ("c32", (2, 3), 2564, 68, 164), ("c64", (3, 4), 2564, 68, 164)]


@pytest.mark.parametrize("layout", ["kk", "rr", "rk"])
@pytest.mark.parametrize("dtype,tiles,k,m,n", SLICED, ids=[s[0] for s in SLICED])
def test_slices_shared_out_between_dies(gpu_handle, oracle_mod, dtype, tiles, k, m, n, layout):
    """Several output tiles in 27 to 41 slices, a number of workgroups that no die's share divides."""
    w = mid_tiles.workload(dtype, layout, m, n, k, 0.75)
    inp = wl.host_inputs(w)
    exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
    ran = 0
    for tile in tiles:
        got, info = mid_tiles.run(gpu_handle, w, inp, tile, 32)
        if got is None:
            continue
        assert "direct" in info["kernel_name"] and info["split_k"] == 32, info
        assert -(-k // info["tile_k"]) >= 160 and k % info["tile_k"] != 0, info
        cases.assert_parity(w, cases.logical_view(w, got), exp, f"{info['kernel_name']} split 32")
        ran += 1
    # (the f32, f64 and complex f32 tiles of these ids take one k-contiguous operand or two, or none, in vectors of the same length)
    assert ran == len(tiles), (w["name"], ran)


# (modes of A, B, D): rows in two modes and columns in two, which lie apart in D; the operands row-contiguous (r) or not (k)
TABLES = {
    "rr": ([0, 1, 20], [10, 20, 11], [10, 0, 11, 1]),
    "kk": ([20, 0, 1], [20, 10, 11], [11, 1, 10, 0]),
    "rk": ([0, 20, 1], [20, 11, 10], [0, 10, 1, 11]),
    "kr": ([20, 1, 0], [10, 20, 11], [10, 0, 11, 1]),
}


def table_workload(dtype, form, m, n, k, beta):
    a, b, d = TABLES[form]
    ext = {0: m[0], 1: m[1], 10: n[0], 11: n[1], 20: k}
    return wl.make_workload(dtype, cases.COMPUTE[dtype], a, b, d, ext, 1.5, beta, name=f"tables_{dtype}_{form}_{m}_{n}_{k}")


def check_tables(handle, oracle_mod, run, w, tile, split, mark):
    inp = wl.host_inputs(w)
    exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
    got, info = run(handle, w, inp, tile, split)
    assert got is not None and mark in info["kernel_name"], (w["name"], tile, info)
    assert info["n_pdims"] == 2 and info["n_qdims"] == 2, info
    cases.assert_parity(w, cases.logical_view(w, got), exp, f"{info['kernel_name']} split {split}")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("tile", list(mid_tiles.TILES))
@pytest.mark.parametrize("form", list(TABLES))
def test_rows_from_tables_16_bit(gpu_handle, oracle_mod, dtype, tile, form):
    for m, n, k, split in (((24, 7), (16, 13), 330, 1), ((32, 9), (24, 11), 200, 1), ((8, 5), (40, 3), 1030, 4)):
        for beta in (None, 0.75):
            check_tables(gpu_handle, oracle_mod, mid_tiles.run, table_workload(dtype, form, m, n, k, beta), tile, split, "direct_ring")


@pytest.mark.parametrize("dtype", list(any_tiles.BK))
@pytest.mark.parametrize("tile", list(any_tiles.TILES))
@pytest.mark.parametrize("form", list(TABLES))
def test_rows_from_tables_32_64_bit(gpu_handle, oracle_mod, dtype, tile, form):
    for m, n, k, split in (((24, 7), (16, 13), 77, 1), ((32, 9), (24, 11), 131, 1), ((8, 5), (40, 3), 517, 4)):
        for beta in (None, 0.75):
            check_tables(gpu_handle, oracle_mod, any_tiles.run, table_workload(dtype, form, m, n, k, beta), tile, split, "_any_x")


def infinite(dtype):
    return {"f16": np.uint16(0x7C00), "bf16": np.uint16(0x7F80)}.get(dtype, np.inf)


def check_infinities(handle, module, dtype, layout, tile, k, vec, pad):
    """One infinity in a row of A or a column of B at each of the last `vec` + 1 k and at the first: that row (column) of D is infinite and
    nothing else changes.  The padding behind every row holds NaN."""
    m, n = 136, 72
    w = module.workload(dtype, layout, m, n, k, None, pad=pad)
    inp = wl.host_inputs(w)
    plain, info = module.run(handle, w, inp, tile)
    assert plain is not None, w["name"]
    plain = cases.logical_view(w, plain)  # (columns of B, rows of A)
    for side, rows in (("A", m), ("B", n)):
        lens, strides = w["lens"][side], w["strides"][side]
        free, kk = (0, 1) if layout["AB".index(side)] == "r" else (1, 0)
        row = rows - 3
        for at in sorted({0} | set(range(k - vec - 1, k))):
            x = dict(inp)
            x[side] = inp[side].copy()
            flat = x[side].view(np.uint16) if dtype in ("f16", "bf16") else x[side]
            flat[row * strides[free] + at * strides[kk]] = infinite(dtype)
            got, _ = module.run(handle, w, x, tile)
            got = cases.logical_view(w, got)
            hit = got[:, row] if side == "A" else got[row, :]
            rest = np.delete(got, row, axis=1 if side == "A" else 0)
            same = np.delete(plain, row, axis=1 if side == "A" else 0)
            what = f"{info['kernel_name']} {w['name']} {side} k {at}"
            assert rest.tobytes() == same.tobytes(), what
            f = wl.to_float(dtype, np.ascontiguousarray(hit))
            if dtype.startswith("c"):  # (inf times a complex number has NaN parts)
                assert not np.any(np.isfinite(f)), what
            else:
                assert np.all(np.isinf(f)), what


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_infinities_beside_the_k_tail_16_bit(gpu_handle, dtype, layout):
    for tile in mid_tiles.TILES:
        for k in (66, 134):  # (one K tile and the short one taken first; K ends inside a vector)
            check_infinities(gpu_handle, mid_tiles, dtype, layout, tile, k, 8, 2)


@pytest.mark.parametrize("dtype", list(any_tiles.BK))
@pytest.mark.parametrize("layout", LAYOUTS)
def test_infinities_beside_the_k_tail_32_64_bit(gpu_handle, dtype, layout):
    bk = any_tiles.BK[dtype]
    for tile in any_tiles.TILES:
        for k in (bk + 1, 6 * bk + any_tiles.VEC[dtype] - 1):
            check_infinities(gpu_handle, any_tiles, dtype, layout, tile, k, any_tiles.VEC[dtype], 1)
