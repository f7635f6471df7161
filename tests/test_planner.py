"""Host-side planning, on a device-less handle: mode classification, ordering and fusion,
vector widths, kernel choice, and the eight offset tables against brute-force addressing.
Reference behaviour being replaced: normalizeTensorModes
(library/src/contraction/contraction_solution.cpp:34-160)."""
import itertools

import numpy as np
import pytest

import cases
from hiptensor_amd import api
from hiptensor_amd import workloads as wl

XP, XK, YQ, YK, CP, CQ, DP, DQ = range(8)


def plan(host_handle, w, **kw):
    c = wl.Contraction(host_handle, w, **kw)
    info = dict(c.info)
    tabs = [api.planTable(c.plan, i) for i in range(8)]
    c.close()
    return info, tabs


def test_baseline_configs_fold_to_expected_gemms(host_handle):
    exp = {"cfg1": (256, 256, 256), "cfg2_f16_scale": (4096, 4096, 4096), "cfg3": (1920, 1920, 768),
           "cfg4": (1024, 1024, 512), "cfg5": (5376, 6912, 4080)}
    for name, (M, N, K) in exp.items():
        w = wl.baseline_configs()[name]
        info, _ = plan(host_handle, w)
        # D is contiguous along its first M mode in every configuration: rows come from B
        assert info["swapped"] == 1
        assert (info["Q"], info["P"], info["K"]) == (M, N, K)
        if name != "cfg5":
            # packed column-major: every group fuses into one dim, operands gather along rows
            assert (info["n_pdims"], info["n_qdims"], info["n_kdims"]) == (1, 1, 1)
            assert info["x_kfast"] == 0 and info["y_kfast"] == 0
        else:
            # nothing fuses; A is contiguous along k1 (runs of 8), B along n2
            assert (info["n_pdims"], info["n_qdims"], info["n_kdims"]) == (3, 3, 3)
            assert info["y_kfast"] == 1 and info["x_kfast"] == 0
        maxv = 16 // wl.ELEM_BYTES[w["dtype"]]
        assert info["x_vec"] == maxv and info["y_vec"] == maxv and info["cd_vec"] == maxv


def brute_offsets(w, tensor):
    """offset of every logical element, indexed by the listed modes."""
    lens, strides = w["lens"][tensor if tensor != "C" else "D"], w["strides"][tensor]
    grids = np.meshgrid(*[np.arange(l) for l in lens], indexing="ij")
    return sum(g * s for g, s in zip(grids, strides))


@pytest.mark.parametrize("name", ["cfg5_small", "mode7", "mode9", "rank4_colmajor", "rank3_default"])
def test_tables_address_every_element(host_handle, name):
    """xp[p] + xk[k] enumerates X's offsets exactly once each (likewise Y, C, D), and the same
    (p, q) addresses C and D at the same logical element."""
    w = {"cfg5_small": lambda: wl.config5(extents=(8, 3, 2, 4, 3, 8, 5, 8, 3)),
         "mode7": lambda: cases.mode_case(7, "c32", 1.0, None),
         "mode9": lambda: cases.mode_case(9, "f16", 1.0, None),
         "rank4_colmajor": lambda: cases.rank_case(4, "f32", 1.0, 2.0, col_major=True),
         "rank3_default": lambda: cases.rank_case(3, "f64", 1.0, 2.0)}[name]()
    info, t = plan(host_handle, w)
    P, Q, K = info["P"], info["Q"], info["K"]
    M, N, Kw = wl.dims(w)
    assert sorted((P, Q)) == sorted((M, N)) and K == Kw
    X, Y = ("B", "A") if info["swapped"] else ("A", "B")
    for tens, rows, ks in ((X, t[XP], t[XK]), (Y, t[YQ], t[YK])):
        got = np.add.outer(np.array(rows), np.array(ks)).ravel()
        want = brute_offsets(w, tens).ravel()
        assert len(got) == len(want) and np.array_equal(np.sort(got), np.sort(want)), tens
    gotd = np.add.outer(np.array(t[DP]), np.array(t[DQ]))
    assert np.array_equal(np.sort(gotd.ravel()), np.sort(brute_offsets(w, "D").ravel()))
    if w["beta"] is not None:
        gotc = np.add.outer(np.array(t[CP]), np.array(t[CQ]))
        # C and D share modes: the element D reaches at (p, q) is the one C reaches
        dmap = {int(o): idx for idx, o in np.ndenumerate(brute_offsets(w, "D"))}
        cmap = {int(o): idx for idx, o in np.ndenumerate(brute_offsets(w, "C"))}
        for p, q in itertools.product(range(0, P, max(1, P // 7)), range(0, Q, max(1, Q // 7))):
            assert dmap[int(gotd[p, q])] == cmap[int(gotc[p, q])]


def test_operand_pairing_is_consistent(host_handle):
    """For every (p, q, k) the X and Y elements the tables reach carry the same k index, and
    the D element carries p's and q's indices: check through an einsum on index-coded data."""
    w = cases.mode_case(8, "f64", 1.0, None)
    w["compute"] = api.HIPTENSOR_COMPUTE_64F
    info, t = plan(host_handle, w)
    inp = wl.host_inputs(w)
    X, Y = (inp["B"], inp["A"]) if info["swapped"] else (inp["A"], inp["B"])
    xp, xk, yq, yk, dp, dq = (np.array(t[i]) for i in (XP, XK, YQ, YK, DP, DQ))
    acc = np.einsum("pk,qk->pq", X[np.add.outer(xp, xk)], Y[np.add.outer(yq, yk)])
    import oracle

    ref = oracle.contract(w, inp["A"], inp["B"], None)
    assert np.allclose(acc, ref[np.add.outer(dp, dq)], rtol=0, atol=1e-11)


def test_vector_width_follows_runs_not_alignment(host_handle):
    ext = {0: 16, 1: 6, 10: 8, 11: 10, 20: 16, 21: 5}
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["cd_vec"]) == (8, 8, 8)
    # pointers that are only element-aligned keep the vectors: global memory takes vector loads
    # and stores at any element-aligned address
    info, _ = plan(host_handle, w, align=2)
    assert (info["x_vec"], info["y_vec"], info["cd_vec"]) == (8, 8, 8)
    ext[0], ext[1] = 12, 5  # the fused M run has 60 elements: not a multiple of 8
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    # 16-bit kernels exist for (8,8), (4,4), (2,2), (8,1), (1,8), (1,1): the pair is narrowed jointly
    assert (info["x_vec"], info["y_vec"]) == (4, 4)
    ext[0], ext[1] = 10, 3  # runs of 30 elements: 4-byte vectors
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"]) == (2, 2)
    ext[0], ext[1] = 5, 3  # odd run: that operand is a scalar gather (staged k-fast), the other keeps 16 bytes
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["y_kfast"]) == (8, 1, 1)
    ext[10], ext[11] = 12, 3  # ... and a 4-element run beside a scalar operand falls to scalar as well
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["x_kfast"], info["y_kfast"]) == (1, 1, 1, 1)
    # f32 kernels exist for (4,4), (4,1), (1,4), (1,1) and (2,2): a run of 30 elements beside one of 80 narrows both to 8 bytes
    ext = {0: 6, 1: 5, 10: 8, 11: 10, 20: 16, 21: 5}
    w = wl.make_workload("f32", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"]) == (2, 2)
    ext[0] = 5  # ... an odd run is a scalar gather, and the other operand keeps 16 bytes
    w = wl.make_workload("f32", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"]) == (4, 1)
    # the other wide classes have full-width or scalar kernels only (f32 tensors contracted in 16-bit arithmetic: 4 or 1)
    ext[0] = 6
    w = wl.make_workload("f32", api.HIPTENSOR_COMPUTE_16F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"]) == (4, 1)
    # an odd row pitch (leading dimension padded by one element) does not narrow anything either
    ext = {0: 16, 1: 6, 10: 8, 11: 10, 20: 16, 21: 5}
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None,
                         strideA=[1, 16, 97, 97 * 16], strideB=[1, 8, 81, 81 * 16])
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["x_kfast"], info["y_kfast"]) == (8, 8, 0, 0)


def test_ragged_contiguous_rows_and_columns_keep_their_vectors(host_handle):
    """A row (column) index that is one contiguous run of at least 256 elements carries vectors
    even when its extent is odd: the last tile is moved back to end at the extent.  Shorter or
    multi-dim ragged indices fall to scalars as before."""
    ext = {0: 15, 1: 19, 10: 17, 11: 21, 20: 16, 21: 4}  # M = 285, N = 357, packed: each fuses to one run
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, 0.5)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["cd_vec"], info["x_kfast"], info["y_kfast"]) == (8, 8, 8, 0, 0)
    assert info["n_pdims"] == 1 and info["n_qdims"] == 1
    w32 = wl.make_workload("f32", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w32)
    assert (info["x_vec"], info["y_vec"], info["cd_vec"]) == (4, 4, 4)
    ext = {0: 15, 1: 13, 10: 17, 11: 11, 20: 16, 21: 4}  # M = 195, N = 187: only tiles of at most 128 can be moved back
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["cd_vec"]) == (8, 8, 8) and max(info["tile_p"], info["tile_q"]) <= 128
    ext = {0: 15, 1: 3, 10: 17, 11: 3, 20: 16, 21: 4}  # M = 45, N = 51: shorter than the smallest tile
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["cd_vec"]) == (1, 1, 1)
    # a contiguous K of odd extent keeps k-fast vectors (the straddling vector is handled in the last K tile)
    ext = {0: 16, 1: 6, 10: 8, 11: 10, 20: 15, 21: 7}
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [20, 21, 0, 1], [20, 21, 10, 11], [10, 11, 0, 1], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["x_kfast"], info["y_kfast"], info["n_kdims"]) == (8, 8, 1, 1, 1)
    w = wl.make_workload("f64", api.HIPTENSOR_COMPUTE_64F, [20, 21, 0, 1], [20, 21, 10, 11], [10, 11, 0, 1], ext, 1.0, None)
    info, _ = plan(host_handle, w)
    assert (info["x_vec"], info["y_vec"], info["x_kfast"], info["y_kfast"]) == (2, 2, 1, 1)
    # padded leading dimension: M stays two dims (15 | 19), vectors cannot straddle the gap
    ext = {0: 15, 1: 19, 10: 17, 11: 21, 20: 16, 21: 4}
    w = wl.make_workload("f16", api.HIPTENSOR_COMPUTE_32F, [0, 1, 20, 21], [10, 11, 20, 21], [0, 1, 10, 11], ext, 1.0, None,
                         strideA=[1, 16, 16 * 19, 16 * 19 * 16])
    info, _ = plan(host_handle, w)
    assert info["n_pdims"] + info["n_qdims"] >= 3 and 1 in (info["x_vec"], info["y_vec"])


def test_extent_one_modes_and_missing_groups(host_handle):
    # no K modes at all (outer product), and extent-1 modes everywhere
    ext = {0: 4, 1: 1, 10: 3, 11: 1}
    w = wl.make_workload("f32", api.HIPTENSOR_COMPUTE_32F, [0, 1], [10, 11], [0, 10, 1, 11], ext, 1.0, None)
    info, t = plan(host_handle, w)
    assert info["K"] == 1 and sorted((info["P"], info["Q"])) == [3, 4]
    # all of D's modes come from A: N is empty
    w = wl.make_workload("f32", api.HIPTENSOR_COMPUTE_32F, [0, 20], [20], [0], {0: 5, 20: 7}, 1.0, None)
    info, t = plan(host_handle, w)
    assert sorted((info["P"], info["Q"])) == [1, 5] and info["K"] == 7


def test_plans_are_cached_per_handle(host_handle):
    w = cases.rank_case(3, "f32", 1.0, 2.0)
    a = wl.Contraction(host_handle, w)
    b = wl.Contraction(host_handle, w)
    assert a.info == b.info
    a.close()
    b.close()


def test_workspace_preferences(host_handle):
    w = wl.config1()  # 256^3: too few tiles for 256 CUs without split-K
    t = wl.HIP_TYPE[w["dtype"]]
    c = wl.Contraction(host_handle, w, pref=api.HIPTENSOR_WORKSPACE_MIN)
    assert c.workspace_bytes == 0 and c.info["split_k"] == 1
    c.close()
    rec = wl.Contraction(host_handle, w, pref=api.HIPTENSOR_WORKSPACE_RECOMMENDED)
    mx = wl.Contraction(host_handle, w, pref=api.HIPTENSOR_WORKSPACE_MAX)
    assert mx.workspace_bytes >= rec.workspace_bytes
    assert rec.info["workspace_bytes"] <= rec.workspace_bytes
    if rec.info["split_k"] > 1:
        assert rec.info["workspace_bytes"] == rec.info["split_k"] * 256 * 256 * 4
    rec.close()
    mx.close()


def test_direct_load_kernels_keep_32_bit_offsets_in_range(host_handle, monkeypatch):
    """The kernels that load straight into LDS address an operand with 32-bit byte offsets, and some keep a bias of up
    to 3 KiB in a lane's offset (loads that share one write of M0): an operand whose last vector ends within that of
    4 GiB is not offered to them, one that ends a few KiB earlier is.  (A: 512 rows contiguous, 128 k at a stride that
    puts the last vector where the case wants it.)"""
    ext = {0: 512, 10: 512, 20: 128}
    top = (2 ** 31 - 512 - 8) // 127 // 8 * 8  # largest k stride, a multiple of 8 elements, whose last vector ends below 4 GiB

    def kernel(stride, force):
        if force:
            monkeypatch.setenv("HIPTENSOR_AMD_FORCE_KERNEL", force)
        else:
            monkeypatch.delenv("HIPTENSOR_AMD_FORCE_KERNEL", raising=False)
        w = wl.make_workload("f16", cases.COMPUTE["f16"], [0, 20], [10, 20], [0, 10], ext, 1.0, None, strideA=[1, stride],
                             name=f"a_ends_near_4GiB_{stride}")
        try:
            info, _ = plan(host_handle, w)
        except api.HiptensorError as e:
            assert e.status == api.HIPTENSOR_STATUS_EXECUTION_FAILED, e
            return None
        return info["kernel_name"]

    for stride, offered in ((top, False), (top - 8, False), (top - 16, True)):
        room = 2 ** 32 - (2 * (511 + 127 * stride) + 16)
        assert (room > 3072) == offered, (stride, room)
        for force in ("9,1", "10,1", "11,1", "12,1"):
            name = kernel(stride, force)
            assert (name is not None and "direct" in name) == offered, (stride, force, name)
        name = kernel(stride, None)
        assert name is not None and (offered or "direct" not in name), (stride, name)


@pytest.mark.parametrize("dtype,modes,ext,split,packed", [
    # small results of long reductions: the slices' reduction costs about a microsecond more for 64 of them than for two
    ("f16", ([0, 20], [20, 10], [0, 10]), {0: 199, 10: 191, 20: 94385}, 64, 0),
    ("f32", ([20, 21, 0], [20, 10, 21], [0, 10]), {0: 104, 10: 34, 20: 34, 21: 320}, 64, 0),
    ("f64", ([20, 0], [20, 10], [10, 0]), {0: 55, 10: 173, 20: 9726}, 64, 0),
    ("bf16", ([20, 0], [20, 10], [10, 0]), {0: 36, 10: 216, 20: 36540}, 64, 0),
    # ... but slices of few K tiles are mostly prologue
    ("f16", ([0, 20], [10, 20], [0, 10]), {0: 160, 10: 160, 20: 2048}, 8, 0),
    ("f32", ([0, 20], [10, 20], [0, 10]), {0: 256, 10: 256, 20: 256}, 1, 0),
])
def test_slices_of_long_reductions(host_handle, dtype, modes, ext, split, packed):
    w = wl.make_workload(dtype, cases.COMPUTE[dtype], *modes, ext, 1.5, None, name="long_k")
    info, _ = plan(host_handle, w)
    assert (info["split_k"], info["pack_a"] + info["pack_b"]) == (split, packed), info["kernel_name"]
