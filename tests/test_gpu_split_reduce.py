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


def _run(handle, w, inp, split):
    """On the first of the class's small tiles that takes the layout."""
    for tile in TILES[w["dtype"]]:
        os.environ["HIPTENSOR_AMD_FORCE_KERNEL"] = f"{tile},{split}"
        print(f"[case] {w['name']} tile={tile} split={split} beta={w['beta']}", flush=True)
        try:
            return gpu_util.run_gpu(handle, w, inp, pref=api.HIPTENSOR_WORKSPACE_MAX, return_info=True)
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
