"""GPU parity where an operand's base is not aligned for the tile the plan chose: the staged tile that stands in runs in its own
number of slices, in fewer where the call's workspace holds fewer, in one without a workspace."""
import pytest

import cases
import gpu_util
from hiptensor_amd import api
from hiptensor_amd import workloads as wl

pytestmark = pytest.mark.gpu

SIZES = {"f16": (160, 384, 1152), "bf16": (96, 130, 4100), "f64": (48, 80, 3000), "c32": (72, 66, 2050)}


@pytest.mark.parametrize("dtype", list(SIZES))
@pytest.mark.parametrize("kfast", [False, True])
def test_stand_in_and_its_slices(gpu_handle, oracle_mod, dtype, kfast):
    import torch

    m, n, k = SIZES[dtype]
    e = wl.ELEM_BYTES[dtype]
    a, b = ([20, 0], [20, 10]) if kfast else ([0, 20], [10, 20])
    w = wl.make_workload(dtype, cases.COMPUTE[dtype], a, b, [0, 10], {0: m, 10: n, 20: k}, 1.5, 0.75, name=f"off_{dtype}_{m}x{n}x{k}_{kfast}")
    inp = wl.host_inputs(w)
    exp = cases.logical_view(w, oracle_mod.contract(w, inp["A"], inp["B"], inp["C"]))
    c = wl.Contraction(gpu_handle, w, align=e)
    need = int(c.info["workspace_bytes"])
    slices = {need, need + 3 * m * n * max(4, e), c.workspace_bytes}
    C, ws = gpu_util.to_device(inp["C"]), torch.empty(max(max(slices), 256), dtype=torch.uint8, device="cuda")
    for shift in (0, 1, 2, 3):
        A, B = (torch.zeros(inp[t].size * e + 16 * e, dtype=torch.uint8, device="cuda") for t in "AB")
        A[shift * e:(shift + inp["A"].size) * e] = gpu_util.to_device(inp["A"])
        B[shift * e:(shift + inp["B"].size) * e] = gpu_util.to_device(inp["B"])
        for held in sorted(slices):
            D = gpu_util.to_device(wl.nan_buffer(dtype, inp["spanD"]))
            print(f"[case] {w['name']} {c.info['kernel_name']} shift {shift} workspace {held}", flush=True)
            st = c.run(A.data_ptr() + shift * e, B.data_ptr() + shift * e, C.data_ptr(), D.data_ptr(), ws.data_ptr() if held else None,
                       torch.cuda.current_stream().cuda_stream, workspace_bytes=held)
            torch.cuda.synchronize()
            api.check(st, w["name"])
            cases.assert_parity(w, cases.logical_view(w, D.cpu().numpy().view(wl.NP_STORE[dtype])), exp, f"shift {shift} workspace {held}")
    c.close()
