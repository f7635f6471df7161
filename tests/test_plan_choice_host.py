"""Plans that were timed against their alternatives: what the estimates have to choose."""
import pytest

import cases
from hiptensor_amd import api
from hiptensor_amd import workloads as wl


def plan(handle, dtype, modes, ext, pref=api.HIPTENSOR_WORKSPACE_RECOMMENDED, beta=None):
    a, b = modes.split("->")[0].split(",")
    d = modes.split("->")[1]
    w = wl.make_workload(dtype, cases.COMPUTE[dtype], [ord(x) for x in a], [ord(x) for x in b], [ord(x) for x in d],
                         {ord(k): v for k, v in ext.items()}, 1.5, beta, name=f"{dtype}_{modes}")
    c = wl.Contraction(handle, w, pref=pref)
    out = dict(c.info, recommended=c.workspace_bytes)
    c.close()
    return out


@pytest.mark.parametrize("dtype,m,n,k", [("f64", 5487, 55, 5035), ("f64", 9000, 46, 1733)])
def test_rows_off_the_lines_read_from_memory_in_slices(host_handle, dtype, m, n, k):
    """k-contiguous operands of odd rows that no cache holds, in slices: 121 and 72 us on tiles loaded straight into LDS, 88 and 58
    staged through registers."""
    info = plan(host_handle, dtype, "xa,xi->ai", dict(a=m, i=n, x=k))
    assert "_any_" not in info["kernel_name"], info
