"""Whether a plan moves operands into packed copies: the estimates of the two plans are compared with the same correction for
slices, and the plan is the one whose workspace was recommended."""
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


# unpacked in slices against packed, as timed: 8.8 and 17.2 us, 9.9 and 16.9, 8.2 and 11.9, 9.6 and 11.6
IN_PLACE = [("f16", "bxca,ix->abci", dict(a=5, b=7, c=4, i=229, x=1825)), ("bf16", "axbycz,ixyz->abci", dict(a=9, b=3, c=11, i=184, x=6, y=12, z=22)),
            ("bf16", "abxy,ixy->abi", dict(a=10, b=109, i=7, x=41, y=38)), ("f16", "axby,ixjyk->abijk", dict(a=3, b=8, i=8, j=20, k=12, x=48, y=28))]
# ... and 89 and 61 us, 20.5 and 16.8 (f16 384 x 56 x 8640: read where they lie 20.6 all the same), 15.6 and 12.7
PACKED = [("bf16", "axby,ixy->aib", dict(a=44, b=30, i=4220, x=34, y=86)), ("f16", "axyz,ixjyz->aij", dict(a=1012, i=14, j=39, x=9, y=4, z=20))]


@pytest.mark.parametrize("dtype,modes,ext", IN_PLACE)
def test_operands_read_where_they_lie(host_handle, dtype, modes, ext):
    info = plan(host_handle, dtype, modes, ext)
    assert not info["pack_a"] and not info["pack_b"] and info["split_k"] >= 8, info


@pytest.mark.parametrize("dtype,modes,ext", PACKED)
def test_operands_packed(host_handle, dtype, modes, ext):
    info = plan(host_handle, dtype, modes, ext)
    assert info["pack_a"] or info["pack_b"], info


def test_no_copy_in_tiles_of_a_few_elements(host_handle):
    """B in tiles of 3 x 3 complex numbers, the copy alone 135 us: 179 us in all, 42 where it lies."""
    info = plan(host_handle, "c32", "ax,kixj->aijk", dict(a=252, i=3, j=4, k=3, x=27336))
    assert "2x3x3" not in info["pack_a_kernel"] + info["pack_b_kernel"], info


@pytest.mark.parametrize("dtype", ["f64", "c32"])
@pytest.mark.parametrize("m,n,k", [(3, 1111, 2009), (5, 700, 1501), (1111, 3, 2009), (61, 803, 1107)])
def test_the_recommended_workspace_is_enough_for_the_plan_it_was_computed_for(host_handle, dtype, m, n, k):
    """A plan made with the recommended workspace is the one made with all of it (packed copies had been weighed by another
    tile than they run, so that the recommendation for them did not bring them about: c32 3 x 1111 x 2009 20.7 -> 44.7 us)."""
    for modes in ("ax,ix->ai", "xa,ix->ai"):
        ext = dict(a=m, i=n, x=k)
        few, all_ = (plan(host_handle, dtype, modes, ext, pref) for pref in (api.HIPTENSOR_WORKSPACE_RECOMMENDED, api.HIPTENSOR_WORKSPACE_MAX))
        assert {x: few[x] for x in ("kernel_name", "split_k", "pack_a", "pack_b")} == {x: all_[x] for x in ("kernel_name", "split_k", "pack_a", "pack_b")}, (modes, few, all_)
