"""Which permutations of f16 with pairs on one side and single elements on the other take 16-byte vectors at any element."""
import pytest

from hiptensor_amd import api


@pytest.mark.parametrize("lens,perm,kernel", [
    ((136519, 660), (1, 0), "permute_tiled_f16_512x32_r1_w2"),  # written in pairs from 32 columns
    ((148981, 84), (1, 0), "permute_tiled_f16_512x32_r1_w2"),
    ((895, 79906), (1, 0), "permute_tiled_f16_128x128_r1_w2"),  # large matrices
    ((124, 600001), (1, 0), "permute_tiled_f16_128x128_r2_w1"),
    ((10862, 11813), (1, 0), "permute_tiled_f16_256x128_r2_w1"),
    ((12203, 9772), (1, 0), "permute_tiled_f16_256x128_r8_w8_loose"),
    ((3125, 10538), (1, 0), "permute_tiled_f16_256x128_r8_w8_loose"),  # up to 2^25 elements
    ((246, 126985), (1, 0), "permute_tiled_f16_256x128_r8_w8_loose"),
    ((638, 918, 225), (2, 0, 1), "permute_tiled_f16_256x128_r8_w8_loose"),  # short columns
    ((572, 595, 231), (1, 0, 2), "permute_tiled_f16_128x128_r8_w8_loose"),  # more modes
    ((8025, 3025), (1, 0), "permute_tiled_f16_256x128_r8_w8_loose"),  # single elements on both sides
    ((69889, 157), (1, 0), "permute_tiled_f16_512x32_r8_w8_loose"),
])
def test_pairs_against_single_elements(host_handle, lens, perm, kernel):
    dA = api.check(api.hiptensorInitTensorDescriptor(host_handle, lens, None, api.HIP_R_16F))
    dB = api.check(api.hiptensorInitTensorDescriptor(host_handle, [lens[p] for p in perm], None, api.HIP_R_16F))
    info = api.check(api.permutationInfo(dA, list(range(len(lens))), dB, list(perm), 4096, 1 << 40))
    api.destroy("tensor", dA)
    api.destroy("tensor", dB)
    assert info["kernel_name"] == kernel
