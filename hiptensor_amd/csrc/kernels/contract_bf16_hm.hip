// bf16 kernels with operand tiles of 64 and 128 rows loaded straight into LDS (contract_hm.hpp).
#include "contract_hm.hpp"

namespace hiptk
{
    static const KernelEntry k_entries[] = {
        HIPTK_HM_TILE(TraitsBF16, 13, 64, 64, 4),
        HIPTK_HM_TILE(TraitsBF16, 14, 128, 64, 3),
        HIPTK_HM_TILE(TraitsBF16, 15, 64, 128, 3),
    };

    const KernelEntry* entries_bf16_hm(int* count)
    {
        *count = (int)(sizeof(k_entries) / sizeof(k_entries[0]));
        return k_entries;
    }
}
