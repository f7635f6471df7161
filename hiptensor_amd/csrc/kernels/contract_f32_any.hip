// f32 kernels whose operand tiles are loaded straight into LDS from any element (contract_wx_kernel, contract_wd.hpp).
#include "contract_wd.hpp"

namespace hiptk
{
    static const KernelEntry k_entries[] = {
        HIPTK_WX_TILE(WTraitsF32, 4, 16, 4, 0),
        HIPTK_WX_TILE(WTraitsF32, 5, 16, 4, 1),
    };

    const KernelEntry* entries_f32_any(int* count)
    {
        *count = (int)(sizeof(k_entries) / sizeof(k_entries[0]));
        return k_entries;
    }
}
