// Exchanges between the lanes of a wave.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cora {

// The value of lane ^ kMask. Masks below 16 within the row of 16 lanes by DPP moves (quad
// permutations, the half mirror and the rotation by 8), the others through the LDS crossbar.
template <uint32_t kMask>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    if constexpr (kMask == 1)
        return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);
    else if constexpr (kMask == 2)
        return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);
    else if constexpr (kMask == 4)  // 7 ^ 3: half mirror, then each quad reversed
        return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true), 0x1B, 0xF,
                                           0xF, true);
    else if constexpr (kMask == 8)
        return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, true);
    else
        return __shfl_xor(v, kMask, 64);
}

}  // namespace cora
