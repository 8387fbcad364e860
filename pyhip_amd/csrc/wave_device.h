// Scans and reductions over the 64 lanes of a wave in the vector ALU.  A shuffle is an LDS operation with its latency
// (about 100 cycles, six of them in a row for a wave-wide result); a DPP move rides in the instruction that uses it.
#pragma once
#include "common.h"

// the value `v` of the lane that the DPP control selects, `old` in the lanes that it leaves out
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ u32 dpp_u32(u32 old, u32 v)
{
    return (u32)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROW_MASK, 0xF, false);
}
#define DPP_ROW_SHR(n) (0x110 + (n))
#define DPP_ROW_BCAST15 0x142
#define DPP_ROW_BCAST31 0x143

// inclusive prefix sum over the lanes: inside the rows of 16, then rows 0 and 2 into 1 and 3, then the lower half into the upper
__device__ __forceinline__ u32 wave_scan_add(u32 v)
{
    v += dpp_u32<DPP_ROW_SHR(1), 0xF>(0, v);
    v += dpp_u32<DPP_ROW_SHR(2), 0xF>(0, v);
    v += dpp_u32<DPP_ROW_SHR(4), 0xF>(0, v);
    v += dpp_u32<DPP_ROW_SHR(8), 0xF>(0, v);
    v += dpp_u32<DPP_ROW_BCAST15, 0xA>(0, v);
    v += dpp_u32<DPP_ROW_BCAST31, 0xC>(0, v);
    return v;
}

// maximum over the lanes (fmaxf's: a NaN loses against a number), the same in every lane
__device__ __forceinline__ float wave_max_dpp(float f)
{
    auto step = [&](auto C, auto M) __attribute__((always_inline)) {
        const u32 v = __builtin_bit_cast(u32, f);
        f = fmaxf(f, __builtin_bit_cast(float, dpp_u32<decltype(C)::value, decltype(M)::value>(v, v)));
    };
    using Rows = std::integral_constant<int, 0xF>;
    step(std::integral_constant<int, DPP_ROW_SHR(1)>{}, Rows{});
    step(std::integral_constant<int, DPP_ROW_SHR(2)>{}, Rows{});
    step(std::integral_constant<int, DPP_ROW_SHR(4)>{}, Rows{});
    step(std::integral_constant<int, DPP_ROW_SHR(8)>{}, Rows{});
    step(std::integral_constant<int, DPP_ROW_BCAST15>{}, std::integral_constant<int, 0xA>{});
    step(std::integral_constant<int, DPP_ROW_BCAST31>{}, std::integral_constant<int, 0xC>{});
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(u32, f), WAVE - 1));
}
