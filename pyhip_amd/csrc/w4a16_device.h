// What the bf16-activation kernels share (moe_gemm_w4a16.hip, moe_gemm_pairs.hip).
#pragma once
#include "common.h"

#define W4A16_THREADS 256

// 32 e2m1 values (4 dwords) times 2^(scale byte - 127) -> four MFMA operands of 8 bf16
__device__ __forceinline__ void expand_fp4(const v4i& w, u32 scale_byte, v8bf (&o)[4])
{
    const float sc = __builtin_bit_cast(float, scale_byte << 23);
#pragma unroll
    for(int i = 0; i < 4; i++)
    {
        const u32 d = (u32)w[i];
        v2bf p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, sc, 0);
        v2bf p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, sc, 1);
        v2bf p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, sc, 2);
        v2bf p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(d, sc, 3);
        o[i] = (v8bf){p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
    }
}

// The K split of a launch of `tiles` tiles of 256 weight rows.  split_k: 0 = decide here, 1 = never, 4 / 16 = always that many
// waves per 64-row tile, 32 = sixteen waves per 32-row tile with three K-steps in flight (down GEMM; the gate_up GEMM takes 16
// instead)
static inline int w4a16_split(int stage, int block_m, int64_t tiles, int K, int split_k)
{
    if(split_k == 0 && tiles < 2048)
        // sixteen waves when the four-way split would still start fewer workgroups than there are CUs and the K loop
        // is long enough to matter (Mixtral shape, one token: the layer 54.0 -> 49.7 us; forced onto the gate_up GEMM as well,
        // which already starts 896 workgroups there, 57.5 us)
        // (the down GEMM then takes the sixteen-wave split on 32-row tiles with three K-steps in flight, split 32:
        // Mixtral shape, one token, the down GEMM 16.9 -> see the measurements in the kernel's comment)
        return (tiles * 4 < 256 && K >= 8192 && block_m == 16) ? (stage == 2 ? 32 : 16) : 4;
    if(stage == 1 && split_k == 32)       // (the 32-row tile exists for the down GEMM: gate_up takes sixteen waves, or four)
        return K >= 2048 ? 16 : 4;
    return split_k == 1 ? 0 : split_k;
}
