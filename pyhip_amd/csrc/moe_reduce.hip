// Top-k reduction of the down-projection output: out[t, :] = sum over slots of in[t, slot, :],
// slots added in index order in fp32, one rounding to the output type at the end
// (what the reference's moe_gemm_final_reduce_bf16 computes, src/contrib/moe_gemm_mxfp4.py:199-282).
//
// ROUTED: the kernel also sees the routing (top-k ids, expert count, expert mask, local token count) and leaves
// out every slot that the sort dropped (id outside [0, experts), masked expert): the down GEMM never wrote those
// slots, so they are neither read nor need to be cleared beforehand.  Rows of tokens past the local count are
// written as zeros.
#include "common.h"

struct ReduceRouting
{
    const int* topk_ids;       // [T, k]
    const int* expert_mask;    // [experts] or null
    const int* num_local_tok;  // device scalar or null
    int experts;
};

// One wave per (token, 64 * PIECES pieces of 16 bytes): everything about the routing is then the same for the whole wave.  Lanes
// 0..7 fetch the ids of eight slots, one ballot says which of them count, and the loop over slots branches on scalar
// bits, so a slot that was dropped costs neither a load nor an addition.  (One thread per piece that read its token's
// ids and mask entries for itself issued sixteen loads, one after the other, for every eight of data.)
// Without a mask or a local token count nearly every slot counts as a rule, and its data could be fetched along with the
// ids (the rows exist in memory whether they were written or not; what a dropped one holds is not looked at).  But a
// caller may drop slots by their ids alone, and an expert-parallel rank of eight that does then reads eight times what
// it needs.  So only calls of up to ALONG_PIECES (4 MiB), where reading every slot takes less than asking first, do.
// Bound: HBM at prefill sizes, latency at decode sizes.  This kernel alone, us, the thread-per-piece kernel / data along with
// the ids / ids first (k slots of H bf16):
//   k = 8, H = 7168, 4001 tokens, one slot in eight kept: by ids 44.5 / 83.2 / 29.7, by a mask 53.7 / - / 30.3
//     all kept: 87.2 / 84.2 / 85.1; 8192 tokens 181.0 / 170.7 / 172.7 (6.1 TB/s)
//     32 tokens (3.5 MiB): all kept 4.27 / 3.87 / 3.87, one in eight 3.78 / 3.71 / 3.58
//     64 tokens (7 MiB): all kept 4.57 / 4.18 / 4.18, one in eight 3.79 / 3.99 / 3.56
//   k = 2, H = 4096, 256 tokens (4 MiB): all kept 3.97 / 3.84 / 4.28, half 3.72 / 3.78 / 3.98
//     512 tokens: all kept 5.42 / 4.58 / 5.04; 4001 tokens 21.4 / 18.2 / 19.7
// In the layer, where the ids come from memory rather than a cache, asking first costs decode sizes 0.1-0.35 us.
#define ALONG_PIECES (1 << 18)
template <bool OUT_F32, bool ROUTED, int PIECES>
__device__ __forceinline__ void topk_reduce(const uint4* __restrict__ in, void* __restrict__ out, long long T, int k, int H8,
                                            const u32* __restrict__ tokens_limit, const ReduceRouting& rt)
{
    if(tokens_limit)
    {
        long long lim = (long long)tokens_limit[1];
        T             = T < lim ? T : lim;
    }
    const int lane   = lane_id();
    const u32 wave   = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const u32 pieces = WAVE * PIECES, chunks = ((u32)H8 + pieces - 1) / pieces;
    // this wave's first (token, chunk) and the step to its next one: no 64-bit division
    const u32 first = blockIdx.x * 4u + wave, step = gridDim.x * 4u;
    const u32 step_t = step / chunks, step_c = step - step_t * chunks;
    long long t = first / chunks;
    u32 ch      = first - (u32)t * chunks;
    const bool ask_first = ROUTED && (rt.expert_mask || rt.num_local_tok || T * k * H8 > ALONG_PIECES);
    long long T_local    = T;
    if(ROUTED && rt.num_local_tok)
    {
        const long long lim = (long long)*rt.num_local_tok;
        T_local             = lim < 0 ? 0 : (lim < T ? lim : T);
    }
    while(t < T)
    {
        int c[PIECES];
        const uint4* p[PIECES];
        float acc[PIECES][8] = {};
#pragma unroll
        for(int q = 0; q < PIECES; q++)
        {
            c[q] = (int)(ch * pieces) + q * WAVE + lane;
            p[q] = in + (t * k) * H8 + (c[q] < H8 ? c[q] : H8 - 1);      // (lanes past the row read its last piece and store nothing)
        }
        for(int s0 = 0; s0 < k; s0 += 8)            // up to 8 independent loads in flight for each piece, added in slot order
        {
            const int n = k - s0 < 8 ? k - s0 : 8;
            u32 on      = (1u << n) - 1u;           // slots that count, the same in every lane
            int e       = -1;
            if(ROUTED && lane < n && t < T_local)
                e = rt.topk_ids[t * k + s0 + lane];
            if(ROUTED && ask_first)
                on = (u32)__ballot(moe_pair_is_kept(e, rt.experts, rt.expert_mask));
            v4i v[PIECES][8];
#pragma unroll
            for(int j = 0; j < 8; j++)
                if((on >> j) & 1u)
#pragma unroll
                    for(int q = 0; q < PIECES; q++)
                        v[q][j] = __builtin_nontemporal_load((const v4i*)(p[q] + (long long)(s0 + j) * H8));
            if(ROUTED && !ask_first)
                on = (u32)__ballot(moe_pair_is_kept(e, rt.experts, nullptr));
#pragma unroll
            for(int j = 0; j < 8; j++)
            {
                // (leaving a slot out is adding +0.0: the sums start at +0.0 and can never become -0.0)
                if(!((on >> j) & 1u))
                    continue;
#pragma unroll
                for(int q = 0; q < PIECES; q++)
#pragma unroll
                    for(int i = 0; i < 4; i++)
                    {
                        acc[q][2 * i] += bf16_bits_to_f32((u32)v[q][j][i] & 0xFFFFu);
                        acc[q][2 * i + 1] += bf16_bits_to_f32((u32)v[q][j][i] >> 16);
                    }
            }
        }
#pragma unroll
        for(int q = 0; q < PIECES; q++)
            if(c[q] < H8)
            {
                const long long id = t * H8 + c[q];
                if(OUT_F32)
                {
                    float4* o = (float4*)out + id * 2;
                    o[0]      = make_float4(acc[q][0], acc[q][1], acc[q][2], acc[q][3]);
                    o[1]      = make_float4(acc[q][4], acc[q][5], acc[q][6], acc[q][7]);
                }
                else
                {
                    uint4 o;
                    o.x = pack_bf16x2(acc[q][0], acc[q][1]);
                    o.y = pack_bf16x2(acc[q][2], acc[q][3]);
                    o.z = pack_bf16x2(acc[q][4], acc[q][5]);
                    o.w = pack_bf16x2(acc[q][6], acc[q][7]);
                    ((uint4*)out)[id] = o;
                }
            }
        t += step_t;
        ch += step_c;
        if(ch >= chunks)
        {
            ch -= chunks;
            t++;
        }
    }
}

template <bool OUT_F32, bool ROUTED>
__global__ void __launch_bounds__(256)
    moe_topk_reduce_kernel(const uint4* __restrict__ in, void* __restrict__ out, long long T, int k, int H8,
                           const u32* __restrict__ tokens_limit, ReduceRouting rt)
{
    topk_reduce<OUT_F32, ROUTED, 1>(in, out, T, k, H8, tokens_limit, rt);
}

// Under an expert mask a wave waits for ids, mask and data one after the other and fetches little: two pieces to a lane share the
// chain.  Layer, us, one / two / four: one of 8 ranks of the DeepSeek-V3 shape, 4001 tokens 209.5 / 206.9 / 209.1, 2000 tokens 166.6 / 164.2 /
// 165.2; one of 4 of the Qwen3 shape, 2000 tokens 93.2 / 91.7 / 92.3.  Without a mask (8192 tokens, 1875 / 1882) and in small calls, whose
// waves are all resident at once (0.2-0.6 us), one is the faster.
template <bool OUT_F32>
__global__ void __launch_bounds__(256)
    moe_topk_reduce_masked_kernel(const uint4* __restrict__ in, void* __restrict__ out, long long T, int k, int H8, ReduceRouting rt)
{
    topk_reduce<OUT_F32, true, 2>(in, out, T, k, H8, nullptr, rt);
}

static int launch_reduce(const char* name, const void* in_bf16, void* out, int64_t tokens, int topk, int hidden,
                         int out_is_f32, const uint32_t* num_valid_ids, const ReduceRouting* rt, hipStream_t stream)
{
    PYHIP_REQUIRE(in_bf16 && out, "%s: null pointer", name);
    PYHIP_REQUIRE(hidden > 0 && hidden % 8 == 0, "%s: hidden=%d must be a multiple of 8", name, hidden);
    PYHIP_REQUIRE(topk >= 1, "%s: topk=%d", name, topk);
    PYHIP_REQUIRE(((uintptr_t)in_bf16 % 16) == 0 && ((uintptr_t)out % 16) == 0, "%s: unaligned pointer", name);
    if(tokens <= 0)
        return PYHIP_OK;
    // a wave for every (token, 64 or 128 pieces of 16 bytes), four to a workgroup; a launch past 65536 workgroups strides
    const bool masked     = rt && rt->expert_mask && (long long)tokens * topk * (hidden / 8) > ALONG_PIECES;
    const int pieces      = WAVE * (masked ? 2 : 1);
    const long long waves = (long long)tokens * ((hidden / 8 + pieces - 1) / pieces);
    long long grid        = (waves + 3) / 4;
    grid                  = grid > 65536 ? 65536 : grid;
    const ReduceRouting none = {nullptr, nullptr, nullptr, 0};
#define REDUCE_LAUNCH(F32, ROUTED)                                                                                  \
    hipLaunchKernelGGL((moe_topk_reduce_kernel<F32, ROUTED>), dim3((unsigned)grid), dim3(256), 0, stream,           \
                       (const uint4*)in_bf16, out, (long long)tokens, topk, hidden / 8, num_valid_ids, rt ? *rt : none)
    if(masked)
    {
        if(out_is_f32)
            hipLaunchKernelGGL((moe_topk_reduce_masked_kernel<true>), dim3((unsigned)grid), dim3(256), 0, stream, (const uint4*)in_bf16, out,
                               (long long)tokens, topk, hidden / 8, *rt);
        else
            hipLaunchKernelGGL((moe_topk_reduce_masked_kernel<false>), dim3((unsigned)grid), dim3(256), 0, stream, (const uint4*)in_bf16, out,
                               (long long)tokens, topk, hidden / 8, *rt);
    }
    else if(rt)
    {
        if(out_is_f32)
            REDUCE_LAUNCH(true, true);
        else
            REDUCE_LAUNCH(false, true);
    }
    else
    {
        if(out_is_f32)
            REDUCE_LAUNCH(true, false);
        else
            REDUCE_LAUNCH(false, false);
    }
#undef REDUCE_LAUNCH
    PYHIP_CHECK_LAUNCH("moe_topk_reduce_kernel");
    return PYHIP_OK;
}

extern "C" int pyhip_moe_topk_reduce(const void* in_bf16, void* out, int64_t tokens, int topk, int hidden,
                                     int out_is_f32, const uint32_t* num_valid_ids, hipStream_t stream)
{
    return launch_reduce("topk_reduce", in_bf16, out, tokens, topk, hidden, out_is_f32, num_valid_ids, nullptr, stream);
}

extern "C" int pyhip_moe_topk_reduce_routed(const void* in_bf16, void* out, int64_t tokens, int topk, int hidden,
                                            int out_is_f32, const int32_t* topk_ids, int experts,
                                            const int32_t* expert_mask, const int32_t* num_local_tokens,
                                            hipStream_t stream)
{
    PYHIP_REQUIRE(topk_ids && experts > 0, "topk_reduce_routed: topk_ids and the expert count are needed");
    const ReduceRouting rt = {topk_ids, expert_mask, num_local_tokens, experts};
    return launch_reduce("topk_reduce_routed", in_bf16, out, tokens, topk, hidden, out_is_f32, nullptr, &rt, stream);
}
