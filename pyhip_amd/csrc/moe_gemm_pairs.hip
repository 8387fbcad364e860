// The layer call's GEMMs in blocks of 16 rows (MXFP4 activations: or 32 or 64): few tokens, so the call is a weight stream and a chain of launches.  With bf16
// activations the arithmetic (and with it every bit of the result) is that of moe_gemm_w4a16.hip, with MXFP4 ones that of
// moe_gemm_mxfp4.hip but for the order of the sums (see pairs_tile); their entry points serve callers that run the stages one by one.  What is different is what a call of 20-100 us spends beside its weights:
//   * Up to 128 pairs (token, slot) there is no sort: every wave reads the routing, one or two pairs to a lane, and finds its block's
//     expert and rows with a few ballots (find_block).
//   * Activations come at their own row pitch and width, and neither the padding rows nor the padding columns of the weights
//     are fetched (raw buffer loads: a lane or a row group that has nothing to fetch is out of its descriptor's range).
//   * Where nearly every pair has an expert of its own, the down GEMM goes by token instead of by expert: a workgroup holds
//     all of a token's slots for 16 to 64 output channels, so it sums them and no reduction follows (bf16 activations).
//   * With MXFP4 activations a workgroup is one tile of 64 weight rows, not a persistent loop over tiles that meets a barrier
//     for each K-step, and its waves hold two or three K-steps in flight without LDS between them and the matrix cores.  What is
//     left to save is the vector cache's time for the activations: where a block is full, a gather of its rows costs it more than the weights.
// Bound: the weight stream from about 40 us on, the launches and their latency chains below.  Layer call, us, sort + moe_gemm_w4a16
// kernels + reduction (padded layers: after a widening of the activations) / this: gpt-oss shape, 2 tokens 39.5 / 28.7, 5 tokens
// 67.0 / 51.3 (bound at 6.9 TB/s: 38); 32 experts, top-1, 2144 x 3040, 3 tokens 36.7 / 18.4; 1024 x 512, 8 experts, 10 tokens 25.0 / 17.6;
// Mixtral shape, 5 tokens 100.6 / 94.5, 29 tokens 129.9 / 124.1 (5.75 -> 6.0 TB/s).  MXFP4 activations, sort with quantisation + persistent
// kernels + reduction / this: gpt-oss shape, 16 tokens 121.5 / 108.8 (bound 97.7); Qwen3 shape, 5 tokens 57.7 / 43.0, 30 tokens 88.7 / 77.1;
// DeepSeek-V3 shape, 16 tokens 374.8 / 355.6, 100 tokens 868 / 821 (6.7 -> 7.1 TB/s), 128 tokens, 32-row blocks, 906 / 852; Qwen3
// shape, 180 tokens, 64-row blocks, 158 / 147.
#include "w4a16_device.h"
#include "moe_gemm_pairs.h"

#define AUX_NT 2      // streamed once

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t buffer_of(const void* p, u32 bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ v4i load16(rsrc_t b, int voff, int soff) { return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(b, voff, soff, 0)); }
__device__ __forceinline__ v4i load16_nt(rsrc_t b, int voff, int soff) { return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(b, voff, soff, AUX_NT)); }
__device__ __forceinline__ u32 load4(rsrc_t b, int voff, int soff) { return (u32)__builtin_amdgcn_raw_buffer_load_b32(b, voff, soff, 0); }
#define NOWHERE ((int)0x80000000)      // an offset past every range; OR-ed, so two of them stay one

// local id of an expert under a mask: the experts this rank holds before it
__device__ __forceinline__ int local_expert(int e, const int* mask, int lane)
{
    if(!mask)
        return e;
    int n = 0;
    for(int i0 = 0; i0 < e; i0 += WAVE)
        n += __builtin_popcountll(__ballot(i0 + lane < e && mask[i0 + lane] != 0));
    return __builtin_amdgcn_readfirstlane(n);
}

// Block m_blk of the unsorted call, or false.  Lane p holds pairs p and p + 64; pairs that share an expert are found by a ballot for each
// bit of the expert number; every 16th of them, in pair order, starts a block, and blocks are numbered by the pair that starts them.
// -> expert (local id) and, in lane r of each 16, the pair of the block's row r (-1: no row)
// blocks: how many there are.  TWO: more than 64 pairs.  (The sort's launch in front of the GEMMs costs the host 3.3 us and the device 5-7.  This
// costs every workgroup a few hundred ns, more with two pairs to a lane: see leaves_sort_out in moe_forward.hip for where that pays.  So
// gate_up leaves what it has found to the down GEMM: Qwen3 shape, 8 tokens, 47.3 -> 46.7; Mixtral shape, 29 tokens, 121.2 -> 119.9; 96 experts, top-4, 16
// tokens 61.7 -> 60.0.)
template <bool TWO>
__device__ __forceinline__ bool find_block(const PairArgs& g, int m_blk, int lane, int& e, int& pair, int& blocks)
{
    constexpr int H = TWO ? 2 : 1;
    int n = g.T * g.topk;
    if(g.local_tok)
    {
        const int lim = *g.local_tok;
        n             = lim < 0 ? 0 : lim < g.T ? lim * g.topk : n;
    }
    int id[H];
    bool kept[H];
    u64 same[H][H];      // [of the lane's pair h][among pairs 64 * i ..]
#pragma unroll
    for(int h = 0; h < H; h++)
        id[h] = h * WAVE + lane < n ? g.ids[h * WAVE + lane] : -1;
#pragma unroll
    for(int h = 0; h < H; h++)
        kept[h] = moe_pair_is_kept(id[h], g.experts, g.mask);
#pragma unroll
    for(int h = 0; h < H; h++)
#pragma unroll
        for(int i = 0; i < H; i++)
            same[h][i] = __ballot(kept[i]);
    for(int b = 0; (g.experts - 1) >> b; b++)
    {
        u64 s[H];
#pragma unroll
        for(int i = 0; i < H; i++)
            s[i] = __ballot((id[i] >> b) & 1);
#pragma unroll
        for(int h = 0; h < H; h++)
#pragma unroll
            for(int i = 0; i < H; i++)
                same[h][i] &= (id[h] >> b) & 1 ? s[i] : ~s[i];
    }
    const u64 below = (1ull << lane) - 1ull;
    u64 hits[H];
    blocks = 0;
#pragma unroll
    for(int h = 0; h < H; h++)
    {
        const int rank   = (h ? __builtin_popcountll(same[h][0]) : 0) + __builtin_popcountll(same[h][h] & below);
        const bool start = kept[h] && (rank & 15) == 0;
        const u64 starts = __ballot(start);
        hits[h]          = __ballot(start && blocks + __builtin_popcountll(starts & below) == m_blk);
        blocks += __builtin_popcountll(starts);
    }
    // (straight on from here: a loop over h with a way out in it is left a loop, and same[][] then lies in scratch memory to be indexed)
    const bool second = TWO && !hits[0];      // which word the pair that starts the block is in
    const u64 hit     = second ? hits[H - 1] : hits[0];
    if(!hit)
        return false;
    const int lead = __builtin_ctzll(hit);
    auto of_lead = [&](u64 v) __attribute__((always_inline)) -> u64 {
        return (u64)(u32)__builtin_amdgcn_readlane((int)v, lead) | (u64)(u32)__builtin_amdgcn_readlane((int)(v >> 32), lead) << 32;
    };
    // the pairs of its expert from that one on
    const u64 from = ~((1ull << lead) - 1ull);
    u64 row0 = second ? 0ull : of_lead(same[0][0]) & from;
    u64 row1 = !TWO ? 0ull : second ? of_lead(same[H - 1][H - 1]) & from : of_lead(same[0][H - 1]);
    e    = local_expert(__builtin_amdgcn_readlane(second ? id[H - 1] : id[0], lead), g.mask, lane);
    pair = -1;
    for(int r = 0; r < 16; r++)
    {
        int p = -1;
        if(row0)
        {
            p = __builtin_ctzll(row0);
            row0 &= row0 - 1ull;
        }
        else if(row1)
        {
            p = WAVE + __builtin_ctzll(row1);
            row1 &= row1 - 1ull;
        }
        if(p < 0)
            break;
        pair = (lane & 15) == r ? p : pair;
    }
    return true;
}

// the lane's four biases of channels c .. c + 3 (element-aligned tensors: one by one)
__device__ __forceinline__ uint2 load_bias4(const uint16_t* b)
{
    if(((unsigned long long)b & 7) == 0)
        return *(const uint2*)b;
    return make_uint2((u32)b[0] | (u32)b[1] << 16, (u32)b[2] | (u32)b[3] << 16);
}
__device__ __forceinline__ v4f add_bias4(v4f v, uint2 b)
{
    v[0] += bf16_bits_to_f32(b.x & 0xFFFFu);
    v[1] += bf16_bits_to_f32(b.x >> 16);
    v[2] += bf16_bits_to_f32(b.y & 0xFFFFu);
    v[3] += bf16_bits_to_f32(b.y >> 16);
    return v;
}

// 32 bf16 of a row (a lane's K-elements of a K-step, which are one MX block) as the quantiser gives them (quant_device.h): eight e2m1
// codes to a dword, and the block's scale byte
__device__ __forceinline__ void quantise32(const v4i (&x)[4], v4i& q, int& e8)
{
    u32 am = 0;
#pragma unroll
    for(int i = 0; i < 4; i++)
#pragma unroll
        for(int c = 0; c < 4; c++)
            am = amax15x2(am, (u32)x[i][c]);
    const u32 s = mx_scale_byte(amax15_fold(am));
#pragma unroll
    for(int i = 0; i < 4; i++)
        q[i] = (int)cvt8(__builtin_bit_cast(uint4, x[i]), s);
    e8 = (int)s;
}
// acc += W(16 rows x 128 K, e2m1) * A(128 K x 16 rows, e2m1), scales in the low bytes
__device__ __forceinline__ v4f mfma_fp4(const v4i& w, int ws, const v4i& a, int as, const v4f& acc)
{
    const v8i w8 = {w.x, w.y, w.z, w.w, 0, 0, 0, 0}, a8 = {a.x, a.y, a.z, a.w, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w8, a8, acc, 4, 4, 0, ws, 0, as);
}

// STAGE 1 = gate_up (+ the gated activation), 2 = down (* routing weight).  SPLIT 0: a wave owns 64 weight rows over the whole K;
// 4: the four waves share 64 weight rows, wave w takes K-steps w, w + 4, .. and the partial sums meet in LDS.
// NB K-steps of operands are in flight; a register set is refilled as soon as its MFMAs are issued.
// ACT: the activations are BF16 (their products with the weights expanded to bf16), or MXFP4, quantised by whoever wrote them (QUANTISED)
// or on the way to the matrix cores (TO_FP4: 40 instructions a K-step, where expanding the weights takes 64).  With MXFP4 the products are
// multiples of powers of two.  While the block scales along a row span a few bits, as those of N(0, 1) data do, 32-bit sums hold them exactly
// in whatever order, and the bits are those of moe_gemm_mxfp4.hip; with channels that stand far out (factors of 1000 between blocks) four
// partial sums and one chain are rounded at different places, and differ in the last bits.  The gate_up GEMM
// quantises its result as that one does: a workgroup's 32 channels are one MX block of a row, which wave 0 finishes.
enum { BF16, TO_FP4, QUANTISED };
template <int STAGE, int SPLIT, int ACT, bool STAGED, int BT, int MT>
__device__ __forceinline__ void pairs_tile(const PairArgs& g, float* red, int lane, int wave, int m_blk, int nt, int e,
                                           const int* arow, const int* orow, const float* rw)
{
    constexpr bool SPLITK = SPLIT != 0;
    static_assert(SPLITK || ACT == BF16, "MXFP4 activations: the four waves split K");
    static_assert(!STAGED || (ACT == BF16 && MT == 1), "staged: bf16 rows");
    static_assert(BT == 1 || ACT == QUANTISED, "several row tiles: activations that take few registers");
    // (bf16 activations take 16 registers a K-step: two K-steps in flight and four waves per SIMD, not three and three.  Layer, us, three / two: 60
    // experts, 2048 x 1408, 10 tokens 31.8 / 29.4, 50 tokens 57.7 / 53.4; 28, 2048 x 4096, 20 tokens 75.9 / 71.4; 24, 2048 x 2048, 12 tokens 33.2 / 29.8;
    // Mixtral shape, 20 tokens 118.5 / 117.5; 32, 2880 x 2880, 10 tokens 54.5 / 55.1.  Staged, four waves do not fit without spilling.)
    constexpr int NB = (ACT == BF16 && !STAGED) || (BT > 1 && MT > 1) ? 2 : 3, KSTRIDE = SPLITK ? 4 : 1;
    constexpr int NA = ACT == QUANTISED ? 1 : 4;                  // 16-byte pieces of a row in a lane's K-step
    const int r = lane & 15, kb = lane >> 4;
    const int Kb = g.K / 2, I = g.N / 2;
    // first output channel of this wave's rows (stage 1: within the gate half; the up half is I further)
    const int chbase = STAGE == 1 ? (SPLITK ? nt * 32 : nt * 128 + wave * 32) : (SPLITK ? nt * 64 : nt * 256 + wave * 64);
    if(STAGE == 1 && chbase >= I - g.n_pad && !g.all_channels)      // (channels of padding: the down GEMM does not read them)
        return;
    // row group j = 0..3 (stage 1: 0, 1 gate rows, 2, 3 the matching up rows); two of them share a scale tile of 32 rows
    const u32 sc_tile = (u32)(g.SC / 8) * 256u;
    rsrc_t wb[4], sb[2];
    auto row_of = [&](int j) __attribute__((always_inline)) -> u32 {
        return (u32)e * (u32)g.N + (u32)(STAGE == 1 ? (j >> 1) * I + chbase + (j & 1) * 16 : chbase + j * 16);
    };
    auto is_real = [&](int j) __attribute__((always_inline)) -> bool {
        return STAGE == 1 ? chbase + (j & 1) * 16 < I - g.n_pad : chbase + j * 16 < g.N - g.n_pad;
    };
#pragma unroll
    for(int j = 0; j < 4; j++)
        wb[j] = buffer_of(g.w + (size_t)row_of(j) * Kb, is_real(j) ? (u32)(16 * Kb) : 0u);
#pragma unroll
    for(int h = 0; h < 2; h++)
        sb[h] = buffer_of(g.w_s + (size_t)(row_of(2 * h) / 32) * sc_tile, sc_tile);
    const rsrc_t ab = buffer_of(g.a, g.a_bytes), asb = buffer_of(g.a_s, g.as_bytes);
    const int SK     = (g.K + 511) / 512 * 16;      // bytes of a row's scales (moe_quant.hip)
    // gate_up: quantised tokens are fetched with a row's four groups of 32 in adjacent lanes, and change places on their way to the
    // matrix cores: 64 bytes to four lanes are one access of the vector cache, 16 bytes of four rows are four.  The down GEMM's
    // operand lies as its lanes read it: [16-row tile][K-step][lane][16 bytes], and scales [tile][4 K-steps][lane][a byte for each].
    // Qwen3 shape, 128 tokens in 16-row blocks, rows fetched as they lie / the first / both: 160.9 / 156.8 / 151.8 us; DeepSeek-V3 shape,
    // 200 tokens: 909.5 / 903.6 / 879.3.
    constexpr bool SWAP = ACT == QUANTISED && STAGE == 1, TILES = ACT == QUANTISED && STAGE == 2;
    const int lk = SWAP ? lane & 3 : kb, from = (r * 4 + kb) * 4;
    int a_off[MT], as_off[MT];
#pragma unroll
    for(int m = 0; m < MT; m++)
    {
        const int row = SWAP ? __builtin_amdgcn_ds_bpermute((lane >> 2) * 4, arow[m]) : arow[m], tile = m_blk * BT + m;
        a_off[m]      = row < 0 ? NOWHERE : TILES ? tile * 16 * Kb + lane * 16 : SWAP ? row * Kb + lk * 16 : row * g.a_pitch * 2 + kb * 64;
        as_off[m]     = row < 0 ? NOWHERE : TILES ? tile * 16 * SK + lane * 4 : row * SK + lk * 4;
    }

    // Staged bf16 rows: a load fetches 256 bytes of each of four rows, 16 lanes to a row; a K-step's four loads are written to the wave's own
    // 4 KB of LDS and read back as the matrix cores want them, piece p of row r at r * 16 + (p ^ r) (no two of eight lanes in a bank).
    // As the rows lie, a load is 64 accesses of the vector cache, four times what the weights of a K-step cost it.
    int st_off[4];
    v4i* const mine = (v4i*)red + wave * 256;
    if constexpr(STAGED)
#pragma unroll
        for(int i = 0; i < 4; i++)
        {
            const int row = __builtin_amdgcn_ds_bpermute((i * 4 + kb) * 4, arow[0]);
            st_off[i]     = row < 0 ? NOWHERE : row * g.a_pitch * 2 + r * 16;
        }
    v4f acc[4][MT];
#pragma unroll
    for(int j = 0; j < 4; j++)
#pragma unroll
        for(int m = 0; m < MT; m++)
            acc[j][m] = (v4f){0.f, 0.f, 0.f, 0.f};
    const int KT = (g.k_real + 127) / 128;
    v4i wf[NB][4], af[NB][MT][NA];
    u32 wsc[NB][2], asc[NB][MT];
    auto load_step = [&](auto BB, int kt) __attribute__((always_inline)) {
        constexpr int b = decltype(BB)::value;
        const int away  = kt * 128 + kb * 32 >= g.k_real ? NOWHERE : 0;
        const int aaway = kt * 128 + (STAGED ? r >> 2 : lk) * 32 >= g.k_real ? NOWHERE : 0;
#pragma unroll
        for(int h = 0; h < 2; h++)
            wsc[b][h] = load4(sb[h], lane * 4 | away, (kt >> 1) * 256);
#pragma unroll
        for(int j = 0; j < 4; j++)
            wf[b][j] = load16_nt(wb[j], lane * 16 | away, kt * 1024);
#pragma unroll
        for(int m = 0; m < MT; m++)
        {
#pragma unroll
            for(int i = 0; i < NA; i++)
                af[b][m][i] = STAGED ? load16(ab, st_off[i] | aaway, kt * 256) : load16(ab, (a_off[m] + i * 16) | aaway, kt * (TILES ? 1024 : 64 * NA));
            if constexpr(ACT == QUANTISED)
                asc[b][m] = load4(asb, as_off[m] | aaway, (kt >> 2) * (TILES ? 256 : 16));
        }
    };
    auto step = [&](auto BB, int kt) __attribute__((always_inline)) {
        constexpr int b = decltype(BB)::value;
        if constexpr(STAGED)
        {
#pragma unroll
            for(int i = 0; i < 4; i++)
                mine[(i * 4 + kb) * 16 + (r ^ (i * 4 + kb))] = af[b][0][i];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for(int i = 0; i < 4; i++)
                af[b][0][i] = mine[r * 16 + ((kb * 4 + i) ^ r)];
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for(int m = 0; m < MT; m++)
        {
            v4i aq;
            int as;
            if constexpr(ACT == TO_FP4)
                quantise32(af[b][m], aq, as);
            else if constexpr(ACT == QUANTISED)
            {
                aq = af[b][m][0];
                as = (int)asc[b][m];
                if constexpr(SWAP)
                {
#pragma unroll
                    for(int i = 0; i < 4; i++)
                        aq[i] = __builtin_amdgcn_ds_bpermute(from, aq[i]);
                    as = __builtin_amdgcn_ds_bpermute(from, as);
                }
                as >>= 8 * (kt & 3);
            }
#pragma unroll
            for(int j = 0; j < 4; j++)
            {
                const u32 ws = wsc[b][j >> 1] >> (8 * ((kt & 1) * 2 + (j & 1)));
                if constexpr(ACT != BF16)
                    acc[j][m] = mfma_fp4(wf[b][j], (int)ws, aq, as, acc[j][m]);
                else
                {
                    v8bf wq[4];
                    expand_fp4(wf[b][j], ws & 0xFFu, wq);
#pragma unroll
                    for(int i = 0; i < 4; i++)
                        acc[j][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wq[i], __builtin_bit_cast(v8bf, af[b][m][i]), acc[j][m], 0, 0, 0);
                }
            }
        }
    };
    // (the loads carry no condition: K-steps past the last one are out of range.  A branch around them costs the loop its prefetch
    // distance: the register sets then meet in copies, which wait for what is in flight.  So does a scheduler that moves a K-step's
    // loads behind the next one's waits: gpt-oss shape, 16 tokens, MXFP4, 132.7 us with both, 108.2 without.)
    const int kt0 = SPLITK ? wave : 0;
    static_for<NB>([&](auto BB) __attribute__((always_inline)) {
        load_step(BB, kt0 + decltype(BB)::value * KSTRIDE);
        __builtin_amdgcn_sched_barrier(0);
    });
    int kt = kt0;
    for(; kt + NB * KSTRIDE < KT; kt += NB * KSTRIDE)
        static_for<NB>([&](auto BB) __attribute__((always_inline)) {
            step(BB, kt + decltype(BB)::value * KSTRIDE);
            __builtin_amdgcn_sched_barrier(0);
            load_step(BB, kt + (decltype(BB)::value + NB) * KSTRIDE);
            __builtin_amdgcn_sched_barrier(0);
        });
    static_for<NB>([&](auto BB) __attribute__((always_inline)) {
        if(kt + decltype(BB)::value * KSTRIDE < KT)
            step(BB, kt + decltype(BB)::value * KSTRIDE);
    });

    // ---- epilogue: lane (r, kb) holds channels kb*4 .. + 3 of row group j for row r.  Under the K split wave w finishes row
    // group w (stage 1: gate group w and its up group, waves 0 and 1; where the result is quantised wave m finishes row tile m)
    auto channel = [&](int j) __attribute__((always_inline)) -> int {
        return (STAGE == 1 ? (j >> 1) * I + chbase + (j & 1) * 16 : chbase + j * 16) + kb * 4;
    };
    auto with_bias = [&](int j, v4f v) __attribute__((always_inline)) -> v4f {
        return g.bias ? add_bias4(v, load_bias4(g.bias + (size_t)e * g.N + channel(j))) : v;
    };
    auto finish = [&](int j, int m, v4f lo, v4f hi) __attribute__((always_inline)) {      // hi: stage 1, the up group
        lo = with_bias(j, lo);
        if(STAGE == 1)
            hi = with_bias(j + 2, hi);
        if(arow[m] < 0)
            return;
        float v[4];
#pragma unroll
        for(int i = 0; i < 4; i++)
            v[i] = STAGE == 1 ? gated_act_f32(g.act, lo[i], hi[i]) : lo[i] * rw[m];
        *(uint2*)((uint16_t*)g.out + (size_t)orow[m] * (STAGE == 1 ? I : g.N) + channel(j)) =
            make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    };
    // as the epilogue of the persistent kernels (gemm_device.h), with the same functions: round to bf16, eight consecutive channels to a lane, the block's maximum
    // over the lane rows, e2m1 codes and the scale byte.  x: the sums of row tile m, a row group each
    auto quantise_row = [&](const v4f (&x)[4], int m, bool here) __attribute__((always_inline)) {
        u32 d[2][2];
#pragma unroll
        for(int j = 0; j < 2; j++)
        {
            const v4f lo = with_bias(j, x[j]), hi = with_bias(j + 2, x[j + 2]);
            float v[4];
#pragma unroll
            for(int i = 0; i < 4; i++)
                v[i] = g.swiglu ? swiglu_f32(lo[i], hi[i], g.act.limit) : silu_f32(lo[i]) * hi[i];
            d[j][0] = pack_bf16x2(v[0], v[1]);
            d[j][1] = pack_bf16x2(v[2], v[3]);
        }
        const uint4 o = join_channels8(d);
        const u32 e8  = mx_scale_of_row(o);
        if(here)
        {
            const int blk = chbase / 32, kt = blk / 4;
            const size_t at = (size_t)(m_blk * BT + m) * (I / 128) + kt, lane2 = (blk & 3) * 16 + r;
            *(u32*)((uint8_t*)g.out + (at * WAVE + lane2) * 16 + (kb & 1) * 8 + (kb >> 1) * 4) = cvt8(o, e8);
            if(kb == 0)
                g.out_s[((at / 4) * WAVE + lane2) * 4 + (kt & 3)] = (uint8_t)e8;
        }
    };
    if constexpr(SPLITK)
    {
        // (two row tiles at a time, in 32 KB)
        constexpr int MR = MT < 2 ? MT : 2;
#pragma unroll
        for(int m0 = 0; m0 < MT; m0 += MR)
        {
            if(m0)
                __syncthreads();
#pragma unroll
            for(int j = 0; j < 4; j++)
#pragma unroll
                for(int m = 0; m < MR; m++)
                    if(m0 + m < MT)
                        *(v4f*)&red[(((wave * 4 + j) * MR + m) * WAVE + lane) * 4] = acc[j][m0 + m];
            __syncthreads();
            auto sum_of = [&](int j, int m) __attribute__((always_inline)) -> v4f {
                v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for(int w = 0; w < 4; w++)
                    sum += *(const v4f*)&red[(((w * 4 + j) * MR + m) * WAVE + lane) * 4];
                return sum;
            };
            if constexpr(STAGE == 1 && ACT != BF16)
            {
                if(wave < MR && m0 + wave < MT)
                {
                    const v4f x[4] = {sum_of(0, wave), sum_of(1, wave), sum_of(2, wave), sum_of(3, wave)};
                    bool here      = arow[m0] >= 0;
                    if(MR == 2 && m0 + 1 < MT && wave == 1)
                        here = arow[m0 + 1] >= 0;
                    quantise_row(x, m0 + wave, here);
                }
            }
            else if(STAGE == 2 || wave < 2)
#pragma unroll
                for(int m = 0; m < MR; m++)
                    if(m0 + m < MT)
                        finish(wave, m0 + m, sum_of(wave, m), STAGE == 1 ? sum_of(wave + 2, m) : (v4f){0.f, 0.f, 0.f, 0.f});
        }
    }
    else
#pragma unroll
        for(int j = 0; j < (STAGE == 1 ? 2 : 4); j++)
            finish(j, 0, acc[j][0], acc[STAGE == 1 ? j + 2 : j][0]);
}

// BT: 16-row tiles of a block.  The real rows of a block come first; what a block computes are the row tiles that have any.
template <int STAGE, int SPLIT, int ACT, int BT = 1, bool STAGED = false>
__global__ void __launch_bounds__(W4A16_THREADS, ACT == BF16 && !STAGED ? 4 : BT > 1 || STAGED ? 3 : 1) moe_gemm_pairs_kernel(PairArgs g)
{
    // [wave][row group][row tile][lane][4]; staged rows: [wave][row][16 pieces of 16 bytes]
    __shared__ __attribute__((aligned(16))) float red[SPLIT || STAGED ? 4 * 4 * (BT < 2 ? 1 : 2) * WAVE * 4 : 1];
    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int r = lane & 15;
    const int m_blk = blockIdx.x / g.n_tiles, nt = blockIdx.x - m_blk * g.n_tiles;
    // the block's expert, and for row r: the activation row, the output row, the routing weight
    int e, arow[BT], orow[BT];
    float rw[BT];
#pragma unroll
    for(int m = 0; m < BT; m++)
    {
        arow[m] = -1;
        orow[m] = -1;      // (as arow: the same registers in the sorted down GEMM, whose 64-row blocks would spill two otherwise)
        rw[m]   = 0.f;
    }
    if(BT == 1 && g.ids)
    {
        int pair, blocks;
        const bool found = g.T * g.topk > WAVE ? find_block<true>(g, m_blk, lane, e, pair, blocks) : find_block<false>(g, m_blk, lane, e, pair, blocks);
        if(STAGE == 1 && nt == 0 && wave == 0 && g.tab_ids)
        {
            // for the down GEMM, as the sort would have written it
            if(m_blk == 0 && lane == 0)
                g.tab_valid[0] = (u32)(blocks * 16);
            if(found && lane < 16)
            {
                const int tok              = (int)((u32)pair / (u32)g.topk);
                g.tab_ids[m_blk * 16 + lane] = pair < 0 ? ~0u : (u32)tok | (u32)(pair - tok * g.topk) << 24;
                g.tab_w[m_blk * 16 + lane]   = pair < 0 ? 0.f : g.weights[pair];
                if(lane == 0)
                    g.tab_e[m_blk] = (u32)e;
            }
        }
        if(!found)
            return;
        if(pair >= 0)
        {
            arow[0] = STAGE == 1 ? (int)((u32)pair / (u32)g.topk) : pair * g.row_step;
            orow[0] = STAGE == 1 ? pair * g.row_step : pair;
            if(STAGE == 2)
                rw[0] = g.weights[pair];
        }
    }
    else
    {
        // (all read together: the arrays are there for every block that is launched, whether or not it holds rows)
        const u32 last = g.num_valid[0];
        e              = __builtin_amdgcn_readfirstlane((int)g.sorted_e[m_blk]);
        u32 id[BT];
#pragma unroll
        for(int m = 0; m < BT; m++)
        {
            const int p = (m_blk * BT + m) * 16 + r;
            id[m]       = g.sorted_ids[p];
            if(STAGE == 2)
                rw[m] = g.sorted_w[p];
        }
        if((u32)(m_blk * BT * 16) >= last)
            return;
#pragma unroll
        for(int m = 0; m < BT; m++)
        {
            const int tok = (int)(id[m] & 0xFFFFFFu), slot = (int)(id[m] >> 24);
            if(slot < g.topk && tok < g.T)
            {
                const int pair = tok * g.topk + slot;
                arow[m]        = STAGE == 1 ? tok : pair;
                orow[m]        = pair;
            }
        }
    }
    // (a mask with more entries than there are matrices, one that is still being written for instance: no weights past their tensor)
    if((u32)e >= (u32)g.held)
        return;
    if constexpr(BT == 1)
        pairs_tile<STAGE, SPLIT, ACT, STAGED, 1, 1>(g, red, lane, wave, m_blk, nt, e, arow, orow, rw);
    else
    {
        int tiles = 1;
#pragma unroll
        for(int m = 1; m < BT; m++)
            tiles = __ballot(arow[m] >= 0) ? m + 1 : tiles;
        if(tiles == 1)
            pairs_tile<STAGE, SPLIT, ACT, STAGED, BT, 1>(g, red, lane, wave, m_blk, nt, e, arow, orow, rw);
        else if(BT == 2 || tiles == 2)
            pairs_tile<STAGE, SPLIT, ACT, STAGED, BT, 2>(g, red, lane, wave, m_blk, nt, e, arow, orow, rw);
        else if(BT == 4 && tiles == 3)
            pairs_tile<STAGE, SPLIT, ACT, STAGED, BT, BT == 4 ? 3 : 2>(g, red, lane, wave, m_blk, nt, e, arow, orow, rw);
        else
            pairs_tile<STAGE, SPLIT, ACT, STAGED, BT, BT>(g, red, lane, wave, m_blk, nt, e, arow, orow, rw);
    }
}

// The down GEMM by token, with the sum over the token's slots.  A workgroup owns NR groups of 16 output channels of one token: groups
// of four waves, a K split each (wave w: K-steps w, w + 4, ..), take the token's slots in turns, one after the other in one pipeline.
// Partial sums, biases and routing weights meet in LDS, where a thread per channel finishes slot after slot: the arithmetic and
// order of moe_gemm_pairs_kernel<2, 4> and the reduction.
// Bound: the weight stream, less well fed than by expert (a wave brings the activations of one row for 1, 2 or 4 KB of weights),
// against the reduction's launch.  Layer, us, down by expert + reduction / NR = 1 / 2 / 4: gpt-oss shape, 1 token 21.9 / 19.3 / 20.8 /
// 24.0, 2 tokens 26.8 / 28.2 / 25.1 / 28.3, 4 tokens 41.7 / 50.3 / 43.1 / 40.5; DeepSeek-V3 shape, 1 token 37.2 / 39.8 / 35.3 / 38.7, 2 tokens
// 61.2 / 71.0 / 61.9 / 58.9, 3 tokens 87.7 / 104.5 / 89.8 / 89.9, 4 tokens 111.5 / 128 / 115.6 / 111.2; 256 experts, top-1, 5120 x 1536,
// 30 tokens 62.1 / 67.0 / 59.9 / 56.7.  (Sixteen waves, every slot on waves of its own: 113 us at 3 tokens of the DeepSeek-V3 shape.)
template <int NR>
__global__ void __launch_bounds__(512) moe_pairs_down_sum_kernel(PairArgs g)
{
    constexpr int NB = NR == 4 ? 2 : 3;      // K-steps in flight
    __shared__ float red[8][4][NR * 16], bias_l[8][NR * 16], rw_l[8];
    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int w = wave & 3, q = wave >> 2, groups = blockDim.x / (4 * WAVE);
    const int r = lane & 15, kb = lane >> 4;
    const int t = blockIdx.x / g.n_tiles, ch0 = (blockIdx.x - t * g.n_tiles) * (16 * NR);
    const int Kb = g.K / 2;
    const u32 sc_tile = (u32)(g.SC / 8) * 256u;
    // lane s: slot s's expert
    const bool here = !(g.local_tok && t >= *g.local_tok);
    const int id    = here && lane < g.topk ? g.ids[t * g.topk + lane] : -1;
    u32 on          = (u32)__ballot(moe_pair_is_kept(id, g.experts, g.mask));
    if(g.mask)      // (no weights past their tensor, see moe_gemm_pairs_kernel)
        for(u32 rest = on; rest; rest &= rest - 1u)
            if(local_expert(__builtin_amdgcn_readlane(id, __builtin_ctz(rest)), g.mask, lane) >= g.held)
                on &= ~(rest & -rest);
    u32 turn = 0;                         // this group's slots: in turns, of those that count
    {
        int i = 0;
        for(u32 rest = on; rest; rest &= rest - 1u, i++)
            if(i % groups == q)
                turn |= rest & -rest;
    }
    const rsrc_t ab = buffer_of(g.a, g.a_bytes);
    const int KT = (g.k_real + 127) / 128, steps = (KT - w + 3) / 4;
    const int half = NR == 1 ? (ch0 / 16) & 1 : 0;      // which half of the 32-row scale tile the first row group is
    constexpr int NS = (NR + 1) / 2;      // scale tiles of 32 rows
    rsrc_t wb[NR], sb[NS];
    int a_off, lk = w, ls = 0;
    u32 to_load = turn;
    auto take_slot = [&]() __attribute__((always_inline)) {
        ls = __builtin_ctz(to_load);
        const int e   = local_expert(__builtin_amdgcn_readlane(id, ls), g.mask, lane);
        const u32 row = (u32)e * (u32)g.N + (u32)ch0;
#pragma unroll
        for(int j = 0; j < NR; j++)
            wb[j] = buffer_of(g.w + (size_t)(row + j * 16) * Kb, ch0 + j * 16 < g.N - g.n_pad ? (u32)(16 * Kb) : 0u);
#pragma unroll
        for(int h = 0; h < NS; h++)
            sb[h] = buffer_of(g.w_s + (size_t)(row / 32 + h) * sc_tile, sc_tile);
        const int pair = t * g.topk + ls;
        a_off = r == 0 ? pair * g.row_step * g.a_pitch * 2 + kb * 64 : NOWHERE;      // (row 0 of the products is the token)
    };
    v4f acc[NR];
#pragma unroll
    for(int j = 0; j < NR; j++)
        acc[j] = (v4f){0.f, 0.f, 0.f, 0.f};
    v4i wf[NB][NR], af[NB][4];
    u32 wsc[NB][NS];
    auto load_next = [&](auto BB) __attribute__((always_inline)) {
        constexpr int b = decltype(BB)::value;
        // (no condition around the loads, see moe_gemm_pairs_kernel)
        const int away = !to_load || lk * 128 + kb * 32 >= g.k_real ? NOWHERE : 0;
#pragma unroll
        for(int h = 0; h < NS; h++)
            wsc[b][h] = load4(sb[h], lane * 4 | away, (lk >> 1) * 256);
#pragma unroll
        for(int j = 0; j < NR; j++)
            wf[b][j] = load16_nt(wb[j], lane * 16 | away, lk * 1024);
#pragma unroll
        for(int c = 0; c < 4; c++)
            af[b][c] = load16(ab, (a_off + c * 16) | away, lk * 256);
        lk += 4;
        if(lk >= KT && to_load)
        {
            lk = w;
            to_load &= to_load - 1u;
            if(to_load)
                take_slot();
        }
    };
    if(turn && steps > 0)
    {
        take_slot();
        static_for<NB>([&](auto BB) __attribute__((always_inline)) {
            load_next(BB);
            __builtin_amdgcn_sched_barrier(0);
        });
        u32 mine = turn;
        int kt = w;
        auto step = [&](auto BB) __attribute__((always_inline)) {
            constexpr int b = decltype(BB)::value;
#pragma unroll
            for(int j = 0; j < NR; j++)
            {
                v8bf wq[4];
                expand_fp4(wf[b][j], (wsc[b][j / 2] >> (8 * ((kt & 1) * 2 + half + (j & 1)))) & 0xFFu, wq);
#pragma unroll
                for(int c = 0; c < 4; c++)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wq[c], __builtin_bit_cast(v8bf, af[b][c]), acc[j], 0, 0, 0);
            }
            kt += 4;
            if(kt >= KT)
            {
                kt = w;
                const int s = __builtin_ctz(mine);
                mine &= mine - 1u;
#pragma unroll
                for(int j = 0; j < NR; j++)
                {
                    if(r == 0)
                        *(v4f*)&red[s][w][j * 16 + kb * 4] = acc[j];
                    acc[j] = (v4f){0.f, 0.f, 0.f, 0.f};
                }
            }
        };
        int left = __builtin_popcount(turn) * steps;
        for(; left > NB; left -= NB)
            static_for<NB>([&](auto BB) __attribute__((always_inline)) {
                step(BB);
                __builtin_amdgcn_sched_barrier(0);
                load_next(BB);
                __builtin_amdgcn_sched_barrier(0);
            });
        static_for<NB>([&](auto BB) __attribute__((always_inline)) {
            if(left > decltype(BB)::value)
                step(BB);
        });
    }
    else if(turn)
        for(u32 m = turn; m; m &= m - 1u)      // (fewer K-steps than waves)
        {
            const int s = __builtin_ctz(m);
            if(r == 0)
#pragma unroll
                for(int j = 0; j < NR; j++)
                    *(v4f*)&red[s][w][j * 16 + kb * 4] = acc[j];
        }
    // (asked for here and not at the start, where the wait for them would hold the weights up)
    if(w == 0)
        for(u32 m = turn; m; m &= m - 1u)
        {
            const int s = __builtin_ctz(m);
            const int e = g.bias ? local_expert(__builtin_amdgcn_readlane(id, s), g.mask, lane) : 0;
            if(lane == 0)
                rw_l[s] = g.weights[t * g.topk + s];
            if(g.bias && lane < 16 * NR)
                bias_l[s][lane] = bf16_bits_to_f32(g.bias[(size_t)e * g.N + ch0 + lane]);
        }
    __syncthreads();
    if(tid >= 16 * NR)
        return;
    float out = 0.f;
    for(u32 m = on; m; m &= m - 1u)
    {
        const int s = __builtin_ctz(m);
        float sum   = 0.f;
#pragma unroll
        for(int p = 0; p < 4; p++)
            sum += red[s][p][tid];
        if(g.bias)
            sum += bias_l[s][tid];
        out += bf16_bits_to_f32(pack_bf16x2(sum * rw_l[s], 0.f) & 0xFFFFu);
    }
    const size_t at = (size_t)t * g.N + ch0 + tid;
    if(g.out_f32)
        ((float*)g.out)[at] = out;
    else
        ((uint16_t*)g.out)[at] = (uint16_t)pack_bf16x2(out, 0.f);
}

// the bound of the row blocks that hold rows, as the sorted entry points compute it: the K split depends on it
static int64_t block_bound(int64_t rows, int64_t n_blk, int experts)
{
    const int64_t b = rows < n_blk ? rows : n_blk;
    return experts + rows / 16 < b ? experts + rows / 16 : b;
}

// bf16 activations: the K split of the sorted entry points, so that the sums are theirs.  MXFP4 ones, whose sums are exact or as good in either
// order: always four waves to a tile (without a split, DeepSeek-V3 shape, 16 tokens 372.7 / 354.4 us, 60 tokens 767 / 736)
static int pairs_split(int fp4, int stage, int64_t tiles, int K, int split_k)
{
    return fp4 ? 4 : w4a16_split(stage, 16, tiles, K, split_k);
}

// the row blocks to launch: those of the experts that are here
static int64_t launched_blocks(const PairArgs& g, int64_t n_blk)
{
    const int64_t pairs = (int64_t)g.T * g.topk, b = g.held + pairs / g.rows;
    const int64_t most  = pairs < n_blk ? pairs : n_blk;
    return b < most ? b : most;
}

bool pyhip_pairs_served(int64_t tokens, int topk, int experts, int hidden, int inter, int64_t n_blk, int fp4, int split_k)
{
    const int64_t blocks = block_bound(tokens * topk, n_blk, experts);
    const int s1 = pairs_split(fp4, 1, blocks * (inter / 128), hidden, split_k), s2 = pairs_split(fp4, 2, blocks * (hidden / 256), inter, split_k);
    // (offsets into the activations are 32-bit and signed)
    return (s1 == 0 || s1 == 4) && (s2 == 0 || s2 == 4 || (s2 == 32 && tokens == 1 && topk == 2 && inter >= 2048 && inter <= 16384)) &&      // (pyhip_w4a16_token_top2)
           (n_blk * 16 + tokens) * (int64_t)(hidden > inter ? hidden : inter) * 2 < (1ll << 31);
}

static int prepare(const char* name, PairArgs& g, int64_t rows, int64_t blocks, int64_t tiles)
{
    PYHIP_REQUIRE(g.a && g.w && g.w_s && g.out && (g.ids || (g.sorted_ids && g.sorted_e && g.num_valid)), "%s: null pointer", name);
    PYHIP_REQUIRE(g.K > 0 && g.K % 512 == 0 && g.N > 0 && g.N % 256 == 0, "%s: K=%d must be a multiple of 512, N=%d of 256", name, g.K, g.N);
    PYHIP_REQUIRE(g.held > 0 && g.held <= g.experts && (g.rows == 16 || ((g.rows == 32 || g.rows == 64) && g.fp4 && !g.ids && g.a_s)), "%s: bad blocks", name);
    PYHIP_REQUIRE(g.T > 0 && g.topk > 0 && g.experts > 0 && (!g.ids || (int64_t)g.T * g.topk <= PAIRS_UNSORTED_MAX), "%s: bad sizes", name);
    PYHIP_REQUIRE(g.k_real > 0 && g.k_real <= g.K && g.a_pitch >= (g.k_real + 31) / 32 * 32 && g.a_pitch % 8 == 0,
                  "%s: %d of %d columns, rows of %d", name, g.k_real, g.K, g.a_pitch);
    PYHIP_REQUIRE(((uintptr_t)g.a % 16) == 0 && ((uintptr_t)g.w % 16) == 0 && ((uintptr_t)g.w_s % 4) == 0 && ((uintptr_t)g.out % 8) == 0,
                  "%s: unaligned pointer", name);
    PYHIP_REQUIRE(rows * g.a_pitch * 2 < (1ll << 31) && blocks * tiles * 4 < (1ll << 31), "%s: too large", name);
    g.SC      = (g.K / 32 + 7) / 8 * 8;
    // (the last row need not be a whole pitch long)
    g.a_bytes = (u32)(((rows - 1) * g.a_pitch + (g.k_real + 31) / 32 * 32) * 2);
    if(g.a_s)
    {
        PYHIP_REQUIRE(g.fp4 && ((uintptr_t)g.a_s % 4) == 0, "%s: scales", name);
        g.a_bytes  = (u32)(rows * (g.K / 2));
        g.as_bytes = (u32)(rows * ((g.K + 511) / 512 * 16));
    }
    return PYHIP_OK;
}

template <int STAGE>
static void launch_pairs(const PairArgs& g, int split, dim3 grid, hipStream_t stream)
{
    // bf16 rows go through LDS where blocks are half full.  Layer, us, not / staged, by rows per expert: 24 experts, 2048 x 2048 6.7: 38.9 / 41.1, 7.8:
    // 39.9 / 41.3; 60, 2048 x 1408 6.3: 58.3 / 61.3, 6.7 with a Zipf router 49.0 / 47.8; 28, 2048 x 4096 6.4: 74.3 / 77.3, 7.7: 78.1 / 78.6; Mixtral
    // shape 6: 118.6 / 119.5, 7.3: 122.3 / 120.8, 8: 124.5 / 121.7; 32, 2880 x 2880 7.5: 85.7 / 81.7; 16, 4096 x 4096 7.5 with a Zipf router 75.0 / 70.5
    const bool staged = (int64_t)g.T * g.topk >= 7ll * g.experts;
    const dim3 block(W4A16_THREADS);
    if(g.rows == 64)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 4, QUANTISED, 4>), grid, block, 0, stream, g);
    else if(g.rows == 32)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 4, QUANTISED, 2>), grid, block, 0, stream, g);
    else if(g.fp4 && g.a_s)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 4, QUANTISED>), grid, block, 0, stream, g);
    else if(STAGE == 1 && g.fp4)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<1, 4, TO_FP4>), grid, block, 0, stream, g);
    else if(split && staged)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 4, BF16, 1, true>), grid, block, 0, stream, g);
    else if(split)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 4, BF16>), grid, block, 0, stream, g);
    else if(staged)
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 0, BF16, 1, true>), grid, block, 0, stream, g);
    else
        hipLaunchKernelGGL((moe_gemm_pairs_kernel<STAGE, 0, BF16>), grid, block, 0, stream, g);
}

int pyhip_pairs_gate_up(PairArgs g, int64_t rows, int64_t n_blk, int split_k, int activation, float swiglu_limit, hipStream_t stream)
{
    PYHIP_REQUIRE(activation == 0 || (activation == 1 && swiglu_limit > 0.f),
                  "moe_pairs_gate_up: activation=%d (0 SiLU, 1 SwiGLU with a positive limit)", activation);
    const int64_t blocks = block_bound((int64_t)g.T * g.topk, n_blk, g.experts);
    g.n_tiles            = g.N / 256;
    const int split      = pairs_split(g.fp4, 1, blocks * g.n_tiles, g.K, split_k);
    const int rc         = prepare("moe_pairs_gate_up", g, rows, blocks, g.n_tiles);
    if(rc)
        return rc;
    PYHIP_REQUIRE(split == 0 || split == 4, "moe_pairs_gate_up: split_k=%d", split_k);
    PYHIP_REQUIRE(!g.fp4 || (g.out_s && g.N % 1024 == 0), "moe_pairs_gate_up: quantised output");
    g.act    = make_gated_act(activation, swiglu_limit);
    g.swiglu = activation;
    // (tiles whose channels are all padding are not launched)
    const int tile = split ? 32 : 128;
    g.n_tiles      = (g.N / 2 - (g.all_channels ? 0 : g.n_pad) + tile - 1) / tile;
    const dim3 grid((unsigned)(launched_blocks(g, n_blk) * g.n_tiles));
    launch_pairs<1>(g, split, grid, stream);
    PYHIP_CHECK_LAUNCH("moe_gemm_pairs_kernel");
    return PYHIP_OK;
}

int pyhip_pairs_down(PairArgs g, int64_t rows, int64_t n_blk, int split_k, hipStream_t stream)
{
    const int64_t blocks = block_bound((int64_t)g.T * g.topk, n_blk, g.experts);
    g.n_tiles            = g.N / 256;
    const int split      = pairs_split(g.fp4, 2, blocks * g.n_tiles, g.K, split_k);
    const int rc         = prepare("moe_pairs_down", g, rows, blocks, g.n_tiles);
    if(rc)
        return rc;
    PYHIP_REQUIRE(split == 0 || split == 4, "moe_pairs_down: split_k=%d", split_k);
    if(split)
        g.n_tiles *= 4;
    const dim3 grid((unsigned)(launched_blocks(g, n_blk) * g.n_tiles));
    launch_pairs<2>(g, split, grid, stream);
    PYHIP_CHECK_LAUNCH("moe_gemm_pairs_kernel");
    return PYHIP_OK;
}

// Whether a token's slots are few and short enough for a workgroup of the summing GEMM to take them in turns: it streams topk x inter columns.  Layer,
// us, by expert + reduction / summed, 128 experts, one token: top-8, 1024 x 2048 0.99 (16 experts 16.6 / 14.6), 1536 x 1536 16.9 / 16.2, 2048 x 2048 17.0 / 19.7, 1536 x 3072 18.5 / 23.4, 4096 x
// 4096 40.0 / 42.9; top-4, 3072 x 3072 19.4 / 18.4, 3072 x 4096 20.4 / 21.3; two tokens, top-6, 1024 x 3072 19.4 / 21.5.  With 7168 channels over
// the tokens there are workgroups enough: top-8, one token, hidden 7168, inter 2048 35.8 / 34.7, 4096 62.0 / 60.7; two, 4096 x 4096 0.97; top-4, three, 2560 x 4096 0.96.
// (Under an expert mask a token has topk * held / experts slots here: 32 experts, top-8, 4096 x 4096, one of 8 ranks 17.8 / 14.1.)
extern "C" int pyhip_layer_sums(int64_t tokens, int topk, int experts, int held, int hidden, int inter)
{
    return (int64_t)topk * inter * held <= (hidden <= 1024 ? 16384ll : 12288ll) * experts || tokens * hidden >= 7168;
}

int pyhip_pairs_down_sum(PairArgs g, int64_t rows, int64_t n_blk, int split_k, hipStream_t stream)
{
    const int64_t pairs  = (int64_t)g.T * g.topk;
    const int64_t blocks = block_bound(pairs, n_blk, g.experts);
    // by token the weights of an expert are fetched for each of its pairs: only where pairs rarely share one
    if(!g.ids || g.fp4 || g.topk > 8 || !pyhip_layer_sums(g.T, g.topk, g.experts, g.held, g.N, g.K) || (g.T > 1 && 8 * pairs > g.experts) || w4a16_split(2, 16, blocks * (g.N / 256), g.K, split_k) != 4)
        return -1;
    PYHIP_REQUIRE(((uintptr_t)g.out % 16) == 0, "moe_pairs_down_sum: unaligned pointer");
    const int rc = prepare("moe_pairs_down_sum", g, rows, blocks, g.N / 64);
    if(rc)
        return rc;
    // As wide a tile as still gives half of the CUs a workgroup.  Layer, us, NR = 2 / 4, by at4: 256 experts, top-8, 7168 x 2048 224: 62.9 / 58.9, 336: 89.8 /
    // 89.9, 448: 118.1 / 110.4; 3584 x 1024 224: 35.6 / 33.4; top-6, 3584 x 2048 280: 59.5 / 60.3, 4608 x 1024 360: 42.7 / 40.1; 512, top-8, 2560 x 1024 320:
    // 49.8 / 48.5; 256, top-8, 6144 x 1536 288: 65.3 / 65.8
    const int64_t at4 = (int64_t)g.T * (g.N / 64);
    const int nr      = at4 >= 140 ? 4 : at4 >= 80 ? 2 : 1;
    g.n_tiles         = g.N / (16 * nr);
    const dim3 grid((unsigned)(g.T * g.n_tiles)), block((g.topk > 1 ? 2 : 1) * 4 * WAVE);
    if(nr == 4)
        hipLaunchKernelGGL((moe_pairs_down_sum_kernel<4>), grid, block, 0, stream, g);
    else if(nr == 2)
        hipLaunchKernelGGL((moe_pairs_down_sum_kernel<2>), grid, block, 0, stream, g);
    else
        hipLaunchKernelGGL((moe_pairs_down_sum_kernel<1>), grid, block, 0, stream, g);
    PYHIP_CHECK_LAUNCH("moe_pairs_down_sum_kernel");
    return PYHIP_OK;
}
