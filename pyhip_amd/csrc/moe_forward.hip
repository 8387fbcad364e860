// The whole layer behind one call: sort (+ input quantisation) -> gate_up GEMM -> down GEMM -> top-k reduce, with
// every intermediate buffer carved out of a workspace the caller provides.  It is what pyhip_amd/fused_moe.py does
// step by step (the reference's operator, src/contrib/fused_moe.py:128-576, allocates its intermediates with torch
// and launches its kernels one by one from Python); the choice of kernel family and row block stays with the caller.
#include "common.h"
#include "moe_gemm_pairs.h"
#include "quant_device.h"
#include <math.h>

extern "C" {
int64_t pyhip_moe_sorting_max_blocks(int64_t tokens, int topk, int experts, int block_size);
int64_t pyhip_moe_sorting_workspace_bytes(int64_t tokens, int topk, int experts);
int64_t pyhip_moe_schedule_words(int experts);
int64_t pyhip_moe_act_scale_stride(int K);
int pyhip_moe_sorting(const int32_t*, const float*, int, int, int, int, const int32_t*, const int32_t*, uint32_t*, float*,
                      uint32_t*, uint32_t*, uint32_t*, void*, int64_t, void*, int64_t, hipStream_t);
int pyhip_moe_gemm1_mxfp4(const uint8_t*, const uint8_t*, const uint8_t*, const uint8_t*, const void*, const uint32_t*,
                          const uint32_t*, const uint32_t*, const uint32_t*, void*, uint8_t*, uint8_t*, int, int, int, int,
                          int, int, int, int, int64_t, int, float, hipStream_t);
int pyhip_moe_gemm2_mxfp4(const uint8_t*, const uint8_t*, const uint8_t*, const uint8_t*, const void*, const uint32_t*,
                          const float*, const uint32_t*, const uint32_t*, const uint32_t*, void*, int, int, int, int, int,
                          int, int, int, int64_t, hipStream_t);
int pyhip_moe_gemm1_w4a16(const void*, const uint8_t*, const uint8_t*, const void*, const uint32_t*, const uint32_t*,
                          const uint32_t*, void*, int, int, int, int, int, int, int64_t, int, int, float, hipStream_t);
int pyhip_moe_gemm2_w4a16(const void*, const uint8_t*, const uint8_t*, const void*, const uint32_t*, const float*,
                          const uint32_t*, const uint32_t*, void*, int, int, int, int, int, int, int64_t, int, hipStream_t);
int pyhip_moe_gemm1_w4a16_token(const void*, const uint8_t*, const uint8_t*, const void*, const int32_t*, const int32_t*,
                                const int32_t*, void*, int, int, int, int, int, int, float, hipStream_t);
int pyhip_moe_gemm2_w4a16_token(const void*, const uint8_t*, const uint8_t*, const void*, const int32_t*, const float*,
                                const int32_t*, const int32_t*, void*, int, int, int, int, int, hipStream_t);
int pyhip_moe_route_sorting(const float*, int, int, int, int, int, int, int, const int32_t*, const int32_t*, float*, int32_t*,
                            uint32_t*, float*, uint32_t*, uint32_t*, uint32_t*, void*, int64_t, const void*, int64_t, int64_t,
                            int, uint8_t*, uint8_t*, hipStream_t);
int pyhip_moe_topk_reduce_routed(const void*, void*, int64_t, int, int, int, const int32_t*, int, const int32_t*,
                                 const int32_t*, hipStream_t);
int pyhip_moe_topk_softmax(const float*, int, int, int, int, float*, int32_t*, hipStream_t);
int pyhip_moe_topk_grouped_sigmoid(const float*, int, int, int, int, int, int, float*, int32_t*, hipStream_t);
}

int pyhip_sorting_quant_cols(const int32_t*, const float*, int, int, int, int, const int32_t*, const int32_t*, uint32_t*,
                             float*, uint32_t*, uint32_t*, uint32_t*, void*, int64_t, const void*, int64_t, int64_t, int,
                             uint8_t*, uint8_t*, int, hipStream_t);

int pyhip_w4a16_token_top2(const void*, const uint8_t*, const uint8_t*, const void*, const int32_t*, const float*, const int32_t*,
                           const int32_t*, void*, int, int, int, int, int, int, hipStream_t);

namespace {
struct Carve
{
    int64_t off = 0;
    int64_t take(int64_t bytes)
    {
        int64_t o = off;
        off += (bytes + 255) / 256 * 256;
        return o;
    }
};
struct Layout
{
    int64_t n_blk, rows2;
    int64_t sorted_ids, sorted_w, sorted_e, num_valid, sched, sort_ws, sort_ws_bytes, a1_q, a1_s, a2, a2_q, a2_s, out3;
    int64_t total;
};
Layout make_layout(int64_t T, int k, int E, int H, int I, int bm, int w4a16)
{
    Layout l;
    Carve c;
    l.n_blk         = pyhip_moe_sorting_max_blocks(T, k, E, bm);
    l.rows2         = l.n_blk * bm;
    l.sorted_ids    = c.take(l.rows2 * 4);
    l.sorted_w      = c.take(l.rows2 * 4);
    l.sorted_e      = c.take(l.n_blk * 4);
    l.num_valid     = c.take(8);
    l.sched         = c.take(pyhip_moe_schedule_words(E) * 4);
    l.sort_ws_bytes = pyhip_moe_sorting_workspace_bytes(T, k, E);
    l.sort_ws       = c.take(l.sort_ws_bytes);
    l.a1_q = l.a1_s = l.a2 = l.a2_q = l.a2_s = 0;
    if(w4a16)
        l.a2 = c.take(l.rows2 * (int64_t)I * 2);
    else
    {
        l.a1_q = c.take(T * (int64_t)(H / 2));
        l.a1_s = c.take(T * pyhip_moe_act_scale_stride(H));
        l.a2_q = c.take(l.rows2 * (int64_t)(I / 2));
        l.a2_s = c.take(l.rows2 * pyhip_moe_act_scale_stride(I));
    }
    l.out3  = c.take(T * (int64_t)k * H * 2);
    l.total = c.off;
    return l;
}
}   // namespace

// The choices pyhip_amd/fused_moe.py makes for method="auto" and block_size_M=None (pick_block_m, pick_w4a16; the
// measurements behind them are quoted there), for callers that bind the library without the Python layer.
extern "C" int pyhip_moe_pick_block_m(int64_t tokens, int topk, int experts, int hidden, int w4a16)
{
    const double est = (double)tokens * topk / (experts > 0 ? experts : 1);      // routed rows per expert, on average
    // The tile is chosen from the AVERAGE load, which is all that is known before the sort has run, with room for routers
    // that load their experts unevenly: every extra row block of a busy expert streams that expert's weights again, while
    // a tile that is larger than a quiet expert needs only costs the occupancy of its kernel.  One step up the ladder
    // from "twice the mean" costs 1-2 % under an even router and saves 11-17 % under a Zipf(1.1) one (whole layer, ms,
    // tiles of 16 / 32 / 64 rows; DeepSeek-V3 shape, 128 tokens = 4 rows per expert: 0.904 / 0.917 / 0.942, gpt-oss shape, 256
    // tokens = 8: 0.301 / 0.305 / 0.320; Qwen3 shape with the Zipf router, 64 tokens = 4: 0.123 / 0.103 / 0.108, 128 = 8:
    // 0.169 / 0.140 / 0.137, 256 = 16: 0.218 / 0.191 / 0.169).
    // With a handful of experts (Mixtral: 8) every expert gets many rows, the loads are even in relative terms, and the
    // number of tiles is what such layers are short of: "twice the mean" stays (Mixtral shape, 32 tokens: 0.134 ms with
    // 16-row blocks, 0.158 with 32).
    // The same holds for the bf16-activation kernels, whose 32-row tile already halves the waves per SIMD (DeepSeek-V3
    // shape, 128 tokens, forced: gate_up 623 us with 16-row blocks, 761 with 32); their row block is at most 64.
    if(experts < 32 || w4a16)
    {
        for(int bm = 16; bm <= 64; bm *= 2)
            if(2 * est <= bm)
                return bm;
        // One block of 64 rows holds an expert as long as few experts have more than that, which the mean tells with up to 16
        // experts and up to 44 rows.  Layer, us, 64 / 128 rows, by rows per expert (even router; Zipf router, two seeds):
        //    8 experts, 4096 x 14336:  34: 145 / 153; 171 / 167, 170 / 168      40: 154 / 162; 171 / 169, 170 / 170
        //                              48: 156 / 163; 176 / 176, 175 / 175      50: 169 / 164; 180 / 176, 178 / 174
        //   12 experts, 5120 x 2048:   34: 48.5 / 51.5; 56.0 / 64.2, 56.0 / 63.6   42: 50.2 / 53.0; 57.4 / 65.0, 57.3 / 64.5
        //                              48: 51.0 / 54.3; 74.1 / 66.2, 75.8 / 65.8
        //   16 experts, 4096 x 3584:   34: 77.0 / 82.1; 98.9 / 99.6, 99.9 / 98.6   40: 79.0 / 84.5; 101 / 98.5, 102 / 101
        //                              44: 78.7 / 83.6; 102 / 110, 101 / 98.5      50: 87.1 / 84.5; 105 / 111, 106 / 110
        //   28 experts, 2048 x 4096:   34: 81.4 / 86.1; 101 / 91.3, 102 / 91.5     46: 82.6 / 87.4; 103 / 92.0, 105 / 89.2
        // (5-7 % under even routers against 3 % at most under Zipf ones; with more experts, or nearer to 64 rows, the busy ones
        // need a second block and cost up to 17 %)
        if(!w4a16 && experts <= 16 && est <= 44)
            return 64;
    }
    else
    {
        if(est < 4)
            return 16;
        if(est < 12)
            return 32;
        if(est <= 32)
            return 64;
    }
    if(w4a16)
        return 64;
    // Prefill sizes: 128 rows, except where a taller tile lets nearly every expert fit ONE row block, so that each weight
    // tile is read once instead of two or three times.  The tiles above 128 rows run one wave per SIMD and have a long
    // epilogue, which pays most with a long K loop (hidden >= 6144).  DeepSeek-V3 shape, whole layer, ms, tiles of 128 / 160 /
    // 192 / 256 / 288 rows by expected rows per expert (between machines the order of close neighbours can flip):
    //    96: 1.28 / 1.33 / 1.36 / 1.50 /  -       160: 2.26 / 1.93 / 1.49 / 1.60 / 1.73      232: 1.97 /  -   /  -   / 1.86 / 1.92
    //   104: 1.36 / 1.35 / 1.38 / 1.52 / 1.66     168: 2.08 / 2.22 / 1.55 / 1.62 / 1.75      240: 2.09 /  -   /  -   / 1.96 / 1.94
    //   120: 1.50 / 1.37 / 1.40 / 1.51 / 1.63     176: 2.04 / 2.63 / 1.65 / 1.64 / 1.77      256: 2.26 /  -   /  -   / 2.64 / 2.02
    //   128: 1.72 / 1.39 / 1.42 / 1.53 / 1.65     192: 1.92 / 2.67 / 2.20 / 1.68 / 1.81      272: 2.46 /  -   /  -   / 3.29 / 2.36
    //   136: 1.92 / 1.43 / 1.43 / 1.54 / 1.67     208: 1.91 /  -   /  -   / 1.72 / 1.85      288: 2.57 /  -   /  -   / 3.53 / 2.97
    // With the shorter K loop of hidden 3072 / 4096 only the first step pays, and only under an even router: 100-132
    // expected rows per expert, where the 128-row tile needs a second, nearly empty block for half of the experts (whole
    // layer, ms, 128 / 160 / 192 / 256 rows: Mixtral shape, 512 tokens: 0.210 / 0.191 / 0.198 / 0.216; gpt-oss shape, 4096
    // tokens: 0.564 / 0.499 / 0.513 / 0.556; the Qwen3 shape's Zipf router at 2048 tokens, the same mean: 0.399 / 0.420 /
    // 0.425 / 0.452: most of its experts are far below the mean and pay for the taller tile's empty row groups).  Further
    // up, the taller tiles win by 3-11 % under the even routers at exactly the sizes where an expert fills one block
    // (192 rows at 160 per expert, 288 at 256) and lose up to 20 % under the uneven one and between those sizes: left at
    // 128 rows.
    if(hidden < 6144 && est >= 100 && est <= 132)
        return 160;
    if(hidden >= 6144)
    {
        if(est >= 100 && est <= 132)
            return 160;
        if(est > 132 && est <= 172)
            return 192;
        if(est > 172 && est <= 236)
            return 256;
        if(est > 236 && est <= 276)
            return 288;
    }
    return 128;
}

// Row blocks that hold an expert's rows, on average, when it gets a Poisson number of them with mean m
static double expected_blocks(double m, int rows)
{
    if(m > 12.0 * rows)
        return m / rows + 0.5;
    double n = 1.0 - exp(-m);
    for(int j = 1; j * rows < m + 5.0 * sqrt(m) + 1.0; j++)
        n += 0.5 * erfc((j * rows + 0.5 - m) / sqrt(2.0 * m));
    return n;
}

// What a launch of a tile height costs, us: a tile takes `start + step * K-groups`, `at_once` tiles run side by side (a launch of
// fewer takes as long as one tile), and each further block of an expert costs `again` of the expert's weights in memory traffic (the rest it
// finds in the L2).  Fitted to 490 random layers (8-256 experts, hidden 1024-7200, intermediate 512-14336, 16-8192 tokens, even and
// Zipf routers, every height timed on each): the estimate of a call is within 8 % of its time (root mean square).
struct TileCost
{
    int rows;
    double start, step, at_once, again;
};
static const TileCost tile_costs[] = {{16, 1.2, 1.37, 1e9, 0.35}, {32, 1.5, 1.39, 1e9, 0.4},  {64, 3.3, 1.29, 334, 0.45},
                                      {128, 4.5, 2.10, 307, 0.33}, {160, 5.8, 2.27, 284, 0.75}, {192, 6.8, 2.38, 271, 1.05},
                                      {256, 8.6, 2.84, 276, 1.6},  {288, 9.8, 3.15, 273, 2.0}};

static bool takes_pairs(int64_t tokens, int topk, int experts, int local_experts, int hidden, int inter, int block_m, int w4a16, int split_k);

// The tile height of an MXFP4-activation layer call whose sizes are known: the one of pyhip_moe_pick_block_m, which looks at the rows
// per expert alone, unless that has fewer tiles in the gate_up GEMM than the chip has CUs and 64, 32 or 16 rows are estimated to
// take 5 % less: lower tiles are more of them, and each is done sooner.  Layer, us: 8 experts, 1024 x 512, top-2, 493 tokens, 160 / 16 rows:
// 30.2 / 23.7; 1024 tokens, 128 / 32: 30.2 / 27.1; 2208 x 1792, top-1, 446 tokens, 128 / 32: 36.5 / 27.2; 6176 x 512, Zipf, 371 tokens, 128 / 32:
// 52.3 / 37.1.  The estimate is trusted where lower tiles cannot lose much, else the ladder stays: where the
// ladder, at 128 rows and more, leaves nearly half of the CUs without a tile (388 calls of random layers take 21 % less, the slowest 8 % more; beyond, up to 44 %
// more: 8 experts, 6656 x 3584, 60 rows per expert, 224 tiles of 128 rows), with few enough of them that all run at
// once also under a router that makes more (64 rows: 96 in the gate_up GEMM, 160 up to hidden 2048; 16 and 32: 128), or with a short K loop (16 and 32
// rows: hidden up to 2048, or 2560 where an expert has two blocks and few are here; 64: 1024).  Beyond that it was wrong by up to 40 % (8 experts, 128 / 64
// rows: 6720 x 2944, Zipf, 216 tokens 68.2 / 95.4; 4576 x 2304, 348 tokens 52.6 / 64.7; 5888 x 2528, 466 tokens, 160 / 64: 66.6 / 80.0; 24 experts, 128 / 32: 4960 x
// 512, 1153 tokens 57.8 / 67.0; 64 / 32: 1856 x 1024, Zipf, 162 tokens 30.2 / 37.1).  Of 1400 other
// layers that the rule moves, each under an even and a Zipf router, the calls take 16 % less (geometric mean), and one of 2800 takes more than 3 % more (11:
// 28 experts, 1920 x 512, top-1, Zipf, 4114 tokens).
// (With as many tiles as CUs and more the estimate would find other heights too, and is not good enough for it, nor does it know the
// router: 64 rows instead of 128 cost up to 20 % between 33 and 60 rows per expert, 192 to 288 rows at hidden below 6144 save 14-23 % under
// even routers and cost 6-18 % under Zipf ones.)
extern "C" int pyhip_layer_block_m(int64_t tokens, int topk, int experts, int local_experts, int hidden, int inter)
{
    int ladder = pyhip_moe_pick_block_m(tokens, topk, experts, hidden, 0);
    if(tokens <= 0 || topk <= 0 || experts <= 0 || local_experts <= 0)
        return ladder;
    const double est = (double)tokens * topk / experts;
    // The ladder's lower lines are those of the persistent kernels.  In those of moe_gemm_pairs.hip, which compute the row tiles that have
    // rows, a higher block costs next to nothing and holds the busy experts of an uneven router.  Layer, us, 16 / 32 rows: DeepSeek-V3 shape, 80
    // tokens (2.5 rows per expert) 771 / 775; 64 experts, top-6, 2048 x 1408, 40 tokens (3.8) 54.7 / 55.4; Qwen3 shape, 45 tokens (2.8) 88.5 / 86.4;
    // under Zipf routers 256 experts, top-8, 2048 x 512, 100 tokens (3.1) 41.0 / 37.7; 96, top-4, 6272 x 1920, 90 tokens (3.8) 123 / 108.
    // 32 / 64 rows (three waves per SIMD instead of four, which a short K loop feels): DeepSeek-V3 shape 6.3: 881 / 887, 9.4: 913 / 917; gpt-oss shape
    // 6.3: 257 / 257, 11.6: 272 / 277; Qwen3 shape 6.3: 120 / 118, 11: 155 / 147; 96 experts, Zipf, 5: 121 / 114, 7.5: 152 / 143, 11.7: 211 / 189; hidden
    // 2048: 256 experts, top-1 9.8: 338 / 355; 128, top-8, 11: 70.7 / 74.2; 60, top-4, 10: 56.4 / 58.7
    // 64 rows with a K loop of 1024 columns in the down GEMM cost 2-4 % (3072 x 1024, 512 experts, 8 rows per expert, 32 / 64 rows 417.9 / 423.0, the persistent
    // kernels 412.5).  And only where those kernels serve the higher block
    auto served = [&](int rows) { return takes_pairs(tokens, topk, experts, local_experts, hidden, inter, rows, 0, 0); };
    if(ladder == 16 && experts >= 32 && est >= 2.0 && tokens * topk > WAVE && served(32))
        ladder = 32;
    else if(ladder == 32 && experts >= 32 && est >= 5.0 && hidden >= 3072 && inter > 1024 && served(64))
        ladder = 64;
    // (the estimate is of the persistent kernels; 16 rows instead of 32 were not measured)
    if(local_experts * expected_blocks(est, ladder) * (inter / 128) >= 256.0 || ladder <= 32 || served(ladder))
        return ladder;
    auto estimate = [&](const TileCost& c) {
        const double hit = local_experts * (1.0 - exp(-est)), nb = local_experts * expected_blocks(est, c.rows);
        // sort, reduction and the passes over the activations
        double us = 12.0 + (double)tokens * (topk + 2) * hidden / 2.5e6;
        for(int stage = 0; stage < 2; stage++)
        {
            const int n = stage ? hidden / 256 : inter / 128, groups = stage ? inter / 512 : hidden / 512;
            const double run = (c.start + c.step * groups) * (nb * n > c.at_once ? nb * n / c.at_once : 1.0);
            const double mem = (hit + c.again * (nb - hit)) * n * groups * (512.0 * 256.0 * 17.0 / 32.0) / 6.6e6;
            us += sqrt(sqrt(run * run * run * run + mem * mem * mem * mem));
        }
        return us > 20.0 ? us : 20.0;       // (a call takes the host that long)
    };
    double best = 0.0;
    for(const TileCost& c : tile_costs)
        if(c.rows == ladder)
            best = 0.95 * estimate(c);
    int rows = ladder;
    for(const TileCost& c : tile_costs)
        if(c.rows < ladder && c.rows <= 64 && est <= 10.0 * c.rows && estimate(c) < best)      // (beyond ten blocks an expert: not measured)
        {
            best = estimate(c);
            rows = c.rows;
        }
    const double at_ladder = local_experts * expected_blocks(est, ladder) * (inter / 128);
    if(ladder >= 128 && at_ladder <= 145.0 && (rows == 64 || local_experts * expected_blocks(est, rows) * (inter / 128) <= 280.0))
        return rows;
    const double tiles = local_experts * expected_blocks(est, rows) * (inter / 128);
    const bool short_k = hidden <= 2048 || (hidden <= 2560 && est <= 2.0 * rows && local_experts <= 12);
    const bool trusted = rows == 64 ? hidden <= 1024 || tiles <= (hidden <= 2048 ? 160.0 : 96.0)
                                    : tiles <= 128.0 || (short_k && (ladder > 64 || tiles <= 192.0));
    return trusted ? rows : ladder;
}

extern "C" int pyhip_moe_pick_w4a16(int64_t tokens, int topk, int experts, int hidden)
{
    // bf16 activations win (a) when at most one expert in eight gets a row at all (DeepSeek-V3 shape: 1 token 0.046
    // against 0.051 ms, 4 tokens 0.128 against 0.127 ms, 16 tokens 0.393 against 0.377 ms; gpt-oss shape: 4 tokens 0.053
    // against 0.055 ms, 16 tokens 0.141 against 0.134 ms), and (b) in layers with so few experts that the down GEMM of
    // the MXFP4-activation path has fewer than 512 tiles, which the bf16 kernel splits K-wise over four times as many
    // workgroups (Mixtral shape: 1 token 0.054 against 0.071 ms, 16 tokens 0.132 against 0.137 ms, 64 tokens 0.181
    // against 0.140 ms)
    const int64_t pairs  = tokens * topk;
    const bool sparse    = 8 * pairs <= (int64_t)experts;
    const bool few_tiles = (pairs < experts ? pairs : experts) * (hidden / 256) < 512 && pairs <= 8 * (int64_t)experts;
    return sparse || few_tiles;
}

extern "C" int64_t pyhip_moe_forward_workspace_bytes(int64_t tokens, int topk, int experts, int hidden, int inter,
                                                     int block_m, int w4a16)
{
    if(tokens <= 0 || topk <= 0 || experts <= 0 || hidden <= 0 || inter <= 0 || block_m <= 0)
        return 0;
    return make_layout(tokens, topk, experts, hidden, inter, block_m, w4a16).total;
}

namespace {
struct Router
{
    const float* gating = nullptr;      // [tokens, experts] or null: topk_ids / topk_weights are inputs
    int n_group = 0, topk_group = 0, renormalize = 1;
};
}   // namespace

// Whether forward_pairs below serves the call.  MXFP4 activations: without a sort, or while experts have few rows on average, so that
// a busy one has few blocks, and few blocks are full.  With more, blocks that fetch the weights of their expert again, and activations that
// every 64 weight rows fetch again, cost more than the persistent kernels, whose workgroups have 256.  With a handful of experts loads are
// even in relative terms and the lines lie higher.  Layer, us, persistent kernel / this, by rows per expert:
//   16 rows: DeepSeek-V3 shape 0.5: 374.8 / 355.6, 3.1: 868 / 821; Qwen3 shape 1.9: 88.7 / 77.1, 4: 121 / 107; gpt-oss shape 2: 220 / 214; 96
//     experts, top-4, Zipf router, 6272 x 1920 1.7: 95.9 / 91.4, 3.8: 133 / 123, 6.3: 166 / 166, 10: 231 / 243
//   32 rows: DeepSeek-V3 shape 4: 906 / 852, 6.3: 928 / 881, 11.6: 949 / 935, 16: 964 / 984; Qwen3 shape 4: 103.7 / 99.8, 11: 158 / 155; gpt-oss shape
//     6.3: 273 / 257, 11.6: 280 / 272, 16: 284 / 288; 64 experts, top-6, 2048 x 1408 9.4: 62.2 / 58.4; 96 experts 7.5: 150 / 152, 11.7: 212 / 211;
//     8 experts, 4096 x 14336, 10: 136 / 121, 16, Zipf: 154 / 146, 25: 152 / 147, 40: 166 / 218; 28 experts, top-6, 2048 x 4096, 15: 78.5 / 71.7
//   64 rows (against the persistent kernel of the better height): Qwen3 shape 6.3: 128 / 118, 11: 158 / 147; gpt-oss shape 9.4: 277 / 268, 11.6: 280 /
//     277, 31: 323 / 357; DeepSeek-V3 shape 11.6: 949 / 939, 16: 964 / 981; 96 experts 5: 128 / 114, 11.7: 212 / 189; 8 experts 17.5: 140 / 123, 25: 142 /
//     129, 40: 147 / 149; 16, top-2, 4096 x 4096 25: 84.3 / 83.0, 31: 85.0 / 88.4; 12, 5120 x 2048 22: 46.8 / 47.4, 28: 47.6 / 51.2
// With a handful of experts and hidden 2560 and more the line lies lower where the persistent kernels' tiles of the gate_up GEMM (`tiles`) make most of one
// round of the chip.  (From 232 to 256 an uneven router takes them into a second round, which costs them up to 25 %.)  Layer, us, persistent kernels / this, or the
// ratio, by rows per expert:
//   192 tiles, 24 experts, top-4, 7168 x 1024 under a Zipf router 10: 58.6 / 63.5, 23: 64.2 / 72.0, under an even one 10: 0.98
//   224, 28 experts, top-2, 7168 x 1024 23: 71.9 / 79.4; 4096 x 1024 13: 43.6 / 45.3, 23: 47.4 / 51.3
//   240, 20 experts, 3072 x 1536 13: 0.95, under a Zipf router 0.77; 64, 8 experts, 5120 x 1024 10: 0.69; 320, 20 experts, 4096 x 2048 19: 67.3 / 59.2
static bool few_enough_rows(int64_t pairs, int experts, int local_experts, int hidden, int inter, int block_m)
{
    if(experts >= 32 || block_m == 16)
        return pairs <= (int64_t)experts * (experts < 32 ? 8 : block_m == 16 ? 4 : 12);
    const double tiles = local_experts * expected_blocks((double)pairs / experts, block_m) * (inter / 128);
    const bool full = tiles > 136.0 && tiles <= 232.0 && hidden >= 2560;
    const int most = block_m == 32 ? 16 : 24, most_full = hidden < 5120 ? 21 : tiles <= 216.0 ? 14 : 17;
    return pairs <= (int64_t)experts * (full && most_full < most ? most_full : most);
}
// Whether they find their rows themselves, in blocks of 16: up to a pair to a lane; with two, which costs every workgroup of the gate_up
// GEMM more, if all of its workgroups run at once (and the list of blocks fits where a sort into 32 rows would put its own).
// Layer, us, sorted / this: 8 experts, 1024 x 512, top-2, 40 tokens 21.3 / 17.9, 64 tokens 21.2 / 17.7; 12, 1024 x 1024, top-1, 100 tokens 22.9 /
// 19.0.  With more workgroups it goes either way: DeepSeek-V3 shape, 16 tokens 356.0 / 347.5; 96 experts, top-4, 6272 x 1920, 30 tokens 204.6 / 198.2;
// 60, 2048 x 1408, 32 tokens 49.2 / 47.0; gpt-oss shape, 32 tokens 167.9 / 170.6; Qwen3 shape, 16 tokens 65.9 / 68.3; Mixtral shape, 50 tokens, bf16
// activations 121.4 / 131.4: left to the sort.  Nor, with more than 8 rows per expert, in large layers, which fetch the weights of their
// second blocks again.  Layer, us, persistent kernels / this, 8 experts, top-2, 64 tokens: 2560 x 1536 27.8 / 23.9, 3584 x 1024 28.1 / 23.6, 3072 x 1536 28.8 / 27.4, 5120 x
// 1536 36.2 / 39.7, 7168 x 1536 43.8 / 52.0; 40 tokens, 7168 x 1024 0.69.
static bool leaves_sort_out(int64_t tokens, int topk, int experts, int hidden, int inter, int block_m, int w4a16)
{
    const int64_t pairs = tokens * topk, blocks = pairs < experts + pairs / 16 ? pairs : experts + pairs / 16;
    if(block_m > 32 || (w4a16 && block_m > 16) || pairs > PAIRS_UNSORTED_MAX)
        return false;
    return (block_m == 16 && pairs <= WAVE) || (blocks * (inter / 32) <= 768 && blocks <= 64 &&
                                                pairs <= 16ll * experts && (w4a16 || pairs <= 8ll * experts || pairs * hidden * inter <= (80ll << 20) * experts));
}
// A workgroup's start and end against its K loop, of which 512 columns are a single K-step to each of its four waves.  With MXFP4 activations
// such layers are served only while few workgroups follow one another on a CU, or in 16-row blocks with hidden between 1024 and 2048 or few pairs.  Layer, us,
// persistent kernels / this, by the workgroups of both GEMMs: 512 x 512, 16-row blocks, 160 experts, top-6 1300: 22.3 / 19.3, 2280: 22.3 / 24.6, 3420: 27.1 / 29.1; 384
// experts, top-8 8200: 42.8 / 50.9; 512 x 1536 19100: 93.5 / 108.9; 1024 x 512, 128 experts, top-8 2040: 22.8 / 21.9, 3180: 29.7 / 30.5, 32-row blocks 4070: 33.5 /
// 34.8; 3072 x 512, 64 experts, top-6 3260: 35.3 / 36.5, 128, 0.7 rows per expert: 49.4 / 42.8; 4096 x 512, 512 experts, top-8 31800: 236.0 / 250.8; between, 16-row blocks: 1536 x 512, 160
// experts 5700: 47.2 / 45.1; 2048 x 512, 256 experts, top-8 6110: 59.8 / 54.3, 11700: 86.0 / 85.2, 64-row blocks 90.3 / 93.0.  With 1024 columns it is
// no matter any more (512 experts, 3072 x 1024 38900: 381.8 / 375.2; 384, 1024 x 1024 10900: 80.6 / 75.5) but for 64-row blocks with hidden 1024 (160
// experts, 1024 x 1024, 7700: 1.10).  bf16 activations, whose K-steps
// take longer: only where full blocks pass through LDS first (512 x 1024, 160 experts, 9.5 rows per expert 55.4 / 59.1, 6 rows 0.95).
static bool too_short_for_pairs(int64_t pairs, int experts, int local_experts, int hidden, int inter, int block_m, int w4a16)
{
    if(w4a16)
        return hidden < 1024 && experts >= 32 && pairs >= 7ll * experts;
    const double est = (double)pairs / experts, workgroups = local_experts * expected_blocks(est, block_m) * (inter / 32 + hidden / 64);
    if(hidden < 1024)
        return workgroups > 2048.0;
    if(inter < 1024)
        return workgroups > 3000.0 && !(block_m == 16 && ((hidden > 1024 && hidden <= 2048) || (est <= 1.6 && workgroups <= 8192.0)));
    return block_m == 64 && hidden == 1024 && workgroups > 4096.0;
}
static bool takes_pairs(int64_t tokens, int topk, int experts, int local_experts, int hidden, int inter, int block_m, int w4a16, int split_k)
{
    const int64_t pairs = tokens * topk;
    if(block_m != 16 && ((block_m != 32 && block_m != 64) || w4a16))
        return false;
    const int here = local_experts > 0 && local_experts < experts ? local_experts : experts;
    if(topk <= 0)
        return false;
    if(w4a16 ? too_short_for_pairs(pairs, experts, here, hidden, inter, block_m, w4a16)
             : !leaves_sort_out(tokens, topk, experts, hidden, inter, block_m, w4a16) &&
                   (!few_enough_rows(pairs, experts, here, hidden, inter, block_m) || too_short_for_pairs(pairs, experts, here, hidden, inter, block_m, w4a16)))
        return false;
    return hidden % 512 == 0 && inter % 512 == 0 && experts <= 2048 &&
           pyhip_pairs_served(tokens, topk, experts, hidden, inter, pyhip_moe_sorting_max_blocks(tokens, topk, experts, block_m) * (block_m / 16),
                              !w4a16, split_k);
}

// the rows of hidden states that they take: offsets into them are 32-bit and signed, in bytes
static bool takes_rows(int64_t tokens, int64_t row_stride) { return row_stride < (1 << 30) && tokens * row_stride < (1 << 30); }
// ... and with bf16 activations at the true width of a padded layer
static bool takes_bf16_cols(int64_t tokens, int64_t row_stride, int cols)
{
    return takes_rows(tokens, row_stride) && row_stride >= cols && row_stride % 8 == 0 && row_stride < (1 << 24);
}

// The layer by the kernels of moe_gemm_pairs.hip.  Up to 128 pairs the kernels find their rows themselves
// and the sort is left out; where pairs rarely share an expert the down GEMM sums the slots and the reduction is left out too: two
// launches (with the router three) instead of four.  What that saves is the launch on the host (3.3 us each) and the latency chain of the stage
// on the device (sort 4.5-5.5, reduction 3-5 us).
static int forward_pairs(const void* hidden_bf16, int64_t row_stride, int hidden_cols, const uint8_t* w1, const uint8_t* w1_scale,
                         const uint8_t* w2, const uint8_t* w2_scale, const void* bias1_bf16, const void* bias2_bf16,
                         const Router& router, int32_t* topk_ids, float* topk_weights, const int32_t* expert_mask,
                         const int32_t* num_local_tokens, void* out, int out_is_f32, int tokens, int topk, int experts,
                         int hidden, int inter, int hidden_pad, int inter_pad, int block_m, int w4a16, int split_k, int activation,
                         float swiglu_limit, int held, const Layout& l, uint8_t* ws, hipStream_t stream)
{
    uint8_t* a2         = ws + (w4a16 ? l.a2 : l.a2_q);      // a row for every pair
    const bool unsorted = leaves_sort_out(tokens, topk, experts, hidden, inter, block_m, w4a16);
    uint32_t* s_ids     = (uint32_t*)(ws + l.sorted_ids);
    float* s_w          = (float*)(ws + l.sorted_w);
    uint32_t *s_e = (uint32_t*)(ws + l.sorted_e), *n_valid = (uint32_t*)(ws + l.num_valid), *sched = (uint32_t*)(ws + l.sched);
    int rc = PYHIP_OK;
    if(!w4a16 && unsorted)
    {
        // (what the launch that quantises them asks of the hidden states)
        QuantArgs q;
        rc = pyhip_make_quant_args("moe_forward", hidden_bf16, row_stride, tokens, hidden, ws + l.a1_q, ws + l.a1_s, nullptr, &q, hidden_cols);
        if(rc)
            return rc;
    }
    // (the launch that routes and sorts refuses it as well)
    PYHIP_REQUIRE(!router.gating || router.n_group >= 0, "moe_forward: n_group=%d (0 groups = softmax router)", router.n_group);
    if(router.gating && unsorted)
        rc = router.n_group > 0 ? pyhip_moe_topk_grouped_sigmoid(router.gating, tokens, experts, topk, router.n_group, router.topk_group,
                                                                 router.renormalize, topk_weights, topk_ids, stream)
                                : pyhip_moe_topk_softmax(router.gating, tokens, experts, topk, router.renormalize, topk_weights, topk_ids, stream);
    else if(router.gating)
        rc = pyhip_moe_route_sorting(router.gating, tokens, topk, experts, router.n_group, router.topk_group, router.renormalize, block_m,
                                     expert_mask, num_local_tokens, topk_weights, topk_ids, s_ids, s_w, s_e, n_valid, sched,
                                     ws + l.sort_ws, l.sort_ws_bytes, w4a16 ? nullptr : hidden_bf16, row_stride, tokens, hidden,
                                     w4a16 ? nullptr : ws + l.a1_q, w4a16 ? nullptr : ws + l.a1_s, stream);
    else if(!unsorted && !w4a16)
        rc = pyhip_sorting_quant_cols(topk_ids, topk_weights, tokens, topk, experts, block_m, expert_mask, num_local_tokens, s_ids, s_w, s_e,
                                      n_valid, sched, ws + l.sort_ws, l.sort_ws_bytes, hidden_bf16, row_stride, tokens, hidden,
                                      ws + l.a1_q, ws + l.a1_s, hidden_cols, stream);
    else if(!unsorted)
        rc = pyhip_moe_sorting(topk_ids, topk_weights, tokens, topk, experts, block_m, expert_mask, num_local_tokens, s_ids, s_w, s_e,
                               n_valid, sched, nullptr, 0, ws + l.sort_ws, l.sort_ws_bytes, stream);
    if(rc)
        return rc;
    PairArgs g;
    if(unsorted)
    {
        g.ids = topk_ids; g.weights = topk_weights; g.mask = expert_mask; g.local_tok = num_local_tokens;
    }
    else
    {
        g.sorted_ids = s_ids; g.sorted_w = s_w; g.sorted_e = s_e; g.num_valid = n_valid;
    }
    g.T = tokens; g.topk = topk; g.experts = experts; g.rows = unsorted ? 16 : block_m; g.held = held;
    PairArgs up = g, down = g;
    up.a = hidden_bf16; up.w = w1; up.w_s = w1_scale; up.bias = (const uint16_t*)bias1_bf16;
    up.out = a2; up.K = hidden; up.N = 2 * inter;
    up.a_pitch = (int)row_stride; up.k_real = hidden_cols ? hidden_cols : hidden - hidden_pad; up.n_pad = inter_pad;
    down.a = a2; down.w = w2; down.w_s = w2_scale; down.bias = (const uint16_t*)bias2_bf16;
    down.out = out; down.out_f32 = out_is_f32; down.K = inter; down.N = hidden;
    down.a_pitch = inter; down.k_real = inter - inter_pad; down.n_pad = hidden_pad;
    up.fp4 = down.fp4 = !w4a16;
    if(!w4a16)
    {
        up.out_s = ws + l.a2_s; down.a_s = ws + l.a2_s;
        if(!unsorted)
        {
            // (the sort's launch has quantised the tokens)
            up.a = ws + l.a1_q; up.a_s = ws + l.a1_s; up.a_pitch = hidden;
        }
    }
    // (the kernels that sum a top-2 token's slots read the rows of a2 where the single-token entry points put them, and all of their
    // columns)
    const bool top2 = w4a16 && tokens == 1 && topk == 2;
    up.row_step = down.row_step = top2 ? 16 : 1;
    up.all_channels             = top2;
    if(unsorted && !top2)
    {
        up.tab_ids = s_ids; up.tab_w = s_w; up.tab_e = s_e; up.tab_valid = n_valid;
    }
    // (unsorted 32-row blocks are two of 16)
    const int64_t n_blk = unsorted ? l.n_blk * (block_m / 16) : l.n_blk;
    rc = pyhip_pairs_gate_up(up, tokens, n_blk, split_k, activation, swiglu_limit, stream);
    if(rc)
        return rc;
    if(top2)
    {
        rc = pyhip_w4a16_token_top2(a2, w2, w2_scale, bias2_bf16, topk_ids, topk_weights, expert_mask, num_local_tokens,
                                    out, out_is_f32, topk, experts, hidden, inter, split_k, stream);
        if(rc >= 0)
            return rc;
    }
    rc = pyhip_pairs_down_sum(down, l.rows2, n_blk, split_k, stream);
    if(rc >= 0)
        return rc;
    down.out = ws + l.out3;
    if(up.tab_ids)
    {
        down.ids = nullptr;
        down.sorted_ids = s_ids; down.sorted_w = s_w; down.sorted_e = s_e; down.num_valid = n_valid;
    }
    rc = pyhip_pairs_down(down, l.rows2, n_blk, split_k, stream);
    if(rc)
        return rc;
    return pyhip_moe_topk_reduce_routed(ws + l.out3, out, tokens, topk, hidden, out_is_f32, topk_ids, experts, expert_mask,
                                        num_local_tokens, stream);
}

// hidden_cols = 0: the hidden states are at the padded width; otherwise they have hidden_cols columns, and the input
// quantisation fills in the zeros of the padding (bf16 activations: the GEMM does, and only where bf16_cols allows it)
static int forward_impl(const void* hidden_bf16, int64_t hidden_row_stride, int hidden_cols, const uint8_t* w1, const uint8_t* w1_scale,
                        const uint8_t* w2, const uint8_t* w2_scale, const void* bias1_bf16, const void* bias2_bf16,
                        const Router& router, int32_t* topk_ids, float* topk_weights, const int32_t* expert_mask,
                        const int32_t* num_local_tokens, void* out, int out_is_f32, int tokens, int topk, int experts,
                        int hidden, int inter, int hidden_pad, int inter_pad, int block_m, int w4a16, int split_k,
                        int activation, float swiglu_limit, void* workspace, int64_t workspace_bytes, hipStream_t stream,
                        bool bf16_cols = false, int local_experts = 0)
{
    PYHIP_REQUIRE(hidden_bf16 && w1 && w1_scale && w2 && w2_scale && topk_ids && topk_weights && out,
                  "moe_forward: null pointer");
    PYHIP_REQUIRE(tokens > 0 && topk > 0 && experts > 0 && hidden > 0 && inter > 0, "moe_forward: bad sizes");
    PYHIP_REQUIRE(block_m == 16 || block_m == 32 || block_m == 64 ||
                      ((block_m == 128 || block_m == 160 || block_m == 192 || block_m == 256 || block_m == 288) && !w4a16),
                  "moe_forward: block_m=%d (16/32/64, and 128/160/192/256/288 with MXFP4 activations)", block_m);
    // (the bf16-activation kernels of the step-by-step path look at no padding and take any; those of the pairs would leave their matrices)
    const bool h_fits = hidden_pad >= 0 && hidden_pad < hidden, i_fits = inter_pad >= 0 && inter_pad < inter, pads_fit = h_fits && i_fits;
    // (columns that do not fit are refused with the hidden states)
    PYHIP_REQUIRE(w4a16 || (i_fits && (h_fits || hidden_cols)), "moe_forward: hidden_pad=%d / inter_pad=%d outside [0, hidden=%d) / [0, inter=%d)",
                  hidden_pad, inter_pad, hidden, inter);
    const bool pairs = pads_fit && takes_pairs(tokens, topk, experts, expert_mask ? local_experts : experts, hidden, inter, block_m, w4a16, split_k) &&
                       takes_rows(tokens, hidden_row_stride);
    bf16_cols        = bf16_cols && pairs && hidden_cols > 0 && takes_bf16_cols(tokens, hidden_row_stride, hidden_cols);
    PYHIP_REQUIRE(!w4a16 || hidden_row_stride == hidden || bf16_cols, "moe_forward: the bf16-activation kernels need contiguous rows");
    PYHIP_REQUIRE(hidden_cols == 0 || ((!w4a16 || bf16_cols) && !router.gating && hidden_cols == hidden - hidden_pad && hidden_cols % 32 == 0),
                  "moe_forward: hidden_cols=%d (0, or hidden - hidden_pad, a multiple of 32, with MXFP4 activations)", hidden_cols);
    const Layout l = make_layout(tokens, topk, experts, hidden, inter, block_m, w4a16);
    PYHIP_REQUIRE(workspace && workspace_bytes >= l.total && ((uintptr_t)workspace % 256) == 0,
                  "moe_forward: workspace of %lld bytes (256-byte aligned) needed, %lld given", (long long)l.total,
                  (long long)workspace_bytes);
    uint8_t* ws       = (uint8_t*)workspace;
    uint32_t* s_ids   = (uint32_t*)(ws + l.sorted_ids);
    float* s_w        = (float*)(ws + l.sorted_w);
    uint32_t* s_e     = (uint32_t*)(ws + l.sorted_e);
    uint32_t* n_valid = (uint32_t*)(ws + l.num_valid);
    uint32_t* sched   = (uint32_t*)(ws + l.sched);
    void* out3        = ws + l.out3;
    int rc;
    if(pairs)
        return forward_pairs(hidden_bf16, hidden_row_stride, hidden_cols, w1, w1_scale, w2, w2_scale, bias1_bf16, bias2_bf16, router,
                             topk_ids, topk_weights, expert_mask, num_local_tokens, out, out_is_f32, tokens, topk, experts, hidden,
                             inter, hidden_pad, inter_pad, block_m, w4a16, split_k, activation, swiglu_limit,
                             expert_mask && local_experts > 0 && local_experts < experts ? local_experts : experts, l, ws, stream);
    if(w4a16 && tokens == 1 && !router.gating)
    {
        // a single token with bf16 activations: no sort; the GEMMs read the routing themselves, one block per slot
        rc = pyhip_moe_gemm1_w4a16_token(hidden_bf16, w1, w1_scale, bias1_bf16, topk_ids, expert_mask, num_local_tokens,
                                         ws + l.a2, topk, experts, hidden, inter, split_k, activation, swiglu_limit, stream);
        if(rc)
            return rc;
        // both slots of a top-2 token in one workgroup: the down GEMM writes the layer's output
        rc = pyhip_w4a16_token_top2(ws + l.a2, w2, w2_scale, bias2_bf16, topk_ids, topk_weights, expert_mask, num_local_tokens,
                                    out, out_is_f32, topk, experts, hidden, inter, split_k, stream);
        if(rc >= 0)
            return rc;
        rc = pyhip_moe_gemm2_w4a16_token(ws + l.a2, w2, w2_scale, bias2_bf16, topk_ids, topk_weights, expert_mask,
                                         num_local_tokens, out3, topk, experts, hidden, inter, split_k, stream);
        if(rc)
            return rc;
        return pyhip_moe_topk_reduce_routed(out3, out, tokens, topk, hidden, out_is_f32, topk_ids, experts, expert_mask,
                                            num_local_tokens, stream);
    }
    if(router.gating)
        // the routing is part of the call: the sort's own workgroup routes the tokens when there are few of them
        rc = pyhip_moe_route_sorting(router.gating, tokens, topk, experts, router.n_group, router.topk_group,
                                     router.renormalize, block_m, expert_mask, num_local_tokens, topk_weights, topk_ids,
                                     s_ids, s_w, s_e, n_valid, sched, ws + l.sort_ws, l.sort_ws_bytes,
                                     w4a16 ? nullptr : hidden_bf16, hidden_row_stride, tokens, hidden,
                                     w4a16 ? nullptr : ws + l.a1_q, w4a16 ? nullptr : ws + l.a1_s, stream);
    else if(w4a16)
        rc = pyhip_moe_sorting(topk_ids, topk_weights, tokens, topk, experts, block_m, expert_mask, num_local_tokens,
                               s_ids, s_w, s_e, n_valid, sched, nullptr, 0, ws + l.sort_ws, l.sort_ws_bytes, stream);
    else
        rc = pyhip_sorting_quant_cols(topk_ids, topk_weights, tokens, topk, experts, block_m, expert_mask,
                                      num_local_tokens, s_ids, s_w, s_e, n_valid, sched, ws + l.sort_ws, l.sort_ws_bytes,
                                      hidden_bf16, hidden_row_stride, tokens, hidden, ws + l.a1_q, ws + l.a1_s, hidden_cols,
                                      stream);
    if(rc)
        return rc;
    if(w4a16)
    {
        rc = pyhip_moe_gemm1_w4a16(hidden_bf16, w1, w1_scale, bias1_bf16, s_ids, s_e, n_valid, ws + l.a2, tokens, topk,
                                   experts, hidden, inter, block_m, l.n_blk, split_k, activation, swiglu_limit, stream);
        if(rc)
            return rc;
        rc = pyhip_moe_gemm2_w4a16(ws + l.a2, w2, w2_scale, bias2_bf16, s_ids, s_w, s_e, n_valid, out3, tokens, topk,
                                   experts, hidden, inter, block_m, l.n_blk, split_k, stream);
    }
    else
    {
        rc = pyhip_moe_gemm1_mxfp4(ws + l.a1_q, ws + l.a1_s, w1, w1_scale, bias1_bf16, s_ids, s_e, n_valid, sched, nullptr,
                                   ws + l.a2_q, ws + l.a2_s, tokens, topk, experts, hidden, inter, hidden_pad, inter_pad,
                                   block_m, l.n_blk, activation, swiglu_limit, stream);
        if(rc)
            return rc;
        rc = pyhip_moe_gemm2_mxfp4(ws + l.a2_q, ws + l.a2_s, w2, w2_scale, bias2_bf16, s_ids, s_w, s_e, n_valid, sched,
                                   out3, tokens, topk, experts, hidden, inter, hidden_pad, inter_pad, block_m, l.n_blk, stream);
    }
    if(rc)
        return rc;
    // Slots the sort dropped (ids outside [0, experts), experts this rank does not hold, tokens past the local count)
    // were never written by the down GEMM: the reduction reads the routing and leaves them out, so out3 needs no
    // clearing and the traffic under expert parallelism is that of the owned slots.
    return pyhip_moe_topk_reduce_routed(out3, out, tokens, topk, hidden, out_is_f32, topk_ids, experts, expert_mask,
                                        num_local_tokens, stream);
}

extern "C" int pyhip_moe_forward(const void* hidden_bf16, int64_t hidden_row_stride, const uint8_t* w1,
                                 const uint8_t* w1_scale, const uint8_t* w2, const uint8_t* w2_scale,
                                 const void* bias1_bf16, const void* bias2_bf16, const int32_t* topk_ids,
                                 const float* topk_weights, const int32_t* expert_mask,
                                 const int32_t* num_local_tokens, void* out, int out_is_f32, int tokens, int topk,
                                 int experts, int hidden, int inter, int hidden_pad, int inter_pad, int block_m,
                                 int w4a16, int split_k, int activation, float swiglu_limit, void* workspace,
                                 int64_t workspace_bytes, hipStream_t stream)
{
    return forward_impl(hidden_bf16, hidden_row_stride, 0, w1, w1_scale, w2, w2_scale, bias1_bf16, bias2_bf16, Router{},
                        const_cast<int32_t*>(topk_ids), const_cast<float*>(topk_weights), expert_mask, num_local_tokens,
                        out, out_is_f32, tokens, topk, experts, hidden, inter, hidden_pad, inter_pad, block_m, w4a16,
                        split_k, activation, swiglu_limit, workspace, workspace_bytes, stream);
}

// pyhip_moe_forward for a padded layer whose hidden states come at their true width, hidden_cols = hidden - hidden_pad: the
// quantisation reads them as they are.  Widening them first was a launch and a pass over memory of its own in front of the
// layer: gpt-oss shape (2880 of 3072 columns), before -> after, 16 tokens 126.3 -> 121.7 us, 4096 tokens 543.3 -> 524.7 us.
extern "C" int pyhip_moe_forward_cols(const void* hidden_bf16, int64_t hidden_row_stride, int hidden_cols, const uint8_t* w1,
                                      const uint8_t* w1_scale, const uint8_t* w2, const uint8_t* w2_scale,
                                      const void* bias1_bf16, const void* bias2_bf16, const int32_t* topk_ids,
                                      const float* topk_weights, const int32_t* expert_mask,
                                      const int32_t* num_local_tokens, void* out, int out_is_f32, int tokens, int topk,
                                      int experts, int hidden, int inter, int hidden_pad, int inter_pad, int block_m,
                                      int w4a16, int split_k, int activation, float swiglu_limit, void* workspace,
                                      int64_t workspace_bytes, hipStream_t stream)
{
    return forward_impl(hidden_bf16, hidden_row_stride, hidden_cols, w1, w1_scale, w2, w2_scale, bias1_bf16, bias2_bf16, Router{},
                        const_cast<int32_t*>(topk_ids), const_cast<float*>(topk_weights), expert_mask, num_local_tokens,
                        out, out_is_f32, tokens, topk, experts, hidden, inter, hidden_pad, inter_pad, block_m, w4a16,
                        split_k, activation, swiglu_limit, workspace, workspace_bytes, stream);
}

// The layer with its router: gating scores in, and the picks (topk_ids, topk_weights) out next to the layer output.
// n_group = 0: softmax over the experts, top-k; n_group > 0: sigmoid scores with grouped selection (DeepSeek-V3).
extern "C" int pyhip_moe_forward_routed(const void* hidden_bf16, int64_t hidden_row_stride, const uint8_t* w1,
                                        const uint8_t* w1_scale, const uint8_t* w2, const uint8_t* w2_scale,
                                        const void* bias1_bf16, const void* bias2_bf16, const float* gating, int n_group,
                                        int topk_group, int renormalize, int32_t* topk_ids, float* topk_weights,
                                        const int32_t* expert_mask, const int32_t* num_local_tokens, void* out,
                                        int out_is_f32, int tokens, int topk, int experts, int hidden, int inter,
                                        int hidden_pad, int inter_pad, int block_m, int w4a16, int split_k,
                                        int activation, float swiglu_limit, void* workspace, int64_t workspace_bytes,
                                        hipStream_t stream)
{
    PYHIP_REQUIRE(gating, "moe_forward_routed: null gating scores");
    Router r;
    r.gating = gating; r.n_group = n_group; r.topk_group = topk_group; r.renormalize = renormalize;
    return forward_impl(hidden_bf16, hidden_row_stride, 0, w1, w1_scale, w2, w2_scale, bias1_bf16, bias2_bf16, r, topk_ids,
                        topk_weights, expert_mask, num_local_tokens, out, out_is_f32, tokens, topk, experts, hidden, inter,
                        hidden_pad, inter_pad, block_m, w4a16, split_k, activation, swiglu_limit, workspace, workspace_bytes,
                        stream);
}

// The layer call of pyhip_amd/fused_moe.py in one argument, a block that the caller packs (24 pointers and sizes cost ctypes longer
// one by one).  Also the only entry point that takes hidden states at the true width with bf16 activations
// (pyhip_layer_takes_cols).
struct LayerCall
{
    const void *x, *w1, *w1_scale, *w2, *w2_scale, *bias1, *bias2, *gating, *topk_ids, *topk_weights, *expert_mask, *num_local_tokens;
    void *out, *workspace;
    int64_t row_stride, workspace_bytes;
    int cols, out_f32, tokens, topk, experts, hidden, inter, hidden_pad, inter_pad, block_m, w4a16, split_k, activation;
    int n_group, topk_group, renormalize;
    float swiglu_limit;
    int local_experts;      // matrices in w1 and w2 (under a mask: the experts that it has), or 0: not told
};
static_assert(sizeof(LayerCall) == 200, "packed by pyhip_amd/fused_moe.py");

extern "C" int pyhip_layer_forward(const LayerCall* c, hipStream_t stream)
{
    Router r;
    r.gating = (const float*)c->gating; r.n_group = c->n_group; r.topk_group = c->topk_group; r.renormalize = c->renormalize;
    return forward_impl(c->x, c->row_stride, c->cols, (const uint8_t*)c->w1, (const uint8_t*)c->w1_scale, (const uint8_t*)c->w2,
                        (const uint8_t*)c->w2_scale, c->bias1, c->bias2, r, (int32_t*)c->topk_ids, (float*)c->topk_weights,
                        (const int32_t*)c->expert_mask, (const int32_t*)c->num_local_tokens, c->out, c->out_f32, c->tokens, c->topk,
                        c->experts, c->hidden, c->inter, c->hidden_pad, c->inter_pad, c->block_m, c->w4a16, c->split_k, c->activation,
                        c->swiglu_limit, c->workspace, c->workspace_bytes, stream, true, c->local_experts);
}

// Whether a call of these sizes runs the kernels of moe_gemm_pairs.hip (for whoever reports on it)
extern "C" int pyhip_layer_takes_pairs(int64_t tokens, int topk, int experts, int hidden, int inter, int block_m, int w4a16, int split_k)
{
    return takes_pairs(tokens, topk, experts, experts, hidden, inter, block_m, w4a16, split_k);
}

// Whether hidden states at the true width of a padded layer, rows row_stride apart, are taken as they are
extern "C" int pyhip_layer_takes_cols(int64_t tokens, int topk, int experts, int hidden, int inter, int block_m, int w4a16, int split_k,
                                      int64_t row_stride)
{
    return !w4a16 || (takes_pairs(tokens, topk, experts, experts, hidden, inter, block_m, w4a16, split_k) && takes_bf16_cols(tokens, row_stride, 0));
}
