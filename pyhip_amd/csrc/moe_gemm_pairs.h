// The layer call's GEMMs for few tokens (moe_gemm_pairs.hip): what moe_forward.hip hands them.
#pragma once
#include "common.h"

struct PairArgs
{
    const void* a      = nullptr;   // activations bf16, rows of a_pitch: gate_up: tokens; down: a2 ...
    const uint8_t* a_s = nullptr;   // ... or e2m1 pairs with these scales: gate_up [T, K/2] (layout: moe_quant.hip), down what gate_up wrote
    const uint8_t* w   = nullptr;   // weights, pre-shuffled    [E, N, K/2]
    const uint8_t* w_s = nullptr;   // weight scales, shuffled  [E*N (padded to 256), SC]
    const uint16_t* bias = nullptr; // bf16 [E, N] or null
    // bf16 a2 has a row for every pair, pair t * topk + slot in row pair * row_step; quantised a2 one for each row of the blocks.
    // The routing as the caller gave it, read by the kernels themselves (at most PAIRS_UNSORTED_MAX pairs) ...
    const int* ids       = nullptr;   // [T, topk], or null: the sort's output below (row_step 1)
    const float* weights = nullptr;   // [T, topk] (down)
    const int* mask      = nullptr;   // [experts] or null
    const int* local_tok = nullptr;   // device scalar or null
    // ... or sorted into blocks (moe_sort.hip)
    const u32* sorted_ids = nullptr;
    const float* sorted_w = nullptr;
    const u32* sorted_e   = nullptr;
    const u32* num_valid  = nullptr;
    // gate_up, unsorted: where it leaves the blocks that it has found, in that form, or null
    u32* tab_ids   = nullptr;
    float* tab_w   = nullptr;
    u32* tab_e     = nullptr;
    u32* tab_valid = nullptr;
    void* out = nullptr;              // gate_up: a2 bf16 [.., N/2], or (fp4) e2m1 pairs, in tiles; down: out3 bf16 [T, topk, N]; down that sums: [T, N]
    uint8_t* out_s = nullptr;         // gate_up, fp4: the scales of a2
    int rows = 16;                    // of a block; 32, 64: sorted, activations quantised
    int T = 0, topk = 0, experts = 0, K = 0, N = 0;
    int held = 0;                     // experts that are here (mask: how many it has)
    int a_pitch = 0, row_step = 1;
    int k_real = 0;                   // columns of the weights that are not padding ...
    int n_pad  = 0;                   // ... and rows of (each half of) an expert's matrix that are
    int all_channels = 0;             // gate_up: channels of padding are written as well (zeros), for a reader that does not know of them
    int out_f32 = 0;                  // down that sums: the type of its output
    int fp4 = 0;                      // the layer's activations are MXFP4: bf16 ones are rounded to it (not for the down that sums)
    // filled in by the launchers
    int SC = 0, n_tiles = 0;
    u32 a_bytes = 0, as_bytes = 0;
    int swiglu = 0;
    GatedAct act = {};
};

#define PAIRS_UNSORTED_MAX 128

// Whether these kernels have the K splits that the sorted entry points take for such a call (split_k as there)
bool pyhip_pairs_served(int64_t tokens, int topk, int experts, int hidden, int inter, int64_t n_blk, int fp4, int split_k);
// rows: of a; n_blk: bound of the row blocks (pyhip_moe_sorting_max_blocks)
int pyhip_pairs_gate_up(PairArgs g, int64_t rows, int64_t n_blk, int split_k, int activation, float swiglu_limit, hipStream_t stream);
int pyhip_pairs_down(PairArgs g, int64_t rows, int64_t n_blk, int split_k, hipStream_t stream);
// the down GEMM that also sums a token's slots and writes the layer's output; -1 where it does not serve the call
int pyhip_pairs_down_sum(PairArgs g, int64_t rows, int64_t n_blk, int split_k, hipStream_t stream);
