// dcq_attn.h — what the attention kernels (dcq_kv.hip, dcq_attn_prompt.hip) share.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dcq {

struct AttnArgs {
    const uint8_t* k_arena;
    const uint8_t* v_arena;
    int n_blocks, n_layer, layer;
    int64_t sb;  // slot bytes
    const int32_t* table;
    int n_table;
    const float* q;
    int64_t q_stride;  // floats between query tokens
    const float* k_cur;
    const float* v_cur;
    int64_t kv_stride;  // floats between current K (V) rows
    float* out;
    int64_t out_stride;
    float* ws_o;  // [splits][N][n_head][HD]
    float* ws_ml;  // [splits][N][n_head][2]
    int n_tokens, n_past, n_head, n_head_kv, hpw, nq;
    int nch_hist, nch_total, cps;  // chunks of history, all chunks, chunks per split
    int splits, groups;
    float scale_log2e;
};

// dcq_attn_prompt.hip: many query rows, on f16 MFMA pieces of the fp32 operands. cps counts its key
// blocks of 32 per split; with splits > 1 the partial results go to ws_o / ws_ml.
hipError_t launch_attn_prompt(int ct, int hd, const AttnArgs& a, hipStream_t st);

}  // namespace dcq
