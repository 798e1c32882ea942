// Launch parameters shared by the dense attention kernels (attention.hip, attention_mfma.hip).
#pragma once

#include "packed_rows.hpp"

struct AttnParams {
    const uint16_t* K;
    const uint16_t* V;
    const float* Q;
    float* Out;
    uint8_t* packed;              // not null: rows as operands of the next product (packed_rows.hpp) instead of Out
    uint32_t packed_pad;
    float* ws;                    // partials: sums [batch][q_heads][nchunks][hd], behind them
    float* ml;                    // [batch][q_heads][nchunks][2]: maximum and denominator
    const uint32_t* seq_ids_dev;  // may be null
    const uint32_t* seq_lens_dev; // may be null
    uint32_t seq_id, seq_len;
    uint32_t max_seq_len, kv_heads, q_heads, window;
    uint32_t chunk, nchunks;
    uint32_t subgroups;           // q-head subgroups per kv head
    uint32_t len_bias;            // added to a device-side length (position -> length)
    uint32_t max_batch;           // device-side sequence ids at or above this are skipped (0 = not checked)
    uint32_t span_limit;          // tokens a row may attend (the length bound the grid and chunking were sized for): rows
                                  // whose device-side length asks for more are skipped
};

// Element d of q head qh of row b; called by the lanes of whole groups of eight d.
template <int HD>
__device__ __forceinline__ void m40_attn_store(const AttnParams& p, uint32_t b, uint32_t qh, uint32_t d, float y) {
    if (p.packed) m40_store_packed(p.packed, (int)p.packed_pad, (int)p.q_heads * HD, (int)b, (int)(qh * HD + d), y);
    else p.Out[((size_t)b * p.q_heads + qh) * HD + d] = y;
}

// attention_mfma.hip: chunks of `p.chunk` tokens (a multiple of 128), G <= 8 q heads per workgroup
void m40_launch_attn_mfma(hipStream_t stream, const AttnParams& p, uint32_t head_dim, uint32_t batch);
