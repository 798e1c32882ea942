// Launch parameters shared by the dense attention kernels (attention.hip, attention_mfma.hip).
#pragma once

#include "packed_rows.hpp"

// One argument of 112 bytes for each kernel: launches one by one are bound by the host, and more bytes or the members as arguments of their own cost it time (one row,
// one launch: 3.6 us, 4.2 with 136 bytes, 4.5 as ten arguments; two launches 7.0, 8.0 with eleven and nine).
struct AttnParams {
    const uint16_t* K;
    const uint16_t* V;
    const float* Q;
    void* out;                    // f32 rows, or with `packed` rows as operands of the next product (packed_rows.hpp)
    float* ws;                    // partials: sums [batch][q_heads][nchunks][hd], behind them
    const uint32_t* seq_ids_dev;  // may be null
    const uint32_t* seq_lens_dev; // may be null
    uint32_t ml_from;             // [batch][q_heads][nchunks][2]: maximum and denominator, that many floats behind ws
    uint32_t packed;              // 0, or the operands' padded rows
    uint32_t seq_id;
    uint32_t len_or_bias;         // the length, or what is added to a device-side one (position -> length)
    uint32_t max_seq_len, kv_heads, q_heads, window;
    uint32_t chunk, nchunks;
    uint32_t subgroups;           // q-head subgroups per kv head
    uint32_t max_batch;           // device-side sequence ids at or above this are skipped (0 = not checked)
    uint32_t span_limit;          // tokens a row may attend (the length bound the grid and chunking were sized for): rows
                                  // whose device-side length asks for more are skipped
    __device__ __forceinline__ uint32_t length(uint32_t b) const { return seq_lens_dev ? seq_lens_dev[b] + len_or_bias : len_or_bias; }
    __device__ __forceinline__ float2* ml() const { return reinterpret_cast<float2*>(ws + ml_from); }
};

// Element d of q head qh of row b; called by the lanes of whole groups of eight d.
template <int HD>
__device__ __forceinline__ void m40_attn_store(const AttnParams& p, uint32_t b, uint32_t qh, uint32_t d, float y) {
    if (p.packed) m40_store_packed(static_cast<uint8_t*>(p.out), (int)p.packed, (int)p.q_heads * HD, (int)b, (int)(qh * HD + d), y);
    else static_cast<float*>(p.out)[((size_t)b * p.q_heads + qh) * HD + d] = y;
}

// One head's chunk partials (sums [chunks][HD], pairs of maximum and denominator [chunks]) merged by a workgroup of 256: HD / 4 lanes take a chunk's sums, four
// columns each; the chunks go round the 1024 / HD such groups.
//
// Bound by its round trips to memory: everything of the first PASS chunks is asked for at once, before it is known how many there are; partials of chunks past
// the row's end are stale values inside the buffer and are left out; an empty chunk (maximum -inf, sums of 0) has no weight.  Every wave forms all weights itself, one
// lane a chunk, so that the waves meet once, with their sums.  (Folding the chunks one after the other under a running maximum, 256 / HD of them side by side:
// the two launches of 8 rows of up to 4093 tokens, head size 128, 13.3 us, now 12.6; 32 rows of up to 1021, 64, 11.8 / 11.3; 2 rows of up to 3000 10.3 / 8.9; one of
// 16000, 125 chunks, 19.6 / 11.8.)
//
// PASS: how many chunks are asked for at once; 64 go on to the next ones, with fewer there must be no more.
template <int HD, int PASS>
struct M40ChunkMerge {
    static constexpr int kLanes = HD / 4, kGroups = 256 / kLanes, kPass = PASS, kEach = kPass / kGroups;
    const float4* v_at;
    const float2* ml_at;
    uint32_t stored, lane, group;
    float4 v[kEach];
    float2 ml0;
    __device__ __forceinline__ void load(uint32_t base) {
#pragma unroll
        for (int u = 0; u < kEach; ++u) {
            const uint32_t c = base + group + u * kGroups;
            v[u] = v_at[(size_t)(c < stored ? c : 0u) * kLanes];
        }
    }
    __device__ __forceinline__ void request(const float* sums, const float2* ml, uint32_t chunks_stored) {
        lane = threadIdx.x & 63; group = threadIdx.x / kLanes; stored = chunks_stored;
        v_at = reinterpret_cast<const float4*>(sums) + threadIdx.x % kLanes;
        ml_at = ml;
        ml0 = ml_at[lane < stored ? lane : 0u];
        load(0);
    }
    // element threadIdx.x of the result, in the first HD threads; n <= stored
    __device__ __forceinline__ float finish(uint32_t n, float (*sums)[HD]) {
        float m = lane < n ? ml0.x : -INFINITY;
        if (kPass == 64)
            for (uint32_t c = kPass + lane; c < n; c += kPass) m = fmaxf(m, ml_at[c].x);
        m = m40_max64(m);
        float den = 0.0f;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        for (uint32_t base = 0; base < (kPass == 64 ? n : 1u); base += kPass) {
            const float2 x = base == 0 ? ml0 : ml_at[base + lane < n ? base + lane : 0u];
            if (base != 0) load(base);
            const bool live = base + lane < n && x.x != -INFINITY;
            const float f = live ? expf(x.x - m) : 0.0f;
            den = fmaf(live ? x.y : 0.0f, f, den);
#pragma unroll
            for (int u = 0; u < kEach; ++u) {
                const uint32_t c = group + u * kGroups;
                const float w = __shfl(f, (int)c, 64);
                if (base + c < n) {
                    sum.x = fmaf(v[u].x, w, sum.x); sum.y = fmaf(v[u].y, w, sum.y);
                    sum.z = fmaf(v[u].z, w, sum.z); sum.w = fmaf(v[u].w, w, sum.w);
                }
            }
        }
        den = m40_sum64(den);
        if (HD == 64) { sum.x = m40_add_xor16(sum.x); sum.y = m40_add_xor16(sum.y); sum.z = m40_add_xor16(sum.z); sum.w = m40_add_xor16(sum.w); }
        sum.x = m40_add_xor32(sum.x); sum.y = m40_add_xor32(sum.y); sum.z = m40_add_xor32(sum.z); sum.w = m40_add_xor32(sum.w);
        if (lane < kLanes) *reinterpret_cast<float4*>(&sums[threadIdx.x >> 6][4 * lane]) = sum;
        __syncthreads();
        if (threadIdx.x >= HD) return 0.0f;
        const float num = (sums[0][threadIdx.x] + sums[1][threadIdx.x]) + (sums[2][threadIdx.x] + sums[3][threadIdx.x]);
        return num / (den > 0.0f ? den : 1.0f);
    }
};

// attention_mfma.hip: chunks of `p.chunk` tokens (a multiple of 128), G <= 8 q heads per workgroup
void m40_launch_attn_mfma(hipStream_t stream, const AttnParams& p, uint32_t head_dim, uint32_t batch);
