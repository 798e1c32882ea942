// Routed feed-forwards of up to 16 rows: the norm that makes their input, the router's product and the choice of experts in one launch; the list of rows by expert is made by the
// experts' first product on its way (few_rows.hip).  They were four launches, of which three of 4 us each moved next to nothing (a launch that reads what the one before
// wrote ends no sooner than 3.5 us after it).
//
// A workgroup a row.  Four of its waves make the row; the other eight have asked for the router's weights (128 KB for 32 experts of 2048) by then, in registers, and multiply them with
// the row from LDS.  The sums are those of the product of few rows (16 sums of every 16th k tile, added in order), so the logits and the experts are the same bits.  (With the list
// made here, by the workgroup that comes last, a step of eight rows gained half as much: the way past the dies' caches and back takes as long as a launch.)
#include "norm_route.hpp"
#include "route.hpp"
#include "sublayer_rows.hpp"

namespace {

constexpr int kRowWaves = kM40RowThreads / 64, kProductWaves = 8, kThreads = 64 * (kRowWaves + kProductWaves);
constexpr int kParts = 16;                               // sums of a product
constexpr uint32_t kMostWidth = 4096;

struct NormAddRow {
    using Args = M40llmNormAdd;
    template <class Sink>
    static __device__ __forceinline__ void make(const Args& a, uint32_t row, uint32_t tid, float* scratch, const Sink& sink) { m40_norm_add_row<m40_bf16, true>(a, row, tid, scratch, sink); }
};
template <int S>
struct StreamRow {
    using Args = M40llmStreamUpdate;
    template <class Sink>
    static __device__ __forceinline__ void make(const Args& a, uint32_t row, uint32_t tid, float* scratch, const Sink& sink) { m40_stream_update_row<m40_bf16, S, true>(a, row, tid, scratch, sink); }
};

// TILES: column tiles of the router's weights, at most
template <class Row, int TILES>
__global__ __launch_bounds__(kThreads) void norm_route_kernel(const m40_bf16* weights, int k_tiles, int n_tiles, M40llmRoute q, typename Row::Args a) {
    constexpr int kAhead = TILES > 3 ? 6 : 8;            // k tiles a wave has in registers: an even number
    __shared__ float scratch[kRowWaves];
    __shared__ __align__(16) m40_bf16 row_s[kMostWidth];
    __shared__ __align__(16) float sums[kParts][TILES * 16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, row = blockIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), part = wave - kRowWaves;
    // The row's waves and the product's go separate ways to as many barriers each, those within the row and one behind it (left in one way the weights' registers would not fit beside
    // the row's).
    if (part < 0) {
        Row::make(a, row, tid, scratch, [&](uint32_t g, const m40_float4& lo, const m40_float4& hi) {        // kM40RowBarriers inside
            m40_store8<m40_bf16>(row_s + g * 8u, lo, hi);
            m40_store_input<m40_bf16>(a, row, g, lo, hi);
        });
        __syncthreads();
    } else {
        uint4 w[kAhead][TILES];
        auto request = [&](int k) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int kt = k + u * kProductWaves;
                if (kt >= k_tiles) break;
#pragma unroll
                for (int t = 0; t < TILES; ++t) w[u][t] = *reinterpret_cast<const uint4*>(weights + ((size_t)(t < n_tiles ? t : n_tiles - 1) * k_tiles + kt) * kM40Tile + lane * 8);
            }
        };
        request(part);
#pragma unroll
        for (int i = 0; i < kM40RowBarriers + 1; ++i) __syncthreads();
        m40_float4 acc[2][TILES];            // k tiles part, part + 16, ... and part + 8, part + 24, ...
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < TILES; ++t) acc[h][t] = m40_float4{0.f, 0.f, 0.f, 0.f};
        for (int k = part;;) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int kt = k + u * kProductWaves;
                if (kt >= k_tiles) break;
                const m40_bf16x8 x = *reinterpret_cast<const m40_bf16x8*>(row_s + kt * 32 + (lane >> 4) * 8);      // every row of the operand is this one
#pragma unroll
                for (int t = 0; t < TILES; ++t) acc[u & 1][t] = M40Act<m40_bf16>::mma(__builtin_bit_cast(m40_bf16x8, w[u][t]), x, acc[u & 1][t]);
            }
            k += kAhead * kProductWaves;
            if (k >= k_tiles) break;
            request(k);
        }
        if ((lane & 15u) == 0u) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < TILES; ++t) *reinterpret_cast<m40_float4*>(&sums[part + h * kProductWaves][t * 16 + 4 * (lane >> 4)]) = acc[h][t];
        }
    }
    float correction[1];
    m40_route_corrections<1>(q, lane, correction);
    __syncthreads();
    if (wave == 0) {
        const uint32_t e = lane < TILES * 16u ? lane : 0u;
        float z[1] = {sums[0][e]};
#pragma unroll
        for (int i = 1; i < kParts; ++i) z[0] += sums[i][e];
        m40_route_logits<1>(q, lane, z, correction, q.ids + row * q.top, static_cast<float*>(q.weight) + row * q.top);
    }
}

template <class Row>
int launch(hipStream_t stream, const typename Row::Args& a) {
    const M40llmRoute* q = static_cast<const M40llmRoute*>(a.route);
    if (a.act_dtype != M40LLM_ACT_BF16 || !a.router || !m40_aligned16(a.router) || a.rows > 16u || q->rows != a.rows || a.ld_h < 2048u || a.ld_h > kMostWidth || a.router_tiles == 0 || a.router_tiles > 4u || q->experts + q->identity > a.router_tiles * 16u)
        return -3;
    const m40_bf16* w = static_cast<const m40_bf16*>(a.router);
    const int k_tiles = (int)(a.ld_h / 32u), n_tiles = (int)a.router_tiles;
    if (n_tiles <= 2) norm_route_kernel<Row, 2><<<a.rows, kThreads, 0, stream>>>(w, k_tiles, n_tiles, *q, a);
    else if (n_tiles == 3) norm_route_kernel<Row, 3><<<a.rows, kThreads, 0, stream>>>(w, k_tiles, n_tiles, *q, a);
    else norm_route_kernel<Row, 4><<<a.rows, kThreads, 0, stream>>>(w, k_tiles, n_tiles, *q, a);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace

int m40_norm_add_route(hipStream_t stream, const M40llmNormAdd& n) { return launch<NormAddRow>(stream, n); }
int m40_stream_update_route(hipStream_t stream, const M40llmStreamUpdate& u) {
    if (u.streams == 1u) return launch<StreamRow<1>>(stream, u);
    return u.streams == 4u ? launch<StreamRow<4>>(stream, u) : -3;
}
