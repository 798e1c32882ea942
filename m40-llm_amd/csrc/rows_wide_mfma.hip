// Row-batched projections of a decode step for 9 to 32 activation rows (f32) against f16 GGUF weights [N][K], one launch per
// projection on v_mfma_f32_16x16x32_f16.
//
// rows_mfma.hip keeps eight whole rows as operand fragments in LDS, which more rows do not fit; skinny_mfma.hip converts every step
// of the rows once per 64 columns and adds its K slices in a second launch, and reads the weights once per sixteen rows.  Here a
// workgroup of eight waves owns T column tiles, and a wave walks blocks of 64 k, every eighth: it turns its block of the rows into f16 hi + lo
// operands (one power-of-two scale per row and block, RMSNorm weights folded in, the RMS factor applied to the sums) and multiplies them
// with its block of every tile.  The waves share nothing until their sums meet in LDS once, after the last block, pair by pair.  So the weights
// are read once for all rows, every result is written once, nothing is left for a second launch and no result depends on timing.
//
// Bound: a launch of one tile a workgroup has about 5 us that no block takes part in (launch, arguments and first requests 2.5, sums and results
// 2), and a block then costs a wave 1.3 us: rows in (8 KB from L2), two passes through LDS, about 200 vector instructions, and two waves a
// SIMD to hide them.  The rows are asked for a quarter of a kilobyte of four rows at a time, whole lines: in operand order (16 rows of 64 bytes an
// instruction) every workgroup reading 32 rows of 2048 takes 11.5 us instead of 4.7.  Requests go out one block ahead and no further: two or
// four blocks of weights or rows on their way (more code, more registers, waits for what was asked for later) take 0.6 to 1.4 us more a launch.
// 32 rows, width 2048, feed-forward 5632, against the form that converted chunks of 512 k for all waves between barriers: Q/K/V 13.9 -> 11.5 us, O
// 7.6 -> 6.7, gate/up 19.0 -> 15.7, down 14.6 -> 11.8, vocabulary of 32000 39.4 -> 35.2; 16 rows 10.1 -> 8.3, 6.2 -> 5.4, 14.6 -> 13.8, 11.4 -> 10.0,
// 31.4 -> 30.5.  (O and down of a decode step come as operands and go to packed_rows.hip: 6.0 and 10.8 us; the residual form here is for f32 rows.)  Weight loads are whole 128-byte lines (eight lanes a column) and pass through a wave-private LDS tile into operand order, as in
// rows_mfma.hip.  A product of few columns onto zeros is cut into two halves of K, which meet in the result element by element: two terms, the
// same bits in either order.
#include "packed_rows.hpp"

#include <type_traits>

namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kShare = 64;                              // k of a block: what one wave converts and multiplies at a time
constexpr int kSteps = kShare / 32;                     // matrix instructions deep
constexpr int kRunLanes = kShare * 2 / 16;              // lanes that cover a column's block with 16 bytes each
constexpr int kColsPerLoad = 64 / kRunLanes;
constexpr int kLoads = 16 / kColsPerLoad;
constexpr int kStageRow = kShare * 2 + 16;              // LDS bytes per column: +16 spreads the columns over the banks
constexpr int kStageBytes = 16 * kStageRow;             // of one column tile
constexpr int kRowBytes = kShare * 4 + 16;              // LDS bytes per row

constexpr int wide_stages(int t) { return t > 1 ? 2 : 1; }      // column tiles a wave has in LDS

enum Mode { kResidual = 0, kSwiglu = 1, kQkv = 2, kNorm = 3 };

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ m40_float4 mfma16x16x32(const uint4& a, const uint4& b, m40_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(m40_half8, a), __builtin_bit_cast(m40_half8, b), c, 0, 0, 0);
}

struct WideArgs {
    const float* x;               // [rows][K]
    const void* norm_w;           // RMSNorm weights (all modes but kResidual)
    uint32_t norm_dtype;          // 0 f16, 1 f32
    float eps;
    const uint16_t *W0, *W1, *W2; // kSwiglu: gate, up; kQkv: q, k, v
    float* out;                   // [rows][N]
    uint8_t* packed;              // kSwiglu: not null, the result goes here as operands of the next product instead (N a multiple of 8)
    const float* residual;        // kResidual: added to the product, or null
    int rows, N, K, tiles, blocks;
    float* zero;                  // cleared on the side, or null
    int zero_count;
    const float *bq, *bk, *bv;
    float* q_out;
    uint16_t *k_cache, *v_cache;
    uint32_t* seq_map;
    const uint32_t *ids_dev, *lens_dev;
    const float* rope_table;      // pair frequencies, or null
    uint32_t max_seq_len, max_batch, q_heads, kv_heads, head_dim, rope_layout;
    float rope_base, rope_scale;
};

// A Q/K/V tile: 16 columns of one head that hold eight whole rotation pairs (split-half layout: eight columns and their partners half a
// head further on).
struct QkvTile {
    int which, head, tt;
    bool split;
};
__device__ __forceinline__ QkvTile qkv_tile(const WideArgs& p, int tile) {
    const int tph = (int)p.head_dim / 16, qt = (int)p.q_heads * tph, kt = (int)p.kv_heads * tph;
    QkvTile t;
    t.which = tile < qt ? 0 : (tile < qt + kt ? 1 : 2);
    const int local = tile - (t.which == 0 ? 0 : (t.which == 1 ? qt : qt + kt));
    t.head = local / tph;
    t.tt = local % tph;
    t.split = t.which != 2 && p.rope_layout == M40LLM_ROPE_LAYOUT_NEOX;
    return t;
}
__device__ __forceinline__ int qkv_col(const WideArgs& p, const QkvTile& t, int i) {
    const int hd = (int)p.head_dim;
    return t.split ? t.head * hd + (i & 8 ? hd / 2 : 0) + 8 * t.tt + (i & 7) : t.head * hd + 16 * t.tt + i;
}

// RT: tiles of 16 rows; T: column tiles per workgroup.  grid (ceil(tiles / T), parts of K)
template <int MODE, int RT, int T>
__global__ __launch_bounds__(kThreads, 1) void rows_wide_kernel(WideArgs p) {
    constexpr bool NORM = MODE != kResidual;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(16))) float scale_s[kWaves][16 * RT];      // undoes the scaling of each row's block
    __shared__ float square_s[kWaves][16 * RT];
    __shared__ float factor_s[16 * RT];                                          // RMSNorm factor of each row

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int b_begin = p.blocks * (int)blockIdx.y / (int)gridDim.y, b_end = p.blocks * ((int)blockIdx.y + 1) / (int)gridDim.y;
    const int tile0 = (int)blockIdx.x * T;
    constexpr int kStages = wide_stages(T);
    uint8_t* stage = lds + wave * (kStages * kStageBytes + 16 * kRowBytes);
    uint8_t* rows_lds = stage + kStages * kStageBytes;

    // ---- what a thread's element needs besides the product (one tile a workgroup), asked for before anything else
    const int e_j = tid & 15, e_row = (tid >> 4) & (16 * RT - 1);
    int q_which = 0, q_col = 0, q_partner = 0;
    bool q_second = false;
    uint32_t q_position = 0, q_seq = 0, q_off = 0;
    float bias_own = 0.0f, bias_other = 0.0f, residual_own = 0.0f;
    if (MODE == kResidual && T == 1 && p.residual) {
        const int col = 16 * tile0 + e_j;
        residual_own = p.residual[(size_t)(e_row < p.rows ? e_row : 0) * p.N + (col < p.N ? col : 0)];
    }
    if (MODE == kQkv) {
        const QkvTile t = qkv_tile(p, tile0);
        const int e_rowc = e_row < p.rows ? e_row : 0;
        q_which = t.which;
        q_col = qkv_col(p, t, e_j);
        q_partner = t.split ? e_j ^ 8 : e_j ^ 1;
        q_second = t.split ? (e_j & 8) != 0 : (e_j & 1) != 0;
        q_off = t.split ? (uint32_t)(8 * t.tt + (e_j & 7)) : (uint32_t)((16 * t.tt + e_j) >> 1);
        const float* bias = t.which == 0 ? p.bq : (t.which == 1 ? p.bk : p.bv);
        q_position = p.lens_dev[e_rowc];
        q_seq = p.ids_dev[e_rowc];
        bias_own = bias ? bias[q_col] : 0.0f;
        bias_other = bias ? bias[qkv_col(p, t, q_partner)] : 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- rows of a block, one ahead: lane (j, g) asks for the elements 4 j .. 4 j + 3 of rows g, 4 + g, 8 + g, ...
    constexpr int kRowLoads = 4 * RT;
    uint32_t x_at[kRowLoads];
#pragma unroll
    for (int u = 0; u < kRowLoads; ++u) x_at[u] = (uint32_t)(4 * u + g < p.rows ? 4 * u + g : 0) * (uint32_t)p.K + 4u * j;
    float4 x[kRowLoads];
    uint4 nw;
    const bool norm16 = NORM && p.norm_dtype == 0u;
    auto load_rows = [&](int kb) {
        kb = kb < b_end ? kb : 0;         // past the end: a valid address, the values are not used
        const float* from = p.x + (size_t)kb * kShare;
#pragma unroll
        for (int u = 0; u < kRowLoads; ++u) x[u] = *reinterpret_cast<const float4*>(from + x_at[u]);
        // f16 weights: the sixteen bytes that hold the lane's four
        if (NORM) nw = *(static_cast<const uint4*>(p.norm_w) + (norm16 ? kb * (kShare / 8) : kb * (kShare / 4)) + (norm16 ? j >> 1 : j));
    };
    load_rows(b_begin + wave);
    __builtin_amdgcn_sched_barrier(0);

    // ---- weights: instruction li of a wave reads its 64 k of columns 8 li .. 8 li + 7 of a tile
    const int run_lane = lane % kRunLanes, run_col = lane / kRunLanes;
    const uint16_t* tile_w[T][kLoads];
    uint32_t w_at[T][kLoads];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int tile = tile0 + t < p.tiles ? tile0 + t : p.tiles - 1;
        if (MODE == kQkv) {
            const QkvTile q = qkv_tile(p, tile);
            const int first = qkv_col(p, q, 0);
#pragma unroll
            for (int li = 0; li < kLoads; ++li) {
                tile_w[t][li] = (q.which == 0 ? p.W0 : (q.which == 1 ? p.W1 : p.W2)) + (size_t)first * p.K;
                w_at[t][li] = (uint32_t)(qkv_col(p, q, li * kColsPerLoad + run_col) - first) * (uint32_t)p.K + 8u * run_lane;
            }
        } else {
            constexpr int kCols = MODE == kSwiglu ? 8 : 16;
#pragma unroll
            for (int li = 0; li < kLoads; ++li) {
                const int c = MODE == kSwiglu ? run_col : li * kColsPerLoad + run_col, left = p.N - 1 - kCols * tile;
                tile_w[t][li] = (MODE == kSwiglu && li * kColsPerLoad >= 8 ? p.W1 : p.W0) + (size_t)(kCols * tile) * p.K;
                w_at[t][li] = (uint32_t)(c < left ? c : left) * (uint32_t)p.K + 8u * run_lane;
            }
        }
    }
    uint4 b[T][kLoads];
    auto issue = [&](int kb, int t) {
        kb = kb < b_end ? kb : 0;       // past the end: a valid address, the value is not used
#pragma unroll
        for (int li = 0; li < kLoads; ++li) b[t][li] = *reinterpret_cast<const uint4*>(tile_w[t][li] + (size_t)kb * kShare + w_at[t][li]);
    };
#pragma unroll
    for (int t = 0; t < T; ++t) issue(b_begin + wave, t);
    __builtin_amdgcn_sched_barrier(0);

    // ---- rows of a block -> f16 hi + lo operands, through an LDS tile of the wave's own: lane (j, g) takes the elements k = 32 i + 8 g .. + 7
    // of rows j and 16 + j
    float sq[kRowLoads];
    uint4 hi[RT][kSteps], lo[RT][kSteps];
#pragma unroll
    for (int u = 0; u < kRowLoads; ++u) sq[u] = 0.0f;
    auto convert = [&]() {
        float m[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if (NORM) {
            const uint4 w = nw;
            const uint32_t w0 = j & 1 ? w.z : w.x, w1 = j & 1 ? w.w : w.y;
            m[0] = norm16 ? m40_h2f((uint16_t)(w0 & 0xffffu)) : __uint_as_float(w.x);
            m[1] = norm16 ? m40_h2f((uint16_t)(w0 >> 16)) : __uint_as_float(w.y);
            m[2] = norm16 ? m40_h2f((uint16_t)(w1 & 0xffffu)) : __uint_as_float(w.z);
            m[3] = norm16 ? m40_h2f((uint16_t)(w1 >> 16)) : __uint_as_float(w.w);
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
            for (int u = 4 * rt; u < 4 * rt + 4; ++u) {
                const float4 a = x[u];
                if (NORM) sq[u] = fmaf(a.x, a.x, fmaf(a.y, a.y, fmaf(a.z, a.z, fmaf(a.w, a.w, sq[u]))));
                *reinterpret_cast<f32x4*>(rows_lds + (4 * (u & 3) + g) * kRowBytes + 16 * j) = NORM ? f32x4{a.x * m[0], a.y * m[1], a.z * m[2], a.w * m[3]} : f32x4{a.x, a.y, a.z, a.w};
            }
            __builtin_amdgcn_wave_barrier();
            f32x4 v[kSteps][2];
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) v[i][h] = *reinterpret_cast<const f32x4*>(rows_lds + j * kRowBytes + 128 * i + 32 * g + 16 * h);
            __builtin_amdgcn_wave_barrier();
            float mx = 0.0f;
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int e = 0; e < 4; e += 2) mx = fmaxf(fmaxf(mx, fabsf(v[i][h][e])), fabsf(v[i][h][e + 1]));
            mx = m40_max_xor32(m40_max_xor16(mx));      // over the row's block
            float scale = 1.0f, inv_scale = 1.0f;
            if (mx > 0.0f && mx < INFINITY) {
                int ex;
                (void)frexpf(mx, &ex);            // mx = f * 2^ex, f in [0.5, 1)
                ex -= 11;                         // scaled maximum in [2^10, 2^11)
                ex = ex < -100 ? -100 : (ex > 100 ? 100 : ex);
                scale = ldexpf(1.0f, ex);
                inv_scale = ldexpf(1.0f, -ex);
            }
            if (g == 0) scale_s[wave][16 * rt + j] = scale;
#pragma unroll
            for (int i = 0; i < kSteps; ++i) {
                // hi = f16(v / scale), lo = f16(v / scale - hi): an instruction each (a multiply-add of mixed widths, rounded to f16)
                f16x2 h2[4], l2[4];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float y = v[i][e >> 2][e & 3];
                    h2[e >> 1][e & 1] = static_cast<_Float16>(fmaf(y, inv_scale, -0.0f));
                    l2[e >> 1][e & 1] = static_cast<_Float16>(fmaf(y, inv_scale, -static_cast<float>(h2[e >> 1][e & 1])));
                }
                hi[rt][i] = make_uint4(__builtin_bit_cast(uint32_t, h2[0]), __builtin_bit_cast(uint32_t, h2[1]), __builtin_bit_cast(uint32_t, h2[2]), __builtin_bit_cast(uint32_t, h2[3]));
                lo[rt][i] = make_uint4(__builtin_bit_cast(uint32_t, l2[0]), __builtin_bit_cast(uint32_t, l2[1]), __builtin_bit_cast(uint32_t, l2[2]), __builtin_bit_cast(uint32_t, l2[3]));
            }
        }
        __builtin_amdgcn_wave_barrier();
    };

    m40_float4 total[T][RT];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) total[t][rt] = {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const uint8_t* from, int t) {
        m40_float4 acc[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt] = {0.f, 0.f, 0.f, 0.f};
        uint4 bw[kSteps];
#pragma unroll
        for (int i = 0; i < kSteps; ++i) bw[i] = *reinterpret_cast<const uint4*>(from + j * kStageRow + 64 * i + 16 * g);
        // Low parts first, while the sum is small: a block's sums then round on the high parts' scale twice, not four times
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[rt] = mfma16x16x32(lo[rt][i], bw[i], acc[rt]);
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) acc[rt] = mfma16x16x32(hi[rt][i], bw[i], acc[rt]);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float4 s = *reinterpret_cast<const float4*>(&scale_s[wave][16 * rt + 4 * g]);
            total[t][rt][0] = fmaf(s.x, acc[rt][0], total[t][rt][0]);
            total[t][rt][1] = fmaf(s.y, acc[rt][1], total[t][rt][1]);
            total[t][rt][2] = fmaf(s.z, acc[rt][2], total[t][rt][2]);
            total[t][rt][3] = fmaf(s.w, acc[rt][3], total[t][rt][3]);
        }
    };
    for (int kb = b_begin + wave; kb < b_end; kb += kWaves) {
        convert();
        load_rows(kb + kWaves);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            uint8_t* to = stage + (t % kStages) * kStageBytes;
#pragma unroll
            for (int li = 0; li < kLoads; ++li)      // built from the elements: a whole-struct copy would keep the array in scratch memory
                *reinterpret_cast<u32x4*>(to + (li * kColsPerLoad + run_col) * kStageRow + 16 * run_lane) = u32x4{b[t][li].x, b[t][li].y, b[t][li].z, b[t][li].w};
            __builtin_amdgcn_wave_barrier();
            issue(kb + kWaves, t);
            multiply(to, t);
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();

    // ---- the waves' sums, and what follows the product
    if (NORM) {
#pragma unroll
        for (int u = 0; u < kRowLoads; ++u) {
            const float sum = m40_sum16(sq[u]);
            if (j == 0) square_s[wave][4 * u + g] = sum;
        }
    }
    float* red = reinterpret_cast<float*>(lds);          // [T][waves][RT * 4][64]: nobody reads the staged weights any more
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((t * kWaves + wave) * RT * 4 + rt * 4 + r) * 64 + lane] = total[t][rt][r];
    __syncthreads();
    if (NORM) {
        if (tid < 16 * RT) {
            float q[kWaves];
#pragma unroll
            for (int k = 0; k < kWaves; ++k) q[k] = square_s[k][tid];
#pragma unroll
            for (int n = kWaves / 2; n >= 1; n /= 2)
#pragma unroll
                for (int k = 0; k < n; ++k) q[k] += q[k + n];
            factor_s[tid] = rsqrtf(q[0] / (float)p.K + p.eps);
        }
        __syncthreads();
    }
    auto sum = [&](int t, int r, int col) {              // element (row r, column col) of tile t
        const float* at = red + ((size_t)t * kWaves * RT * 4 + (r >> 4) * 4 + (r & 3)) * 64 + 16 * ((r >> 2) & 3) + col;
        float s[kWaves];
#pragma unroll
        for (int k = 0; k < kWaves; ++k) s[k] = at[k * RT * 4 * 64];
#pragma unroll
        for (int n = kWaves / 2; n >= 1; n /= 2)
#pragma unroll
            for (int k = 0; k < n; ++k) s[k] += s[k + n];
        return s[0];
    };
    if (MODE == kQkv) {
        if (tid < 256 * RT && e_row < p.rows && q_position < p.max_seq_len && q_seq < p.max_batch) {
            const float f = factor_s[e_row];
            float own = sum(0, e_row, e_j) * f + bias_own;
            const float other = sum(0, e_row, q_partner) * f + bias_other;
            if (q_which != 2) {
                const float2 q_cs = m40_rope_cos_sin_freq(q_position, p.rope_table ? p.rope_table[q_off] : m40_rope_inv_freq(q_off, p.head_dim, p.rope_base), p.rope_scale);
                float r0, r1;
                m40_rope_apply(q_cs, q_second ? other : own, q_second ? own : other, &r0, &r1);
                own = q_second ? r1 : r0;
            }
            if (q_which == 0) {
                p.q_out[(size_t)e_row * p.q_heads * p.head_dim + q_col] = own;
            } else {
                const size_t ept = (size_t)p.kv_heads * p.head_dim;
                uint16_t* dst = (q_which == 1 ? p.k_cache : p.v_cache) + ((size_t)q_seq * p.max_seq_len + q_position) * ept;
                dst[q_col] = m40_f2h(own);
                if (q_which == 1 && q_col == 0) p.seq_map[q_seq] = q_position + 1u;
            }
        }
    } else {
        constexpr int kCols = MODE == kSwiglu ? 8 : 16;
        for (int e = tid; e < T * 16 * RT * kCols; e += kThreads) {
            const int col_in = e % kCols, r = e / kCols % (16 * RT), t = e / (kCols * 16 * RT);
            const int col = kCols * (tile0 + t) + col_in;
            if (r >= p.rows || tile0 + t >= p.tiles || col >= p.N) continue;
            float y = sum(t, r, col_in);
            if (NORM) y *= factor_s[r];
            if (MODE == kSwiglu) {
                const float up = sum(t, r, col_in + 8) * factor_s[r];
                y = y / (1.0f + expf(-y)) * up;
                if (p.packed) {
                    m40_store_packed(p.packed, 16 * RT, p.N, r, col, y);
                    continue;
                }
            }
            float* dst = p.out + (size_t)r * p.N + col;
            if (MODE == kResidual) {
                const float old = T > 1 && p.residual ? p.residual[(size_t)r * p.N + col] : residual_own;
                if (gridDim.y > 1) {
                    // dst holds +0: the half that comes first leaves its sum there (a zero as -0), the other finds it and adds the residual to the
                    // whole product, which rounds on the residual's scale once (adding the halves to it one by one rounds there twice: a residual of
                    // ten times the product, errors of 3.8e-8 instead of 2.8e-8 against 64 bits).  Both see each other past their dies' caches.
                    const uint32_t left = __float_as_uint(y == 0.0f ? -0.0f : y);
                    const uint32_t found = __hip_atomic_exchange(reinterpret_cast<uint32_t*>(dst), left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (found == 0u) continue;
                    y = __uint_as_float(found) + y;
                    __hip_atomic_store(dst, p.residual ? old + y : y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    continue;
                }
                if (p.residual) y = old + y;
            }
            *dst = y;
        }
    }
    if (p.zero)
        for (int i = (int)blockIdx.x * kThreads + tid; i < p.zero_count; i += (int)gridDim.x * kThreads) p.zero[i] = 0.0f;
}

template <int MODE, int RT, int T>
int launch_t(hipStream_t stream, const WideArgs& a, int k_parts) {
    constexpr int staged = kWaves * (wide_stages(T) * kStageBytes + 16 * kRowBytes), sums = T * kWaves * RT * 4 * 64 * 4, bytes = staged > sums ? staged : sums;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(rows_wide_kernel<MODE, RT, T>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (attr != hipSuccess) return -7;
    rows_wide_kernel<MODE, RT, T><<<dim3((a.tiles + T - 1) / T, k_parts), kThreads, bytes, stream>>>(a);
    return hipGetLastError() == hipSuccess ? 0 : -7;
}
// Tiles per workgroup: rounds of workgroups over the CUs times what a workgroup costs, its tiles and about one more for its start.  (Of up to sixteen rows and
// one tile two workgroups fit a CU; they gain less than the start that they repeat.)  All choices measured, K 2048, in the order 1 / 2 / 3 / 4 / 6 tiles, the rule's
// in brackets, us: gate and up of 5632, 16 rows 16.0 / 13.8 / [10.8] / 11.6 / 14.1, 32 rows 27.0 / 21.9 / [13.8] / 15.0 / 18.4; of 11008, 16 rows 28.1 / 20.3 /
// 18.5 / 22.5 / [17.6], 32 rows 52.0 / 32.6 / 25.8 / 28.2 / [21.7]; vocabulary of 32000, 16 rows 39.1 / 30.4 / 30.4 / [30.8] / 35.5, 32 rows 71.8 / 44.4 / 40.6 / [35.3] /
// 42.7; N 4096, 16 rows [8.2] / 9.2 / 10.2 / 11.0 / 13.6.  Of 24 such launches (12 to 32 rows) the rule's is the fastest or within 7 % of it (12 rows, vocabulary of 128256: 114, three tiles 106).
int pick_tiles(int tiles, int num_cus) {
    int best = 1, best_cost = 1 << 30;
    for (const int t : {1, 2, 3, 4, 6}) {
        const int groups = (tiles + t - 1) / t, cost = (groups + num_cus - 1) / num_cus * (t + 1);
        if (cost < best_cost) { best = t; best_cost = cost; }
    }
    return best;
}
template <int MODE, int RT>
int launch_rt(M40llmCudaContext* ctx, hipStream_t stream, const WideArgs& a, int k_parts) {
    const int t = MODE == kQkv || k_parts > 1 ? 1 : pick_tiles(a.tiles, ctx->num_cus);
    if (t == 1) return launch_t<MODE, RT, 1>(stream, a, k_parts);
    if constexpr (MODE != kQkv) {
        if (t == 2) return launch_t<MODE, RT, 2>(stream, a, k_parts);
        if (t == 3) return launch_t<MODE, RT, 3>(stream, a, k_parts);
        if (t == 4) return launch_t<MODE, RT, 4>(stream, a, k_parts);
        return launch_t<MODE, RT, 6>(stream, a, k_parts);
    }
    return -7;
}
template <int MODE>
int launch(M40llmCudaContext* ctx, hipStream_t stream, WideArgs& a, int k_parts = 1) {
    a.blocks = a.K / kShare;
    return a.rows <= 16 ? launch_rt<MODE, 1>(ctx, stream, a, k_parts) : launch_rt<MODE, 2>(ctx, stream, a, k_parts);
}

}  // namespace

namespace {

// Every workgroup reads all rows while others already store their columns and clear their share: what is written must lie apart from the rows
// and from each other.
bool rows_untouched(const WideArgs& a, const float* out, size_t out_cols) {
    const size_t x_bytes = (size_t)a.rows * a.K * 4, out_bytes = (size_t)a.rows * out_cols * 4, zero_bytes = (size_t)a.zero_count * 4;
    return m40_apart(a.x, x_bytes, out, out_bytes) && m40_apart(a.x, x_bytes, a.zero, zero_bytes) && m40_apart(out, out_bytes, a.zero, zero_bytes);
}

}  // namespace

// 9 .. 32 rows: fewer rows have faster kernels (rows_mfma.hip, rows_gemv.hip); the operands 16-byte aligned, K whole steps of 256.
bool m40_rows_wide_supported(int rows, int K) { return rows >= 1 && rows <= 32 && K >= 256 && K % 256 == 0; }

int m40_rows_wide_qkv(M40llmCudaContext* ctx, hipStream_t stream, const M40llmKVCache* kv, const uint32_t* ids_dev, const uint32_t* lens_dev,
                      uint32_t rows, const float* x, const void* norm_w, uint32_t norm_dtype, float eps, const uint16_t* wq, const uint16_t* wk,
                      const uint16_t* wv, const float* bq, const float* bk, const float* bv, uint32_t d_model, uint32_t q_heads, float rope_base,
                      float rope_scale, uint32_t rope_layout, float* q_out, float* zero, int zero_count) {
    if (!m40_rows_wide_supported((int)rows, (int)d_model) || kv->head_dim % 16 != 0) return -6;
    if (!m40_aligned16(x) || !m40_aligned16(norm_w) || !m40_aligned16(wq) || !m40_aligned16(wk) || !m40_aligned16(wv)) return -6;
    WideArgs a{};
    a.x = x; a.norm_w = norm_w; a.norm_dtype = norm_dtype; a.eps = eps; a.W0 = wq; a.W1 = wk; a.W2 = wv;
    a.bq = bq; a.bk = bk; a.bv = bv; a.q_out = q_out; a.k_cache = kv->d_k; a.v_cache = kv->d_v; a.seq_map = kv->d_seq_map;
    a.ids_dev = ids_dev; a.lens_dev = lens_dev;
    a.rope_table = m40_rope_inv_freq_table(ctx, 1, stream, kv->head_dim, rope_base);
    a.max_seq_len = kv->max_seq_len; a.max_batch = kv->max_batch_size; a.q_heads = q_heads; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.rope_layout = rope_layout; a.rope_base = rope_base; a.rope_scale = rope_scale;
    a.rows = (int)rows; a.K = (int)d_model; a.N = (int)((q_heads + 2u * kv->num_heads) * kv->head_dim);
    a.tiles = a.N / 16; a.zero = zero; a.zero_count = zero_count;
    if (!rows_untouched(a, q_out, (size_t)q_heads * kv->head_dim)) return -6;
    return launch<kQkv>(ctx, stream, a);
}

int m40_rows_wide_swiglu(M40llmCudaContext* ctx, hipStream_t stream, const float* x, const void* norm_w, uint32_t norm_dtype, float eps,
                         const uint16_t* wgate, const uint16_t* wup, float* out, uint8_t* packed, int rows, int ffn, int K, float* zero, int zero_count) {
    if (!m40_rows_wide_supported(rows, K) || ffn <= 0 || (packed && (rows <= 8 || ffn % 8 != 0))) return -6;
    if (!m40_aligned16(x) || !m40_aligned16(norm_w) || !m40_aligned16(wgate) || !m40_aligned16(wup)) return -6;
    WideArgs a{};
    a.x = x; a.norm_w = norm_w; a.norm_dtype = norm_dtype; a.eps = eps; a.W0 = wgate; a.W1 = wup; a.out = out; a.packed = packed;
    a.rows = rows; a.N = ffn; a.K = K; a.tiles = (ffn + 7) / 8; a.zero = zero; a.zero_count = zero_count;
    if (!packed && !rows_untouched(a, out, ffn)) return -6;
    return launch<kSwiglu>(ctx, stream, a);
}

int m40_rows_wide_norm(M40llmCudaContext* ctx, hipStream_t stream, const float* x, const void* norm_w, uint32_t norm_dtype, float eps,
                       const uint16_t* W, float* out, int rows, int N, int K) {
    if (!m40_rows_wide_supported(rows, K) || N <= 0) return -6;
    if (!m40_aligned16(x) || !m40_aligned16(norm_w) || !m40_aligned16(W)) return -6;
    WideArgs a{};
    a.x = x; a.norm_w = norm_w; a.norm_dtype = norm_dtype; a.eps = eps; a.W0 = W; a.out = out; a.rows = rows; a.N = N; a.K = K; a.tiles = (N + 15) / 16;
    if (!rows_untouched(a, out, N)) return -6;
    return launch<kNorm>(ctx, stream, a);
}

// onto_zero: out holds zeros (+0), so that two halves of K can meet in it where one tile a workgroup would leave half of the CUs idle; a
// residual that is out itself is read before each element is stored, in one part.
int m40_rows_wide_residual(M40llmCudaContext* ctx, hipStream_t stream, const float* x, const uint16_t* W, const float* residual, float* out, int rows,
                           int N, int K, bool onto_zero) {
    if (!m40_rows_wide_supported(rows, K) || N <= 0) return -6;
    if (!m40_aligned16(x) || !m40_aligned16(W)) return -6;
    WideArgs a{};
    a.x = x; a.W0 = W; a.residual = residual; a.out = out; a.rows = rows; a.N = N; a.K = K; a.tiles = (N + 15) / 16;
    const size_t out_bytes = (size_t)rows * N * 4;
    if (!rows_untouched(a, out, N) || (residual != out && !m40_apart(residual, out_bytes, out, out_bytes))) return -6;
    return launch<kResidual>(ctx, stream, a, onto_zero && residual != out && K >= 1024 && 2 * a.tiles <= ctx->num_cus ? 2 : 1);
}

extern "C" {

int m40llm_ext_batched_wide_norm_qkv_rope_append_async(
    M40llmCudaContext* ctx, M40llmKVCache* kv, const uint32_t* seq_ids_dev, const uint32_t* seq_lens_dev, uint32_t rows, const void* d_x_f32,
    const void* d_norm_w, uint32_t norm_weight_dtype, float eps, const void* d_wq_f16, const void* d_wk_f16, const void* d_wv_f16,
    const void* d_bq_f32, const void* d_bk_f32, const void* d_bv_f32, uint32_t d_model, uint32_t q_heads, float freq_base, float freq_scale,
    uint32_t rope_layout, void* d_q_out_f32, void* d_clear_f32, uint32_t clear_floats) {
    if (!ctx || !kv || !seq_ids_dev || !seq_lens_dev || !d_x_f32 || !d_norm_w || !d_wq_f16 || !d_wk_f16 || !d_wv_f16 || !d_q_out_f32) return -1;
    if (kv->compressed || !kv->d_k || !kv->d_v || clear_floats > (1u << 30)) return -2;
    if (norm_weight_dtype > 1) return -4;
    if (kv->head_dim == 0 || kv->head_dim % 16 != 0 || kv->num_heads == 0 || q_heads == 0) return -3;
    (void)hipGetLastError();
    return m40_rows_wide_qkv(ctx, ctx->decode_stream, kv, seq_ids_dev, seq_lens_dev, rows, static_cast<const float*>(d_x_f32), d_norm_w, norm_weight_dtype,
                             eps, static_cast<const uint16_t*>(d_wq_f16), static_cast<const uint16_t*>(d_wk_f16), static_cast<const uint16_t*>(d_wv_f16),
                             static_cast<const float*>(d_bq_f32), static_cast<const float*>(d_bk_f32), static_cast<const float*>(d_bv_f32), d_model,
                             q_heads, freq_base, freq_scale, rope_layout, static_cast<float*>(d_q_out_f32),
                             clear_floats ? static_cast<float*>(d_clear_f32) : nullptr, (int)clear_floats);
}

int m40llm_ext_batched_wide_norm_gate_up_swiglu_async(M40llmCudaContext* ctx, const void* d_x_f32, const void* d_norm_w, uint32_t norm_weight_dtype,
                                                      float eps, const void* d_wgate_f16, const void* d_wup_f16, void* d_hid_f32, uint32_t rows, int ffn,
                                                      int d_model, void* d_clear_f32, uint32_t clear_floats) {
    if (!ctx || !d_x_f32 || !d_norm_w || !d_wgate_f16 || !d_wup_f16 || !d_hid_f32) return -1;
    if (ffn <= 0 || d_model <= 0 || clear_floats > (1u << 30)) return -2;
    if (norm_weight_dtype > 1) return -4;
    (void)hipGetLastError();
    return m40_rows_wide_swiglu(ctx, ctx->decode_stream, static_cast<const float*>(d_x_f32), d_norm_w, norm_weight_dtype, eps,
                                static_cast<const uint16_t*>(d_wgate_f16), static_cast<const uint16_t*>(d_wup_f16), static_cast<float*>(d_hid_f32), nullptr,
                                (int)rows, ffn, d_model, clear_floats ? static_cast<float*>(d_clear_f32) : nullptr, (int)clear_floats);
}

int m40llm_ext_batched_wide_gemm_residual_onto_zero_async(M40llmCudaContext* ctx, const void* d_a_f32, const void* d_w_f16, const void* d_residual_f32,
                                                          void* d_out_f32, uint32_t rows, int N, int K) {
    if (!ctx || !d_a_f32 || !d_w_f16 || !d_out_f32) return -1;
    if (N <= 0 || K <= 0) return -2;
    (void)hipGetLastError();
    return m40_rows_wide_residual(ctx, ctx->decode_stream, static_cast<const float*>(d_a_f32), static_cast<const uint16_t*>(d_w_f16),
                                  static_cast<const float*>(d_residual_f32), static_cast<float*>(d_out_f32), (int)rows, N, K, true);
}

int m40llm_ext_batched_wide_norm_gemm_async(M40llmCudaContext* ctx, const void* d_x_f32, const void* d_norm_w, uint32_t norm_weight_dtype, float eps,
                                            const void* d_w_f16, void* d_out_f32, uint32_t rows, int N, int K) {
    if (!ctx || !d_x_f32 || !d_norm_w || !d_w_f16 || !d_out_f32) return -1;
    if (N <= 0 || K <= 0) return -2;
    if (norm_weight_dtype > 1) return -4;
    (void)hipGetLastError();
    return m40_rows_wide_norm(ctx, ctx->decode_stream, static_cast<const float*>(d_x_f32), d_norm_w, norm_weight_dtype, eps,
                              static_cast<const uint16_t*>(d_w_f16), static_cast<float*>(d_out_f32), (int)rows, N, K);
}

}  // extern "C"
