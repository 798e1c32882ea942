// Row-batched projections of a decode step for 9 to 32 activation rows (f32) against f16 GGUF weights [N][K], one launch per
// projection on v_mfma_f32_16x16x32_f16.
//
// rows_mfma.hip keeps eight whole rows as operand fragments in LDS, which more rows do not fit; skinny_mfma.hip converts every step
// of the rows once per 64 columns and adds its K slices in a second launch, and reads the weights once per sixteen rows.  Here a
// workgroup of eight waves owns T column tiles and walks K in chunks of 512: the chunk's rows become f16 hi + lo fragments
// (32 or 64 KB, two buffers: the next chunk is converted while this one is multiplied; one power-of-two scale per row and chunk,
// RMSNorm weights folded in, the RMS factor applied to the sums), the eight waves take 64 k of the chunk each, and their sums meet in
// LDS once, after the last chunk, pair by pair.  So the weights are read once for all rows, every result is written once, nothing is
// left for a second launch and no result depends on timing.
//
// Bound: the weight stream, and at one or two tiles a workgroup the chain rows -> fragments -> products of each chunk.  A row costs
// every workgroup as many bytes as two columns of weights; they come from L2 and are requested a chunk ahead.  One workgroup is
// resident per CU (82 or 148 KB of LDS), which T is chosen for.  Weight loads are whole 128-byte lines
// (eight lanes a column) and pass through a wave-private LDS tile into operand order, as in rows_mfma.hip; about 64 KB of them per CU
// are in flight (one, two or four chunks ahead).  A product of few columns onto zeros is cut into two halves of K, which meet
// in the result element by element: two terms, the same bits in either order.
#include "common.hpp"

#include <type_traits>

namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kChunk = 512;                             // k per chunk
constexpr int kShare = kChunk / kWaves;                 // k per wave and chunk
constexpr int kSteps = kShare / 32;                     // matrix instructions deep
constexpr int kRunLanes = kShare * 2 / 16;              // lanes that cover a column's share with 16 bytes each
constexpr int kColsPerLoad = 64 / kRunLanes;
constexpr int kLoads = 16 / kColsPerLoad;
constexpr int kStageRow = kShare * 2 + 16;              // LDS bytes per column: +16 spreads the columns over the banks
constexpr int kStageBytes = 16 * kStageRow;             // per wave
constexpr int kPlane = kChunk / 32 * 64;                // 16-byte entries of one 16-row operand plane of a chunk

enum Mode { kResidual = 0, kSwiglu = 1, kQkv = 2, kNorm = 3 };

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ m40_float4 mfma16x16x32(const uint4& a, const uint4& b, m40_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(m40_half8, a), __builtin_bit_cast(m40_half8, b), c, 0, 0, 0);
}

// Where entry e of an operand plane ([k-step][lane]) lies: the row (low four bits) xor-ed with the four bits above, so that the lanes of
// the conversion, which hold one row at consecutive eights of k, spread over the banks.
__device__ __forceinline__ int frag_slot(int e) { return e ^ ((e >> 4) & 15); }

struct WideArgs {
    const float* x;               // [rows][K]
    const void* norm_w;           // RMSNorm weights (all modes but kResidual)
    uint32_t norm_dtype;          // 0 f16, 1 f32
    float eps;
    const uint16_t *W0, *W1, *W2; // kSwiglu: gate, up; kQkv: q, k, v
    float* out;                   // [rows][N]
    const float* residual;        // kResidual: added to the product, or null
    int rows, N, K, tiles, chunks;
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
    constexpr int kRowLanes = 32 / RT;                  // lanes that convert one row
    constexpr int kEights = kChunk / 8 / kRowLanes;     // eights of k per lane and chunk
    constexpr int kAhead = T >= 3 ? 1 : 4 / T;          // chunks between a weight request and its use
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint4* frag = reinterpret_cast<uint4*>(lds);        // [2 buffers][RT][hi, lo][kPlane]
    uint8_t* stage = lds + 2 * RT * 2 * kPlane * 16 + (threadIdx.x >> 6) * kStageBytes;
    __shared__ __attribute__((aligned(16))) float scale_s[2][16 * RT];      // undoes the chunk's scaling of each row
    __shared__ float factor_s[16 * RT];                                     // RMSNorm factor of each row

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int c_begin = p.chunks * (int)blockIdx.y / (int)gridDim.y, c_end = p.chunks * ((int)blockIdx.y + 1) / (int)gridDim.y;
    const int tile0 = (int)blockIdx.x * T;

    // ---- rows of a chunk, requested ahead: 8-element pieces l, l + kRowLanes, ... of the thread's row
    const int row = tid / kRowLanes, l = tid % kRowLanes;
    const bool live = row < p.rows;
    const float* xr = p.x + (size_t)(live ? row : 0) * p.K;
    const int eights = p.K / 8;
    float4 v[2 * kEights];
    uint4 w[NORM ? 2 * kEights : 1];
    const bool norm16 = NORM && p.norm_dtype == 0u;
    const int w_mul = norm16 ? 1 : 2, w_second = norm16 ? 0 : 1;
    auto load_rows = [&](int c) {
#pragma unroll
        for (int i = 0; i < kEights; ++i) {
            int at = c * (kChunk / 8) + l + kRowLanes * i;
            at = at < eights ? at : 0;
            v[2 * i] = reinterpret_cast<const float4*>(xr)[2 * at];
            v[2 * i + 1] = reinterpret_cast<const float4*>(xr)[2 * at + 1];
            if (NORM) {      // f16 weights are 16 bytes an eight, requested twice: no load under a branch
                w[2 * i] = static_cast<const uint4*>(p.norm_w)[w_mul * at];
                w[2 * i + 1] = static_cast<const uint4*>(p.norm_w)[w_mul * at + w_second];
            }
        }
    };
    load_rows(c_begin);
    __builtin_amdgcn_sched_barrier(0);

    // ---- weights: instruction li of a wave reads its 64 k of columns 8 li .. 8 li + 7 of a tile
    const int run_lane = lane % kRunLanes, run_col = lane / kRunLanes;
    const uint16_t* col_ptr[T][kLoads];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int tile = tile0 + t < p.tiles ? tile0 + t : p.tiles - 1;
#pragma unroll
        for (int li = 0; li < kLoads; ++li) {
            const int i = li * kColsPerLoad + run_col;
            const uint16_t* W = p.W0;
            int col;
            if (MODE == kSwiglu) {
                col = 8 * tile + (i & 7);
                if (li * kColsPerLoad & 8) W = p.W1;
                col = col < p.N ? col : p.N - 1;
            } else if (MODE == kQkv) {
                const QkvTile q = qkv_tile(p, tile);
                col = qkv_col(p, q, i);
                W = q.which == 0 ? p.W0 : (q.which == 1 ? p.W1 : p.W2);
            } else {
                col = 16 * tile + i;
                col = col < p.N ? col : p.N - 1;
            }
            col_ptr[t][li] = W + (size_t)col * p.K;
        }
    }
    uint4 b[kAhead * T][kLoads];
    auto issue = [&](uint4 (&dst)[kLoads], int c, int t) {
        const int k = c * kChunk + wave * kShare + 8 * run_lane;
        const int at = c < c_end && k < p.K ? k : 0;       // past the end: a valid address, the value is not used
#pragma unroll
        for (int li = 0; li < kLoads; ++li) dst[li] = *reinterpret_cast<const uint4*>(col_ptr[t][li] + at);
    };
#pragma unroll
    for (int u = 0; u < kAhead * T; ++u) issue(b[u], c_begin + u / T, u % T);
    __builtin_amdgcn_sched_barrier(0);

    // what a thread's element needs besides the product (one tile a workgroup), asked for early
    const int e_j = tid & 15, e_row = (tid >> 4) & (16 * RT - 1);
    int q_which = 0, q_col = 0, q_partner = 0;
    bool q_second = false;
    uint32_t q_position = 0, q_seq = 0;
    float bias_own = 0.0f, bias_other = 0.0f;
    float2 q_cs = make_float2(1.0f, 0.0f);
    float residual_own = 0.0f;
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
        const uint32_t off = t.split ? (uint32_t)(8 * t.tt + (e_j & 7)) : (uint32_t)((16 * t.tt + e_j) >> 1);
        const float* bias = t.which == 0 ? p.bq : (t.which == 1 ? p.bk : p.bv);
        q_position = p.lens_dev[e_rowc];
        q_seq = p.ids_dev[e_rowc];
        bias_own = bias ? bias[q_col] : 0.0f;
        bias_other = bias ? bias[qkv_col(p, t, q_partner)] : 0.0f;
        const float freq = p.rope_table ? p.rope_table[off] : m40_rope_inv_freq(off, p.head_dim, p.rope_base);
        if (t.which != 2) q_cs = m40_rope_cos_sin_freq(q_position, freq, p.rope_scale);
    }

    // ---- rows of chunk c -> f16 hi + lo fragments of buffer c & 1
    float sq = 0.0f;
    auto convert = [&](int c) {
        float x[kEights][8];
        float mx = 0.0f;
#pragma unroll
        for (int i = 0; i < kEights; ++i) {
            const float4 a0 = v[2 * i], a1 = v[2 * i + 1];
            const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
            const bool in = live && c * (kChunk / 8) + l + kRowLanes * i < eights;
            float f[8] = {1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f};
            if (NORM) {
                if (norm16) {
                    m40_unpack8(w[2 * i], f);
                } else {
                    const uint4 f0 = w[2 * i], f1 = w[2 * i + 1];
                    const uint32_t u[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(u[e]);
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float y = in ? a[e] : 0.0f;
                if (NORM) sq = fmaf(y, y, sq);
                x[i][e] = NORM ? (in ? y * f[e] : 0.0f) : y;
                mx = fmaxf(mx, fabsf(x[i][e]));
            }
        }
        mx = m40_max16(mx);
        if (kRowLanes == 32) mx = m40_max_xor16(mx);
        float scale = 1.0f, inv_scale = 1.0f;
        if (mx > 0.0f && mx < INFINITY) {
            int ex;
            (void)frexpf(mx, &ex);        // mx = f * 2^ex, f in [0.5, 1)
            ex -= 11;                     // scaled maximum in [2^10, 2^11)
            ex = ex < -100 ? -100 : (ex > 100 ? 100 : ex);
            scale = ldexpf(1.0f, ex);
            inv_scale = ldexpf(1.0f, -ex);
        }
        uint4* plane = frag + (size_t)(((c & 1) * RT + (row >> 4)) * 2) * kPlane;
#pragma unroll
        for (int i = 0; i < kEights; ++i) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const f32x2 s2 = {x[i][e] * inv_scale, x[i][e + 1] * inv_scale};
                const f16x2 h2 = __builtin_convertvector(s2, f16x2);
                const f16x2 l2 = __builtin_convertvector(s2 - __builtin_convertvector(h2, f32x2), f16x2);
                hi[e / 2] = __builtin_bit_cast(uint32_t, h2);
                lo[e / 2] = __builtin_bit_cast(uint32_t, l2);
            }
            const int eight = l + kRowLanes * i;
            const int entry = frag_slot((eight >> 2) * 64 + (eight & 3) * 16 + (row & 15));
            plane[entry] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            plane[kPlane + entry] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
        }
        if (l == 0) scale_s[c & 1][row] = scale;
    };
    convert(c_begin);
    __syncthreads();

    m40_float4 total[T][RT];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) total[t][rt] = {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int c, int t) {
        const uint4* planes = frag + (size_t)((c & 1) * RT * 2) * kPlane;
        m40_float4 acc[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt] = {0.f, 0.f, 0.f, 0.f};
        uint4 bw[kSteps];
#pragma unroll
        for (int i = 0; i < kSteps; ++i) bw[i] = *reinterpret_cast<const uint4*>(stage + j * kStageRow + 64 * i + 16 * g);
        // Low parts first, while the sum is small: a chunk's sums then round on the high parts' scale twice, not four times (K 2048 with the norm,
        // against 64 bits: 1.30e-7 -> 1.17e-7, and 1.12e-7 with the waves' sums added pair by pair instead of one after the other)
#pragma unroll
        for (int part = 1; part >= 0; --part)
#pragma unroll
            for (int i = 0; i < kSteps; ++i) {
                const int e = frag_slot((kSteps * wave + i) * 64 + lane);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt] = mfma16x16x32(planes[(2 * rt + part) * kPlane + e], bw[i], acc[rt]);
            }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const float4 s = *reinterpret_cast<const float4*>(&scale_s[c & 1][16 * rt + 4 * g]);
            total[t][rt][0] = fmaf(s.x, acc[rt][0], total[t][rt][0]);
            total[t][rt][1] = fmaf(s.y, acc[rt][1], total[t][rt][1]);
            total[t][rt][2] = fmaf(s.z, acc[rt][2], total[t][rt][2]);
            total[t][rt][3] = fmaf(s.w, acc[rt][3], total[t][rt][3]);
        }
    };
    for (int c0 = c_begin; c0 < c_end; c0 += kAhead) {
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
            const int c = c0 + a;
            if (c >= c_end) break;
            load_rows(c + 1 < c_end ? c + 1 : c);
            const bool mine = c * kChunk + wave * kShare < p.K;       // the last chunk may end in its middle
#pragma unroll
            for (int t = 0; t < T; ++t) {
                uint4 (&set)[kLoads] = b[a * T + t];
#pragma unroll
                for (int li = 0; li < kLoads; ++li)      // built from the elements: a whole-struct copy would keep the array in scratch memory
                    *reinterpret_cast<u32x4*>(stage + (li * kColsPerLoad + run_col) * kStageRow + 16 * run_lane) =
                        u32x4{set[li].x, set[li].y, set[li].z, set[li].w};
                __builtin_amdgcn_wave_barrier();
                issue(set, c + kAhead, t);
                if (mine) multiply(c, t);
                __builtin_amdgcn_wave_barrier();
            }
            if (c + 1 < c_end) convert(c + 1);
            __syncthreads();
        }
    }

    // ---- the waves' sums, and what follows the product
    if (NORM) {
        sq = m40_sum16(sq);
        if (kRowLanes == 32) sq = m40_add_xor16(sq);
        if (l == 0) factor_s[row] = rsqrtf(sq / (float)p.K + p.eps);
    }
    float* red = reinterpret_cast<float*>(lds);          // [T][waves][RT * 4][64]: nobody reads the fragments any more
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[((t * kWaves + wave) * RT * 4 + rt * 4 + r) * 64 + lane] = total[t][rt][r];
    __syncthreads();
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
    constexpr int bytes = 2 * RT * 2 * kPlane * 16 + kWaves * kStageBytes;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(rows_wide_kernel<MODE, RT, T>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (attr != hipSuccess) return -7;
    rows_wide_kernel<MODE, RT, T><<<dim3((a.tiles + T - 1) / T, k_parts), kThreads, bytes, stream>>>(a);
    return hipGetLastError() == hipSuccess ? 0 : -7;
}
// Tiles per workgroup: rounds of workgroups over the CUs (one is resident per CU) times what a workgroup costs, its tiles and about one
// more for its start.
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
    a.chunks = (a.K + kChunk - 1) / kChunk;
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
                         const uint16_t* wgate, const uint16_t* wup, float* out, int rows, int ffn, int K, float* zero, int zero_count) {
    if (!m40_rows_wide_supported(rows, K) || ffn <= 0) return -6;
    if (!m40_aligned16(x) || !m40_aligned16(norm_w) || !m40_aligned16(wgate) || !m40_aligned16(wup)) return -6;
    WideArgs a{};
    a.x = x; a.norm_w = norm_w; a.norm_dtype = norm_dtype; a.eps = eps; a.W0 = wgate; a.W1 = wup; a.out = out;
    a.rows = rows; a.N = ffn; a.K = K; a.tiles = (ffn + 7) / 8; a.zero = zero; a.zero_count = zero_count;
    if (!rows_untouched(a, out, ffn)) return -6;
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
    return launch<kResidual>(ctx, stream, a, onto_zero && residual != out && K >= 2 * kChunk && 2 * a.tiles <= ctx->num_cus ? 2 : 1);
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
                                static_cast<const uint16_t*>(d_wgate_f16), static_cast<const uint16_t*>(d_wup_f16), static_cast<float*>(d_hid_f32),
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
