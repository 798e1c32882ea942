// Projection of up to 32 activation rows that the launch before left as matrix operands (packed_rows.hpp) against f16 weights [N][K], a residual added: the O
// and the down projection of a batched decode step.
//
// With f32 rows every workgroup turns all of them into operands again, and asks for them in pieces that lie K apart.  Here an operand is a contiguous KiB a wave
// reads and multiplies: what is left of the rows' cost is their bytes, which every workgroup of sixteen columns reads once (8 rows as many as its weights,
// 32 rows four times as many: the bound of 32 rows, from L2).  A wave's block is 128 k of sixteen columns, every WAVES-th, its weights as runs of 256 bytes
// a column through an LDS tile of the wave's own.  Nothing is asked for ahead of the block in work: with as many waves as a CU takes, the others' requests are
// what is on its way, and a second block a wave is slower (8 rows, K 11008: 13.7 us against 11.9; 32 rows 18.4 against 16.9).  The weights pass the
// caches by (non-temporal): they are read once, and the rows stay (K 11008, 8 rows 12.7 -> 11.9 us, 32 rows 18.0 -> 16.9; no difference at K 2048 and 5632).
//
// Two halves of K where one tile a workgroup would leave half of the CUs idle, onto a result that holds zeros, as in rows_wide_mfma.hip: no second launch, and no
// result depends on timing.  Measured in a replayed graph with cold weights, N 2048, f32 rows before / packed now, us: K 2048, 8 rows 5.4 / 4.2, 16 rows
// 5.1 / 4.5, 32 rows 6.5 / 5.3; K 5632 7.5 / 6.9, 8.5 / 8.1, 11.6 / 9.9; K 11008, 8 rows 13.5 / 11.9.  (Looking for units far below their block's largest, below,
// is part of that since: 0.1 us a launch at 8 rows, 0.05 at 16 and 32.)
#include "packed_rows.hpp"

namespace {

constexpr int kBlock = 128, kSteps = kBlock / 32;        // k of a wave's block, matrix instructions deep
constexpr int kRunLanes = kBlock * 2 / 16;              // lanes that cover a column's block with 16 bytes each
constexpr int kCols = 64 / kRunLanes, kLoads = 16 / kCols;
constexpr float kFar = 256.0f;                           // a unit that far below the largest of its row and block is multiplied on its own
constexpr int kStageRow = kBlock * 2 + 16;              // LDS bytes per column: +16 spreads the columns over the banks

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ m40_float4 mfma16x16x32(const f16x8& a, const uint4& b, m40_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(m40_half8, a), __builtin_bit_cast(m40_half8, b), c, 0, 0, 0);
}

// PAD: rows, padded.  grid (ceil(N / 16), parts of K)
template <int PAD, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void packed_rows_kernel(const uint8_t* packed, const uint16_t* W, const float* residual, float* out, int rows, int N, int K) {
    constexpr int RT = PAD > 8 ? PAD / 16 : 1, PARTS = PAD > 8 ? 2 : 1;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int blocks = K / kBlock, b_begin = blocks * (int)blockIdx.y / (int)gridDim.y, b_end = blocks * ((int)blockIdx.y + 1) / (int)gridDim.y;
    const int n0 = 16 * (int)blockIdx.x;
    uint8_t* stage = lds + wave * (16 * kStageRow);
    const float* scales = reinterpret_cast<const float*>(packed + (size_t)PAD * K * 4);
    const int run_lane = lane % kRunLanes, run_col = lane / kRunLanes;
    uint32_t w_at[kLoads];
#pragma unroll
    for (int li = 0; li < kLoads; ++li) {
        const int c = li * kCols + run_col, left = N - 1 - n0;
        w_at[li] = (uint32_t)(c < left ? c : left) * (uint32_t)K + 8u * run_lane;
    }
    const uint16_t* w_tile = W + (size_t)n0 * K;

    m40_float4 total[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) total[rt] = {0.f, 0.f, 0.f, 0.f};
    const auto scale_at = [&](int kb, int i, int rt) { return scales[(size_t)(kb * 4 * kSteps + 4 * i + g) * PAD + 16 * rt + (PAD > 8 ? j : j & 7)]; };
    const auto largest = [&](const float (&s)[kSteps]) {         // of a row's sixteen units of the block
        const float most = m40_max_xor32(m40_max_xor16(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
        return most > 0.0f ? most : 1.0f;
    };
    // (rows that are not there hold anything)
    const auto is_far = [&](float s, float most, int rt) { return s > 0.0f && s * kFar < most && 16 * rt + (PAD > 8 ? j : j & 7) < rows; };
    bool left_out = false;
    for (int kb = b_begin + wave; kb < b_end; kb += WAVES) {
        f16x8 a[RT][PARTS][kSteps];
        float s[RT][kSteps];
        const uint8_t* from = packed + (size_t)kb * (kSteps * PAD * 128) + 16 * lane;
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                for (int h = 0; h < PARTS; ++h) a[rt][h][i] = *reinterpret_cast<const f16x8*>(from + ((i * RT + rt) * PARTS + h) * 1024);
                s[rt][i] = scale_at(kb, i, rt);
            }
        __builtin_amdgcn_sched_barrier(0);      // the rows (cache hits) ahead of the weights: loads return in issue order
        u32x4 b[kLoads];
#pragma unroll
        for (int li = 0; li < kLoads; ++li) b[li] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w_tile + (size_t)kb * kBlock + w_at[li]));
        __builtin_amdgcn_sched_barrier(0);
        // One scale for a row's sixteen units of the block, the largest: the others' parts are multiplied by the power of two between, exactly, or off by at most 2^-25 where the
        // largest value is 2^14 and more.  Of a unit that lies further below, beside an outlier, that would take bits which count once the outlier's weights are small: it is left
        // out here and added behind the loop.
        float top[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            top[rt] = largest(s[rt]);
            const float inv = __uint_as_float(0x7f000000u - __float_as_uint(top[rt]));
#pragma unroll
            for (int i = 0; i < kSteps; ++i) {
                const bool far = is_far(s[rt][i], top[rt], rt);
                left_out = left_out || far;
                const _Float16 f = static_cast<_Float16>(far ? 0.0f : s[rt][i] > 0.0f ? s[rt][i] * inv : 1.0f);
#pragma unroll
                for (int h = 0; h < PARTS; ++h) a[rt][h][i] *= f;
            }
        }
#pragma unroll
        for (int li = 0; li < kLoads; ++li) *reinterpret_cast<u32x4*>(stage + (li * kCols + run_col) * kStageRow + 16 * run_lane) = b[li];
        __builtin_amdgcn_wave_barrier();
        uint4 bw[kSteps];
#pragma unroll
        for (int i = 0; i < kSteps; ++i) bw[i] = *reinterpret_cast<const uint4*>(stage + j * kStageRow + 64 * i + 16 * g);
        __builtin_amdgcn_wave_barrier();
        // sums of 64 k, low parts first, while the sum is small
        m40_float4 acc[RT][2];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt][0] = acc[rt][1] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = PARTS - 1; h >= 0; --h)
#pragma unroll
            for (int i = 0; i < kSteps; ++i)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt][i / 2] = mfma16x16x32(a[rt][h][i], bw[i], acc[rt][i / 2]);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float scale = __shfl(top[rt], PAD > 8 ? 4 * g + r : 4 * (g & 1) + r, 64);
                total[rt][r] = fmaf(scale, acc[rt][1][r], fmaf(scale, acc[rt][0][r], total[rt][r]));
            }
    }
    // What was left out: the units of each lane group on their own, the others' parts and weights zero.
    if (__builtin_expect(__ballot(left_out) != 0, 0)) {
        for (int kb = b_begin + wave; kb < b_end; kb += WAVES) {
            float far[RT][kSteps];               // the scale of a unit that was left out, or 0
            bool any = false;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                float s[kSteps];
#pragma unroll
                for (int i = 0; i < kSteps; ++i) s[i] = scale_at(kb, i, rt);
                const float most = largest(s);
#pragma unroll
                for (int i = 0; i < kSteps; ++i) {
                    far[rt][i] = is_far(s[i], most, rt) ? s[i] : 0.0f;
                    any = any || far[rt][i] > 0.0f;
                }
            }
            if (__ballot(any) == 0) continue;
            const uint16_t* w_at_j = w_tile + (size_t)(n0 + j < N ? j : N - 1 - n0) * K + (size_t)kb * kBlock + 8 * g;
            const uint8_t* from = packed + (size_t)kb * (kSteps * PAD * 128) + 16 * lane;
#pragma unroll
            for (int i = 0; i < kSteps; ++i) {
                const uint4 w = *reinterpret_cast<const uint4*>(w_at_j + 32 * i), none = make_uint4(0, 0, 0, 0);
#pragma unroll 1
                for (int u = 0; u < 4; ++u) {
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) {
                        m40_float4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int h = PARTS - 1; h >= 0; --h) {
                            const uint4 part = *reinterpret_cast<const uint4*>(from + ((i * RT + rt) * PARTS + h) * 1024);
                            acc = mfma16x16x32(__builtin_bit_cast(f16x8, g == u ? part : none), g == u ? w : none, acc);
                        }
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float scale = __shfl(far[rt][i], 16 * u + (PAD > 8 ? 4 * g + r : 4 * (g & 1) + r), 64);
                            if (scale > 0.0f) total[rt][r] = fmaf(scale, acc[r], total[rt][r]);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);          // [waves][RT * 4][64]: nobody reads the staged weights any more
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[((wave * RT + rt) * 4 + r) * 64 + lane] = PAD > 8 ? total[rt][r] : m40_add_xor32(total[rt][r]);      // 8 rows: hi + lo
    __syncthreads();
    for (int e = tid; e < 16 * PAD; e += 64 * WAVES) {
        const int c = e & 15, r = e >> 4, col = n0 + c;
        if (r >= rows || col >= N) continue;
        const float* at = red + ((r >> 4) * 4 + (r & 3)) * 64 + 16 * ((r >> 2) & 3) + c;
        float y[WAVES];
#pragma unroll
        for (int k = 0; k < WAVES; ++k) y[k] = at[k * RT * 4 * 64];
#pragma unroll
        for (int n = WAVES / 2; n >= 1; n /= 2)
#pragma unroll
            for (int k = 0; k < n; ++k) y[k] += y[k + n];
        float* dst = out + (size_t)r * N + col;
        const float old = residual ? residual[(size_t)r * N + col] : 0.0f;
        if (gridDim.y > 1) {
            // dst holds +0: the half that comes first leaves its sum there (a zero as -0), the other finds it and adds the residual to the whole product; both
            // see each other past their dies' caches
            const uint32_t left = __float_as_uint(y[0] == 0.0f ? -0.0f : y[0]);
            const uint32_t found = __hip_atomic_exchange(reinterpret_cast<uint32_t*>(dst), left, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (found == 0u) continue;
            const float sum = __uint_as_float(found) + y[0];
            __hip_atomic_store(dst, residual ? old + sum : sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            continue;
        }
        *dst = residual ? old + y[0] : y[0];
    }
}

template <int PAD, int WAVES>
int launch(hipStream_t stream, const uint8_t* packed, const uint16_t* W, const float* residual, float* out, int rows, int N, int K, int parts) {
    constexpr int RT = PAD > 8 ? PAD / 16 : 1, staged = WAVES * 16 * kStageRow, sums = WAVES * RT * 4 * 64 * 4, bytes = staged > sums ? staged : sums;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(packed_rows_kernel<PAD, WAVES>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (attr != hipSuccess) return -7;
    packed_rows_kernel<PAD, WAVES><<<dim3((N + 15) / 16, parts), 64 * WAVES, bytes, stream>>>(packed, W, residual, out, rows, N, K);
    return hipGetLastError() == hipSuccess ? 0 : -7;
}
// Sixteen waves where a workgroup has more than sixteen blocks (K 5632 in halves, 32 rows: 9.9 us, eight waves 10.6; K 11008 16.9 and 17.7), else eight (K 2048 in
// halves, 8 to 32 rows: 4.2 / 4.5 / 5.4 us, sixteen 4.3 / 4.8 / 5.6).
template <int PAD>
int launch_pad(hipStream_t stream, const uint8_t* packed, const uint16_t* W, const float* residual, float* out, int rows, int N, int K, int parts) {
    if (K / kBlock > 16 * parts) return launch<PAD, 16>(stream, packed, W, residual, out, rows, N, K, parts);
    return launch<PAD, 8>(stream, packed, W, residual, out, rows, N, K, parts);
}

}  // namespace

extern "C" {

size_t m40llm_ext_packed_rows_bytes(uint32_t rows, int K) { return rows >= 1 && rows <= 32 && K >= 256 && K % 256 == 0 ? m40_packed_bytes((int)rows, K) : 0; }

int m40llm_ext_batched_packed_supported(uint32_t rows, int d_model) {
    return (rows <= 8 ? m40_rows_mfma_supported((int)rows, d_model) : m40_rows_wide_supported((int)rows, d_model)) ? 1 : 0;
}

int m40llm_ext_batched_norm_gate_up_swiglu_packed_async(M40llmCudaContext* ctx, const void* d_x_f32, const void* d_norm_w, uint32_t norm_weight_dtype, float eps,
                                                        const void* d_wgate_f16, const void* d_wup_f16, void* d_packed, uint32_t rows, int ffn, int d_model,
                                                        void* d_clear_f32, uint32_t clear_floats) {
    if (!ctx || !d_x_f32 || !d_norm_w || !d_wgate_f16 || !d_wup_f16 || !d_packed) return -1;
    if (!d_clear_f32) clear_floats = 0;
    if (ffn <= 0 || d_model <= 0 || clear_floats > (1u << 30)) return -2;
    if (norm_weight_dtype > 1) return -4;
    const size_t bytes = m40llm_ext_packed_rows_bytes(rows, ffn), x_bytes = (size_t)rows * d_model * 4, clear_bytes = (size_t)clear_floats * 4;
    if (!bytes || !m40llm_ext_batched_packed_supported(rows, d_model) || !m40_aligned16(d_packed) || !m40_apart(d_x_f32, x_bytes, d_packed, bytes)) return -6;
    if (clear_floats && (!m40_apart(d_x_f32, x_bytes, d_clear_f32, clear_bytes) || !m40_apart(d_packed, bytes, d_clear_f32, clear_bytes))) return -6;
    (void)hipGetLastError();
    const float* x = static_cast<const float*>(d_x_f32);
    const uint16_t *gate = static_cast<const uint16_t*>(d_wgate_f16), *up = static_cast<const uint16_t*>(d_wup_f16);
    uint8_t* packed = static_cast<uint8_t*>(d_packed);
    float* clear = clear_floats ? static_cast<float*>(d_clear_f32) : nullptr;
    if (rows <= 8)
        return m40_rows_mfma_swiglu(ctx, ctx->decode_stream, x, d_norm_w, norm_weight_dtype, eps, gate, up, nullptr, packed, (int)rows, ffn, d_model, clear, (int)clear_floats);
    return m40_rows_wide_swiglu(ctx, ctx->decode_stream, x, d_norm_w, norm_weight_dtype, eps, gate, up, nullptr, packed, (int)rows, ffn, d_model, clear, (int)clear_floats);
}

int m40llm_ext_batched_packed_gemm_residual_onto_zero_async(M40llmCudaContext* ctx, const void* d_packed, const void* d_w_f16, const void* d_residual_f32,
                                                            void* d_out_f32, uint32_t rows, int N, int K) {
    if (!ctx || !d_packed || !d_w_f16 || !d_out_f32) return -1;
    if (N <= 0 || K <= 0) return -2;
    const size_t bytes = m40llm_ext_packed_rows_bytes(rows, K), out_bytes = (size_t)rows * N * 4;
    if (!bytes || !m40_aligned16(d_packed) || !m40_aligned16(d_w_f16) || !m40_apart(d_packed, bytes, d_out_f32, out_bytes) ||
        !m40_apart(d_residual_f32, out_bytes, d_out_f32, out_bytes))
        return -6;
    (void)hipGetLastError();
    const uint8_t* packed = static_cast<const uint8_t*>(d_packed);
    const uint16_t* W = static_cast<const uint16_t*>(d_w_f16);
    const float* residual = static_cast<const float*>(d_residual_f32);
    float* out = static_cast<float*>(d_out_f32);
    // halves of K up to half a tile a CU (256 tiles, K 4096, 8 and 32 rows: whole 8.8 and 13.3 us, halves 9.1 and 13.7)
    const int parts = K >= 1024 && 2 * ((N + 15) / 16) <= ctx->num_cus ? 2 : 1;
    const int pad = m40_packed_pad((int)rows);
    if (pad == 8) return launch_pad<8>(ctx->decode_stream, packed, W, residual, out, (int)rows, N, K, parts);
    if (pad == 16) return launch_pad<16>(ctx->decode_stream, packed, W, residual, out, (int)rows, N, K, parts);
    return launch_pad<32>(ctx->decode_stream, packed, W, residual, out, (int)rows, N, K, parts);
}

}  // extern "C"
