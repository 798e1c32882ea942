// Many-row GEMM for prefill: C[M,N] f32 = A[M,K] f32 x B (f16, GGUF order [N][K]), f32 accumulation, on the
// matrix cores.  Same contract as the reference's gemm_f32xf16_gguf_f32 (cuda/kernels.cu:5037-5052); used when M is
// beyond what the skinny kernels serve in one pass, where they would stream the weights once per 16 rows.
//
// Tiling: a workgroup of eight waves owns a tile of C and walks K in steps of 32.  The rows of A are split into an f16 high part and an f16
// low part under a per-row power-of-two scale (a = scale (hi + lo) up to 2^-22 relative; the scale multiplies the row of C at the end);
// v_mfma_f32_16x16x32_f16 runs once with the high and once with the low part, so the products carry the f32 activations' precision.
// Four tile shapes, from 128 x 256 (most products per byte of LDS traffic) to 64 x 64 (most workgroups for few rows), and parts of K where
// even those leave CUs idle; pick_tile() weighs them.
//
// The split is done once per call by a packing pass (A -> two f16 planes in a per-stream buffer that grows on
// demand), so the tiles along N do not each repeat it.  When the buffer cannot be grown (the stream is being
// captured) the launch is declined and the caller falls back to the skinny kernels.  Several weight matrices that
// share A (Q/K/V, gate/up) can be served by one packing pass and one launch.
#include "common.hpp"

#include <numeric>
#include <type_traits>
#include <utility>

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kBK = 32;
constexpr int kMaxMats = 3;

// Up to three weight matrices that share the activations (Q/K/V, gate/up): their column tiles are laid side by side.
struct TiledMats {
    int n;
    const uint16_t* B[kMaxMats];
    float* C[kMaxMats];
    const float* R[kMaxMats];       // not null: C = R + product (R may be C itself)
    int N[kMaxMats];
    int tile_start[kMaxMats + 1];   // first column tile of each matrix; [n] = total
    // B[0] and B[1] are gate and up of N[0] / 2 columns each (a multiple of 16), taken 16 columns at a time in turn as one matrix of N[0];
    // C[0], half as wide, gets SwiGLU of the two: [M][N[0] / 2]
    int pair;
};

// Where the rows of A come from: as they are, RMSNorm of the rows (what m40llm_rms_norm_f32_weighted writes: the same
// sums in the same order, cuda/kernels.cu:770-807), or SwiGLU of two arrays (kernels.cu:869-880).  The packing pass
// produces them on the fly, so the normalised / activated rows are never written out as f32 and read back.
struct PackSource {
    const float* a;
    const float* a2;           // SwiGLU: the up array (a is gate)
    const void* norm_w;        // RMSNorm weights
    uint32_t norm_dtype;       // 0 f16, 1 f32
    float eps;
    // RMSNorm of rows that are still parts of K: row = residual + (plane 0 + plane 1 + ...), written to `sum` (which is `a`) on the way
    const float4 *planes, *residual;
    float4* sum;
    int k_splits;
};
enum { kPackPlain = 0, kPackNorm = 1, kPackSwiglu = 2, kPackSumNorm = 3, kPackDone = 4 };      // done: somebody else writes the planes

// A [M][K] f32 -> hi, lo [M][K] f16 planes and one scale per row: a = scale * (hi + lo) up to 2^-22 relative.  The scale is
// the power of two that brings the row's largest magnitude into [2^10, 2^11) -- any finite f32 row fits the f16 planes,
// and small elements keep their low part out of the f16 subnormals.  The row stays in registers between the maximum and
// the split (up to K = 16384; beyond that it is read a second time).  A row that holds an
// infinity or a NaN is packed unscaled with those elements as they are (their low parts zero), so that its products come
// out non-finite as the f32 arithmetic of the reference would give them (cuda/kernels.cu:5037-5052), never as a finite
// value.
constexpr int kPackChunks = 8;       // most 8-element chunks that a thread keeps in registers
constexpr int kPackStaged = 4096;    // longest row that a norm stages

// SwiGLU of one element, the expression of swiglu_kernel (cuda/kernels.cu:869-880)
__device__ __forceinline__ float tiled_swiglu(float g, float u) {
    const float silu = g / (1.0f + expf(-g));
    return silu * u;
}

__device__ __forceinline__ float pack_abs_or_inf(float v) { return fabsf(v) <= 3.402823466e+38f ? fabsf(v) : INFINITY; }

__device__ __forceinline__ void pack_split8(const float4& x0, const float4& x1, float inv_scale, half8& h, half8& l) {
    const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const bool finite = fabsf(x[j]) <= 3.402823466e+38f;
        // (a row with a non-finite element is not scaled: a finite neighbour beyond the f16 range then saturates, in a
        // row whose products are non-finite wherever that element meets a non-zero weight)
        const float xs = finite ? fminf(fmaxf(x[j] * inv_scale, -65504.0f), 65504.0f) : x[j];
        h[j] = static_cast<_Float16>(xs);
        l[j] = finite ? static_cast<_Float16>(xs - static_cast<float>(h[j])) : static_cast<_Float16>(0.0f);
    }
}

// element i of residual + (plane 0 + plane 1 + ...), n4 elements a plane: requested together, added in order
constexpr int kMaxSplits = 8;
__device__ __forceinline__ float4 sum_planes(const float4* planes, int k_splits, size_t n4, size_t i, const float4* residual) {
    float4 part[kMaxSplits], r = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s)
        if (s < k_splits) part[s] = planes[(size_t)s * n4 + i];
    if (residual) r = residual[i];
    float4 a = part[0];
#pragma unroll
    for (int s = 1; s < kMaxSplits; ++s)
        if (s < k_splits) { a.x += part[s].x; a.y += part[s].y; a.z += part[s].z; a.w += part[s].w; }
    return residual ? make_float4(r.x + a.x, r.y + a.y, r.z + a.z, r.w + a.w) : a;
}

// The planes lie in tiles of 16 rows x 32 k, a kilobyte each, all k of sixteen rows one after the other: what an instruction of the tiled kernel
// loads is contiguous.  A row's stores are half lines, which the L2 of the die that has the tile's sixteen rows puts together (4096 rows of 5632: 32.0
// us as whole rows, 35.1 this way, 39.2 with the rows dealt to the dies in turn).  16-byte chunk of a row's first k, and how far on its chunk c is:
__device__ __forceinline__ size_t plane_chunk(int row, int K) { return m40_tiled_row(row, K) / 8; }
__device__ __forceinline__ size_t plane_step(int c) { return m40_tiled_col(8 * c) / 8; }

// ROW_THREADS = 64: a wave per row, four rows per workgroup, no barrier (K <= 4096 keeps the row in registers);
// 256: a workgroup per row (always for the RMSNorm source, whose sum of squares is formed with the thread layout and
// order of rms_norm_kernel so that the fused form gives the bits of the two-launch form).
// CHUNKS: what a thread keeps.  Registers decide how many rows a CU has in flight: a staged norm needs two chunks, not eight (with the staging 4096 rows of
// 2048 20.8 -> 14.6 us, 4.6 TB/s; 522 rows 7.8 -> 7.5, as parts of K 9.8 -> 9.2), a wave to a row of 2048 four (13.3 -> 12.9).  A workgroup to
// a row keeps eight also where four would do: 4096 rows of 5632 take 34.9 us that way and 38.1 with more rows in flight, which write half lines.
template <int ROW_THREADS, int KIND, int CHUNKS>
__global__ __launch_bounds__(256) void pack_hilo_planes_kernel(PackSource src_args, _Float16* __restrict__ hi,
                                                               _Float16* __restrict__ lo, float* __restrict__ row_scale,
                                                               int M, int K) {
    constexpr bool kNorm = KIND == kPackNorm || KIND == kPackSumNorm;
    static_assert(!kNorm || ROW_THREADS == 256, "the norm's sums follow rms_norm_kernel's layout");
    __shared__ float wave_max[4];
    __shared__ float wave_sums[4];
    // A row that is normed passes through LDS from the order of its sums to that of its chunks, and its weights are asked for ahead of the sums: read again
    // behind the barrier, both cost another round trip, and the row a second pass through the caches
    __shared__ __attribute__((aligned(16))) float4 staged[kNorm ? kPackStaged / 4 : 1];
    constexpr int kRowsPerGroup = 256 / ROW_THREADS;
    // the rows of a tile on one die (m40_tile_row; a workgroup of four rows: four workgroups a tile)
    const uint32_t b = blockIdx.x, groups = gridDim.x;
    const uint32_t group = ROW_THREADS == 256 ? m40_tile_row(b, groups) : ((b | 31u) < groups ? (b & ~31u) + (b & 7u) * 4u + ((b & 31u) >> 3) : b);
    const int row = (int)group * kRowsPerGroup + (int)threadIdx.x / ROW_THREADS, tid = (int)threadIdx.x % ROW_THREADS;
    if (ROW_THREADS == 64 && row >= M) return;          // whole waves: no barrier in this form
    const float4* src = reinterpret_cast<const float4*>(src_args.a + (size_t)row * K);
    const float4* src2 = KIND == kPackSwiglu ? reinterpret_cast<const float4*>(src_args.a2 + (size_t)row * K) : nullptr;
    const int chunks = K >> 3;                     // K is a multiple of 32
    float norm_scale = 1.0f;
    constexpr int kStagedChunks = kPackStaged / 8 / 256;
    static_assert(kStagedChunks <= CHUNKS);
    const bool stage = kNorm && K <= kPackStaged;
    uint4 nw[kNorm ? kStagedChunks : 1][2];
    if (kNorm && stage) {
        // f16 weights: the chunk's sixteen bytes, asked for twice (no load under a branch)
        const uint4* w = static_cast<const uint4*>(src_args.norm_w);
        const int step = src_args.norm_dtype == 0u ? 1 : 2, second = src_args.norm_dtype == 0u ? 0 : 1;
#pragma unroll
        for (int i = 0; i < kStagedChunks; ++i) {
            const int c = tid + 256 * i < chunks ? tid + 256 * i : 0;
            nw[kNorm ? i : 0][0] = w[step * c];
            nw[kNorm ? i : 0][1] = w[step * c + second];
        }
    }
    if (kNorm) {
        float ss = 0.0f;
        const size_t row4 = (size_t)row * (K / 4);
        for (int i = tid; i < K / 4; i += 256) {
            float4 v;
            if (KIND == kPackSumNorm) {
                v = sum_planes(src_args.planes, src_args.k_splits, (size_t)M * (K / 4), row4 + i, src_args.residual);
                src_args.sum[row4 + i] = v;       // long rows: read again behind the barrier below
            } else {
                v = src[i];
            }
            if (stage) staged[kNorm ? i : 0] = v;
            ss = fmaf(v.x, v.x, ss);
            ss = fmaf(v.y, v.y, ss);
            ss = fmaf(v.z, v.z, ss);
            ss = fmaf(v.w, v.w, ss);
        }
        ss = m40_sum64(ss);
        if ((tid & 63) == 0) wave_sums[tid >> 6] = ss;
        __syncthreads();
        float total = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) total += wave_sums[w];
        norm_scale = 1.0f / sqrtf(total / static_cast<float>(K) + src_args.eps);
    }
    // x * scale, then * weight: two roundings, as rms_norm_kernel has them
    auto scale_chunk = [&](const float4 a, const float4 b, const float (&w)[8], float4& o0, float4& o1) {
        o0 = make_float4(a.x * norm_scale * w[0], a.y * norm_scale * w[1], a.z * norm_scale * w[2], a.w * norm_scale * w[3]);
        o1 = make_float4(b.x * norm_scale * w[4], b.y * norm_scale * w[5], b.z * norm_scale * w[6], b.w * norm_scale * w[7]);
    };
    // the eight source values of chunk c
    auto load_chunk = [&](int c, float4& o0, float4& o1) {
        o0 = src[2 * c];
        o1 = src[2 * c + 1];
        if (KIND == kPackSwiglu) {
            const float4 u0 = src2[2 * c], u1 = src2[2 * c + 1];
            o0 = make_float4(tiled_swiglu(o0.x, u0.x), tiled_swiglu(o0.y, u0.y), tiled_swiglu(o0.z, u0.z), tiled_swiglu(o0.w, u0.w));
            o1 = make_float4(tiled_swiglu(o1.x, u1.x), tiled_swiglu(o1.y, u1.y), tiled_swiglu(o1.z, u1.z), tiled_swiglu(o1.w, u1.w));
        }
        if (kNorm) {
            float w[8];
            if (src_args.norm_dtype == 0u) {
                m40_unpack8(reinterpret_cast<const uint4*>(src_args.norm_w)[c], w);
            } else {
                const float4 w0 = reinterpret_cast<const float4*>(src_args.norm_w)[2 * c], w1 = reinterpret_cast<const float4*>(src_args.norm_w)[2 * c + 1];
                w[0] = w0.x; w[1] = w0.y; w[2] = w0.z; w[3] = w0.w; w[4] = w1.x; w[5] = w1.y; w[6] = w1.z; w[7] = w1.w;
            }
            scale_chunk(o0, o1, w, o0, o1);
        }
    };
    const bool in_regs = chunks <= CHUNKS * ROW_THREADS;
    float4 x0[CHUNKS], x1[CHUNKS];
    float mx = 0.0f;
    if (in_regs) {
        if (kNorm && stage) {
#pragma unroll
            for (int i = 0; i < kStagedChunks; ++i) {
                const int c = tid + 256 * i;
                if (c >= chunks) continue;
                const uint4 a = nw[kNorm ? i : 0][0], b = nw[kNorm ? i : 0][1];
                float w[8] = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(a.z), __uint_as_float(a.w),
                              __uint_as_float(b.x), __uint_as_float(b.y), __uint_as_float(b.z), __uint_as_float(b.w)};
                if (src_args.norm_dtype == 0u) m40_unpack8(a, w);
                scale_chunk(staged[kNorm ? 2 * c : 0], staged[kNorm ? 2 * c + 1 : 0], w, x0[i], x1[i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < CHUNKS; ++i) {
                const int c = tid + ROW_THREADS * i;
                if (c < chunks) load_chunk(c, x0[i], x1[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
            if (tid + ROW_THREADS * i < chunks) {
                mx = fmaxf(mx, fmaxf(fmaxf(pack_abs_or_inf(x0[i].x), pack_abs_or_inf(x0[i].y)), fmaxf(pack_abs_or_inf(x0[i].z), pack_abs_or_inf(x0[i].w))));
                mx = fmaxf(mx, fmaxf(fmaxf(pack_abs_or_inf(x1[i].x), pack_abs_or_inf(x1[i].y)), fmaxf(pack_abs_or_inf(x1[i].z), pack_abs_or_inf(x1[i].w))));
            }
        }
    } else {
        for (int c = tid; c < chunks; c += ROW_THREADS) {
            float4 a, b;
            load_chunk(c, a, b);
            mx = fmaxf(mx, fmaxf(fmaxf(pack_abs_or_inf(a.x), pack_abs_or_inf(a.y)), fmaxf(pack_abs_or_inf(a.z), pack_abs_or_inf(a.w))));
            mx = fmaxf(mx, fmaxf(fmaxf(pack_abs_or_inf(b.x), pack_abs_or_inf(b.y)), fmaxf(pack_abs_or_inf(b.z), pack_abs_or_inf(b.w))));
        }
    }
    mx = m40_max64(mx);
    if (ROW_THREADS == 256) {
        if ((tid & 63) == 0) wave_max[tid >> 6] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
    }
    float scale = 1.0f, inv_scale = 1.0f;
    if (mx > 0.0f && mx < INFINITY) {
        int ex;
        (void)frexpf(mx, &ex);        // mx = f * 2^ex, f in [0.5, 1)
        ex -= 11;
        ex = ex < -100 ? -100 : (ex > 100 ? 100 : ex);
        scale = ldexpf(1.0f, ex);
        inv_scale = ldexpf(1.0f, -ex);
    }
    if (tid == 0) row_scale[row] = scale;
    half8* hp = reinterpret_cast<half8*>(hi) + plane_chunk(row, K);
    half8* lp = reinterpret_cast<half8*>(lo) + plane_chunk(row, K);
    if (in_regs) {
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
            const int c = tid + ROW_THREADS * i;
            if (c < chunks) {
                half8 h, l;
                pack_split8(x0[i], x1[i], inv_scale, h, l);
                hp[plane_step(c)] = h;
                lp[plane_step(c)] = l;
            }
        }
    } else {
        for (int c = tid; c < chunks; c += ROW_THREADS) {
            float4 a, b;
            load_chunk(c, a, b);
            half8 h, l;
            pack_split8(a, b, inv_scale, h, l);
            hp[plane_step(c)] = h;
            lp[plane_step(c)] = l;
        }
    }
}

// ---- tiles of 16 WM MT x 16 WN NT per workgroup of WM x WN waves (wave tile 16 MT x 16 NT) ---------------------------------
//
// Measured on a 128 x 128 kernel that staged through registers with parts of it switched off (M 4096, N 2048, K 2048): arithmetic alone
// 46 us, loads + LDS traffic + barriers alone 45 us, everything 87 us -- the two did not overlap.  A wave issues in order, and a
// memory instruction holds the issue slot until its unit accepts it; with the four waves of a CU in step behind the
// barrier, sixteen fragment reads, eight LDS writes and eight global loads each queue for ~500 cycles before the first
// matrix instruction of the step can go.  Here:
//  * every memory instruction of a step is issued under the step's matrix instructions (sched_group_barrier), so it waits for its unit
//    while the matrix pipe works;
//  * the fragments of step s + 1 are read from LDS during the arithmetic of step s (two fragment sets in registers);
//  * global data goes straight into LDS (global_load_lds_dwordx4: no registers, no LDS write instruction, no wait
//    before one), kBufs buffers deep -- a lane fetches the 16-byte chunk that belongs at its place in the swizzled
//    row layout, so a wave's instruction fills one contiguous kilobyte; the workgroup waits only for the step after
//    next (vmcnt) ahead of the barrier that publishes it;
//  * an instruction loads whole lines: of A a kilobyte of the packed planes, of B eight columns of 128 bytes, two steps at a time (kBBufs
//    buffers of those, asked for in every second step).  With 16 rows of 64 bytes an instruction, half lines of both, the launches below took, on
//    one card, 378 us (N 11264), 175 (K 5632) and 112 (N 2560); with both as they are 351, 162 and 105 (whole lines of A alone: 1 to 2 % more than
//    that);
//  * a workgroup is eight waves, two to a SIMD, which fill each other's waits (behind the barrier, between fragments and the first products).  With four, wave tiles twice as large
//    read a quarter to two fifths fewer fragment bytes a product and were slower all the same (us, four / eight waves): 128 x 256 tiles, K 2048, M 4096, N 11264 341 / 331, M 522
//    58.0 / 55.5; 128 x 128, M 2000, N 2048 66.6 / 62.4 (median of K 2048 and 5632), M 1000, N 2560 34.7 / 33.0; 64 x 128, M 522, N 2048 in parts of K 5632 22.9 / 20.7, N 2560
//    22.1 / 20.1; 64 x 64, M 60, N 2048, K 11008 in parts 16.4 / 16.0.
// M 4096, N 2048, K 2048: 79 (128 x 128, through registers) -> 63 us; N 11264: 479 -> 338 us; K 5632: 232 -> 155 us (before the whole lines).  Under this load the part lowers
// its clock (1.4-1.9 GHz measured inside the kernel, against 2.0-2.2 GHz in short or memory-bound launches), and a form
// with fewer issue cycles (32 x 32 x 16 instructions: 1370 instead of 1500 cycles per step) ran at a lower clock
// still and took the same time: what is left is energy per product, of which the exact hi + lo split is half.
struct TileWalk {          // which tile (and part of K) a workgroup owns
    int m0, n0, mat, split;
};
// Workgroups are dealt to the eight dies in turn.  Each die gets a contiguous run of tiles, walked in blocks of `band` tile rows, column
// after column: what runs on a die at one time is then a roughly square block of tiles, which shares the steps of both operands in its L2.
__device__ __forceinline__ TileWalk tile_walk(const TiledMats& mats, int tiles_m, int k_splits, int band, int bm, int bn) {
    const int tiles_n = mats.tile_start[mats.n], per_die = (int)gridDim.x / 8;
    int logical = (int)blockIdx.x < per_die * 8 ? ((int)blockIdx.x % 8) * per_die + (int)blockIdx.x / 8 : (int)blockIdx.x;
    TileWalk w;
    w.split = logical / (tiles_m * tiles_n);
    logical -= w.split * tiles_m * tiles_n;
    const int group = logical / (band * tiles_n), in_group = logical - group * band * tiles_n;
    const int rows = tiles_m - group * band < band ? tiles_m - group * band : band;
    w.m0 = (group * band + in_group % rows) * bm;
    int tile_n = in_group / rows;
    w.mat = 0;
#pragma unroll
    for (int i = 1; i < kMaxMats; ++i)
        if (i < mats.n && tile_n >= mats.tile_start[i]) w.mat = i;
    w.n0 = (tile_n - mats.tile_start[w.mat]) * bn;
    return w;
}

// s_waitcnt for vector-memory operations only: at most n of them may still be outstanding
__device__ __forceinline__ constexpr int vmcnt_only(int n) { return 0x0f70 | (n & 15) | ((n >> 4) << 14); }

// stages of a part of K
template <int KS>
__host__ __device__ constexpr int split_stages(int stages, int k_splits) {
    const int per = (stages + k_splits - 1) / k_splits;
    return KS == 1 && k_splits > 1 ? (per + 1) & ~1 : per;
}

template <int... I, class F>
__device__ __forceinline__ void tiled_unrolled(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }

// KS: k steps of 32 a stage (what is loaded together, between two barriers); kBufs: LDS buffers of a stage each (one
// workgroup is resident per CU).  Two steps a stage read whole 128-byte lines of a column: with weights that no cache holds 64 x 64 tiles of N 2048,
// K 2048 take 15.5 us that way and 21.3 us in stages of one step, 64 x 128 tiles 21.0 and 24.6 us (60 rows).
template <int MT, int NT, int WM, int WN, int KS, int kBufs, int kBBufs, bool FINE>
__global__ __launch_bounds__(64 * WM * WN, 1) void gemm_tiled_kernel(const _Float16* __restrict__ A_hi, const _Float16* __restrict__ A_lo,
                                                                      const float* __restrict__ row_scale, TiledMats mats, int M, int K,
                                                                      int k_splits, int band) {
    typedef __attribute__((address_space(3))) void* lds_dst_t;
    typedef const __attribute__((address_space(1))) void* global_src_t;
    constexpr int kThreads = 64 * WM * WN, BM = 16 * WM * MT, BN = 16 * WN * NT;
    constexpr int kRow = 64 * KS, kLoadRows = kThreads / (4 * KS);           // bytes of a row of A in a stage; rows the workgroup loads at a time
    constexpr int kRowB = 128, kLoadRowsB = kThreads / 8;                    // of B, always two steps
    constexpr int kPlane = BM * kRow, kBuf = 2 * kPlane, kBufB = BN * kRowB, kB0 = kBufs * kBuf;      // bytes: a plane of a stage, both, B of two steps; where B starts
    constexpr int AL = BM / kLoadRows, BL = BN / kLoadRowsB;                 // 16-byte loads per thread: rows lrow + kLoadRows i
    extern __shared__ __align__(16) uint8_t tile_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    TileWalk at = tile_walk(mats, (M + BM - 1) / BM, k_splits, band, BM, BN);
    at.m0 = __builtin_amdgcn_readfirstlane(at.m0); at.n0 = __builtin_amdgcn_readfirstlane(at.n0);      // the same in every lane: divisions leave them in vector registers
    at.mat = __builtin_amdgcn_readfirstlane(at.mat); at.split = __builtin_amdgcn_readfirstlane(at.split);
    const int N = mats.N[at.mat], m0 = at.m0, n0 = at.n0;
    // in a pair a wave's eight rows of a load are one matrix's (the next ones an even number of sixteens further)
    const uint16_t* __restrict__ B = mats.B[mats.pair ? (wave >> 1) & 1 : at.mat];
    // loader: thread -> row lrow (+ kLoadRows i) of a plane and a 16-byte place in that row's bytes, which holds the row's chunk of that number
    // xor-ed with bits of the row: the fragment reads of rows that share banks fall into different ones
    auto swizzle = [](int row) { return KS == 1 ? (row >> 2) & 3 : row & 7; };
    const int lrow = tid / (4 * KS), gchunk = tid % (4 * KS) ^ swizzle(lrow), lrow_b = tid / 8, gchunk_b = tid % 8 ^ (lrow_b & 7);
    // (stages of one step: an even number of them to a part of K)
    const int stages_all = K / (kBK * KS), per_split = __builtin_amdgcn_readfirstlane(split_stages<KS>(stages_all, k_splits)), stage0 = at.split * per_split;
    const int stages = stage0 + per_split <= stages_all ? per_split : stages_all - stage0;     // >= 1 by the host's choice of k_splits
    // a scalar address that walks K, and per lane a 32-bit offset from it that does not change
    const uint8_t* hi_base = reinterpret_cast<const uint8_t*>(A_hi + (size_t)m0 * K) + (size_t)stage0 * (KS * 1024);
    const uint8_t* lo_base = reinterpret_cast<const uint8_t*>(A_lo + (size_t)m0 * K) + (size_t)stage0 * (KS * 1024);
    const uint8_t* b_base = reinterpret_cast<const uint8_t*>(B + (size_t)(mats.pair ? n0 / 2 : n0) * K + (size_t)stage0 * (kBK * KS));
    uint32_t a_off[AL], b_off[BL];
#pragma unroll
    for (int i = 0; i < AL; ++i) {
        const int r = m0 + lrow + kLoadRows * i < M ? lrow + kLoadRows * i : M - 1 - m0;      // clamped: computed, never stored
        a_off[i] = (uint32_t)(r >> 4) * (uint32_t)K * 32u + (gchunk >> 2) * 1024u + (r & 15) * 64u + (gchunk & 3) * 16u;
    }
#pragma unroll
    for (int i = 0; i < BL; ++i) {
        const int c = lrow_b + kLoadRowsB * i, last = mats.pair ? N / 2 - 1 - n0 / 2 : N - 1 - n0, col = mats.pair ? c / 32 * 16 + c % 16 : c;
        b_off[i] = (uint32_t)(col < last ? col : last) * (uint32_t)K * 2u + gchunk_b * 16u;
    }
    // one instruction of a wave fills a contiguous kilobyte of a buffer, lane by lane; past the end: the last stage again (no branch around loads)
    auto issue_a = [&](int buf, int stage) __attribute__((always_inline)) {
        int k = (stage < stages ? stage : stages - 1) * (KS * 1024);
        asm("" : "+s"(k));                                                      // keeps it out of the lanes' addresses
        uint8_t* dst = tile_lds + buf * kBuf + wave * 1024;
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            __builtin_amdgcn_global_load_lds((global_src_t)(hi_base + k + a_off[i]), (lds_dst_t)(dst + i * (16 * kThreads)), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((global_src_t)(lo_base + k + a_off[i]), (lds_dst_t)(dst + kPlane + i * (16 * kThreads)), 16, 0, 0);
        }
    };
    // B of the steps 2 pair and 2 pair + 1 (one stage where a stage is two steps); of an odd number of steps the last one is read twice
    const int pairs = KS == 2 ? stages : (stages + 1) / 2;
    const bool odd = KS == 1 && stages % 2 != 0;
    const uint32_t second = gchunk_b >= 4 ? 64u : 0u;
    auto issue_b = [&](int buf, int pair) __attribute__((always_inline)) {
        const int p = pair < pairs ? pair : pairs - 1;
        int k = p * kRowB;
        asm("" : "+s"(k));
        const uint32_t back = odd && p == pairs - 1 ? second : 0u;
        uint8_t* dst = tile_lds + kB0 + buf * kBufB + wave * 1024;
#pragma unroll
        for (int i = 0; i < BL; ++i)
            __builtin_amdgcn_global_load_lds((global_src_t)(b_base + k + (KS == 1 ? b_off[i] - back : b_off[i])), (lds_dst_t)(dst + i * (16 * kThreads)), 16, 0, 0);
    };
    const int wm = wave / WN, wn = wave % WN, frag_row = lane & 15;
    float scale[MT];                   // of the rows this lane will store, requested ahead of everything else
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int row = m0 + (wm * MT + mt) * 16 + frag_row;
        scale[mt] = row_scale[row < M ? row : M - 1];
    }
    struct Frags { half8 hi[MT], lo[MT], b[NT]; } f[2];
    // fragments of a step: which buffers, and which of a buffer's steps
    auto read_frags = [&](Frags& f, int buf, int sub, int buf_b, int sub_b) __attribute__((always_inline)) {
        const uint8_t* a = tile_lds + buf * kBuf + (wm * MT * 16 + frag_row) * kRow + (((lane >> 4) + 4 * sub) ^ swizzle(frag_row)) * 16;
        const uint8_t* b = tile_lds + kB0 + buf_b * kBufB + (wn * NT * 16 + frag_row) * kRowB + (((lane >> 4) + 4 * sub_b) ^ (frag_row & 7)) * 16;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            f.hi[mt] = *reinterpret_cast<const half8*>(a + mt * 16 * kRow);
            f.lo[mt] = *reinterpret_cast<const half8*>(a + kPlane + mt * 16 * kRow);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) f.b[nt] = *reinterpret_cast<const half8*>(b + nt * 16 * kRowB);
    };
    floatx4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    // Per accumulator step by step, high part then low part: the two large tiles give the same bits.  (FINE: the low parts' sums apart.)  The weights are the instruction's
    // first operand, so a lane's four sums are four neighbouring columns of one row and a store is 16 bytes.
    constexpr bool kBlocked = BM * BN <= 64 * 128;
    static_assert(kBlocked || !FINE);
    floatx4 low[FINE ? MT : 1][FINE ? NT : 1];
    if (FINE) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) low[FINE ? i : 0][FINE ? j : 0] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    auto compute = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[nt], f.hi[mt], acc[mt][nt], 0, 0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                floatx4& to = FINE ? low[FINE ? mt : 0][FINE ? nt : 0] : acc[mt][nt];
                to = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[nt], f.lo[mt], to, 0, 0, 0);
            }
        }
    };
    // The barriers are bare s_barrier instructions with the vector-memory wait written out: __syncthreads() would wait for every
    // outstanding load (its fence covers LDS).
    auto wait_and_meet = [&](auto n) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(vmcnt_only(decltype(n)::value));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    // What stage s asks for: A of stage s + kBufs - 1, then B: with two steps a stage that of the same stage, else in every second step the pair whose
    // buffer the step before last was the last to read (fragments are in registers one barrier later).  `at`: how many loads may be outstanding at
    // the end of stage s, behind which the fragments of stage s + 2 are read.
    struct Flight {
        static constexpr bool asks_b(int s) { return KS == 2 || s % 2 == 0; }
        static constexpr int pair(int s) { return KS == 2 ? s + kBBufs - 1 : s / 2 - 1 + kBBufs; }
        static constexpr int of(int s) { return 2 * AL + (asks_b(s) ? BL : 0); }
        static constexpr int at(int s) {
            int behind_a = asks_b(s + 3 - kBufs) ? BL : 0, behind_b = 0;
            for (int t = s + 4 - kBufs; t <= s; ++t) behind_a += of(t);
            for (int t = KS == 2 ? s + 4 - kBBufs : s / 2 * 2 + 5 - 2 * kBBufs; t <= s; ++t) behind_b += of(t);
            return behind_a < behind_b ? behind_a : behind_b;
        }
    };
    constexpr int kEven = 64;           // of the stages before the first, counted from here
    static_assert(kBBufs >= 3 && kBufs >= 4 && (KS == 1 || kBufs == kBBufs));
#pragma unroll
    for (int t = kEven - 2 * kBBufs - kBufs; t < kEven; ++t) {
        if (t + kBufs - 1 >= kEven) issue_a(t + kBufs - 1 - kEven, t + kBufs - 1 - kEven);
        const int pair = KS == 2 ? t - kEven + kBBufs - 1 : t / 2 - kEven / 2 - 1 + kBBufs;
        if (Flight::asks_b(t) && pair >= 0) issue_b(pair, pair);
    }
    wait_and_meet(std::integral_constant<int, Flight::at(kEven - 1)>());               // stages 0 and 1 have landed
    read_frags(f[0], 0, 0, 0, 0);
    // Step u of a stage: the next step's fragments are read (the next stage's first ones behind its last step: its buffers are complete and
    // visible), then its products.  Stage s refills the buffer of stage s - 1 -- whose fragments every wave had in registers before
    // the last barrier -- with stage s + kBufs - 1, and ends with stage s + 2 landed.  ph: the stage's number in a period, after which buffers
    // and fragment sets are back in their order: written out so that their addresses are constants and sums stay in their registers (a loop of
    // two stages moved 200 accumulation registers a turn: 169 against 161 us at M 4096, N 2048, K 5632).
    constexpr int kPeriod = KS == 2 ? kBufs : std::lcm(kBufs, 2 * kBBufs);
    auto sub_step = [&](auto ph_c, auto sub_c, int s) __attribute__((always_inline)) {
        constexpr int ph = decltype(ph_c)::value, sub = decltype(sub_c)::value, set = (ph * KS + sub) & 1;
        constexpr int next = ph + (KS == 1 || sub == 1);          // the next step's stage
        if constexpr (KS == 2) read_frags(f[set ^ 1], next % kBufs, sub ^ 1, next % kBBufs, sub ^ 1);
        else read_frags(f[set ^ 1], next % kBufs, 0, next / 2 % kBBufs, next % 2);
        constexpr bool loads_b = sub == 0 && Flight::asks_b(ph);
        if constexpr (sub == 0) issue_a((ph + kBufs - 1) % kBufs, s + kBufs - 1);
        if constexpr (loads_b) issue_b(Flight::pair(ph) % kBBufs, Flight::pair(s));
        compute(f[set]);
        constexpr int kReads = 2 * MT + NT, kProducts = 2 * MT * NT, kLoads = (sub == 0 ? 2 * AL : 0) + (loads_b ? BL : 0);
#pragma unroll
        for (int i = 0; i < kReads; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if constexpr (kLoads > 0) {
            constexpr int kPerLoad = (kProducts - kReads) / kLoads > 0 ? (kProducts - kReads) / kLoads : 1;
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, kPerLoad, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](auto ph_c, int s) __attribute__((always_inline)) {
        sub_step(ph_c, std::integral_constant<int, 0>(), s);
        if constexpr (KS == 2) sub_step(ph_c, std::integral_constant<int, 1>(), s);
        wait_and_meet(std::integral_constant<int, Flight::at(kEven + decltype(ph_c)::value)>());
    };
    // Small tiles have registers to keep the sums of a period (10 or 12 steps) apart from those before: a fraction of the chain of roundings
    // that all of K would be (as short as the parts of K that small grids are otherwise cut into).  FINE, for one row of tiles, where that costs a hundredth and
    // not several: twice a period, so that few rows, which other kernels would take otherwise, are no further from 64-bit products than those leave them.  Errors in units of 1e-7
    // of a row's mean at K 2048 and 5632: those kernels 1.2-1.3 up to 8 rows and 1.6-1.7 up to 32; a chain a period 1.7-1.9; FINE 1.1-1.2.
    floatx4 total[kBlocked ? MT : 1][kBlocked ? NT : 1];
    if (kBlocked) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) total[kBlocked ? i : 0][kBlocked ? j : 0] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    auto set_aside = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < (kBlocked ? MT : 0); ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                if (FINE) acc[i][j] += low[FINE ? i : 0][FINE ? j : 0];
                total[kBlocked ? i : 0][kBlocked ? j : 0] += acc[i][j];
                acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
                if (FINE) low[FINE ? i : 0][FINE ? j : 0] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
    };
    constexpr auto set_aside_behind = [](int ph) { return kBlocked && (ph + 1 == kPeriod || (FINE && ph + 1 == kPeriod / 2)); };
    int s = 0;
    for (; s + kPeriod <= stages; s += kPeriod) {
        tiled_unrolled(std::make_integer_sequence<int, kPeriod>(), [&](auto ph_c) __attribute__((always_inline)) {
            stage(ph_c, s + decltype(ph_c)::value);
            if constexpr (set_aside_behind(decltype(ph_c)::value)) set_aside();
        });
    }
    tiled_unrolled(std::make_integer_sequence<int, kPeriod - 1>(), [&](auto ph_c) __attribute__((always_inline)) {
        if (s + decltype(ph_c)::value < stages) stage(ph_c, s + decltype(ph_c)::value);
        if constexpr (set_aside_behind(decltype(ph_c)::value)) set_aside();
    });
    if (kBlocked) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                if (FINE) acc[i][j] += low[FINE ? i : 0][FINE ? j : 0];
                acc[i][j] += total[kBlocked ? i : 0][kBlocked ? j : 0];
            }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));      // no write into LDS may be outstanding when the workgroup ends

    // lane: row lane % 16, columns 4 (lane / 16) .. + 3 of each 16 x 16 tile
    float* __restrict__ C = mats.C[at.mat] + (size_t)at.split * M * N;
    const float* R = k_splits == 1 ? mats.R[at.mat] : nullptr;      // a K split adds the residual when it adds the planes
    const bool whole = N % 4 == 0 && m40_aligned16(mats.C[at.mat]) && m40_aligned16(R);
    const int col0 = n0 + wn * NT * 16 + 4 * (lane >> 4);
    // With a residual: per group of 16 rows its values first -- unconditional loads from clamped addresses, no branch and no wait between
    // them -- then the stores; a load that follows a store to memory it might alias is not moved ahead of it, and a load under a
    // per-lane branch is awaited at the branch's end (measured with both mistakes in place: +10 us on a 65 us launch).
    auto store_tile = [&](auto with_residual) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int row = m0 + (wm * MT + mt) * 16 + frag_row;
            const size_t row_off = (size_t)(row < M ? row : M - 1) * N;
            floatx4 res[NT];
            if (decltype(with_residual)::value) {
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const int col = col0 + nt * 16;
                    if (whole) {
                        res[nt] = *reinterpret_cast<const floatx4*>(R + row_off + (col < N ? col : 0));
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) res[nt][r] = R[row_off + (col + r < N ? col + r : N - 1)];
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (row >= M) continue;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int col = col0 + nt * 16;
                floatx4 v = acc[mt][nt];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    v[r] *= scale[mt];       // a power of two: exact, also on the partial sums of a K split
                    if (decltype(with_residual)::value) v[r] = res[nt][r] + v[r];
                }
                if (whole) {
                    if (col < N) *reinterpret_cast<floatx4*>(C + row_off + col) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (col + r < N) C[row_off + col + r] = v[r];
                }
            }
        }
    };
    if (mats.pair) {
        const int half = N / 2, pair_col0 = (n0 + wn * NT * 16) / 2 + 4 * (lane >> 4);
        const bool whole_pair = m40_aligned16(C);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int row = m0 + (wm * MT + mt) * 16 + frag_row;
            if (row >= M) continue;
#pragma unroll
            for (int nt = 0; nt < NT; nt += 2) {
                const int col = pair_col0 + nt * 8;
                if (col >= half) continue;
                floatx4 v;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = tiled_swiglu(acc[mt][nt][r] * scale[mt], acc[mt][nt + 1][r] * scale[mt]);
                float* o = C + (size_t)row * half + col;
                if (whole_pair) {
                    *reinterpret_cast<floatx4*>(o) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = v[r];
                }
            }
        }
        return;
    }
    if (R) store_tile(std::true_type{});
    else store_tile(std::false_type{});
}

template <int MT, int NT, int WM, int WN, int KS, int kBufs, int kBBufs, bool FINE = false>
int launch_tiles(hipStream_t stream, const _Float16* hi, const _Float16* lo, const float* row_scale, TiledMats mats, int M, int K, int k_splits) {
    constexpr int BM = 16 * WM * MT, BN = 16 * WN * NT, bytes = kBufs * 2 * BM * 64 * KS + kBBufs * BN * 128;
    static_assert(bytes <= 160 * 1024);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tiled_kernel<MT, NT, WM, WN, KS, kBufs, kBBufs, FINE>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (attr != hipSuccess) return -2;
    const int tiles_m = (M + BM - 1) / BM;
    long long tiles_n = 0;
    for (int i = 0; i < mats.n; ++i) {
        mats.tile_start[i] = (int)tiles_n;
        tiles_n += (mats.N[i] + BN - 1) / BN;
    }
    mats.tile_start[mats.n] = (int)tiles_n;
    // On the 128 x 256 tile, bands of 1 / 2 / 4 / 6 / 7 / 9 / 16 rows: M 4096 (32 tile rows), N 11264, K 2048 413 / 360 / 320 / 310 / 302 / 305 / 314 us; N 2048, K 5632
    // 157 / 165 / 157 / 146 / 140 / 141 / 141; M 2048, N 11264, K 2048 174 / 200 / 175 / 162 / 163 / 159 / 161.  M 522, N 2048, K 5632 on 64 x 128 (9 tile rows), bands of 1 / 3 / 5 /
    // 9: 44.7 / 46.8 / 45.9 / 43.7
    const int band = tiles_m <= 9 ? tiles_m : 6;
    gemm_tiled_kernel<MT, NT, WM, WN, KS, kBufs, kBBufs, FINE><<<(unsigned)(tiles_m * tiles_n * k_splits), 64 * WM * WN, bytes, stream>>>(hi, lo, row_scale, mats, M, K, k_splits, band);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Which tile, and into how many parts to cut K.  A launch of t workgroups on c CUs takes, per step of 32 k, about
// max(least, start * ceil(t / c) + load * t / c): a workgroup alone on its CU is bound by the round trips of a step, more of them by the step's
// products and LDS traffic, and by caches and clock when the other CUs work too.  The constants were fitted to 50 shapes in tiles of four waves, those of 128 x 128 again for eight.  us with
// eight, the whole of K, weights that no cache holds (128 x 256 / 128 x 128 / 64 x 128 / 64 x 64, in brackets what is chosen where K is not cut):
//   K 2048, N 2048: 60 rows 40.2 / 26.2 / 24.0 / 18.2, 250 rows 41.1 / 25.0 / 17.4 / 13.7, 522 rows 41.8 / 24.7 / [16.8] / 21.4, 1030 rows 44.4 / [28.5] / 32.3 / 35.4, 2048 rows
//     47.7 / [33.5] / 41.9 / 55.1, 4096 rows [56.3] / 62.9 / 72.5 / 96.6, 4300 rows [92.3] / 82.6 / 90 / 108;  K 5632: 4096 rows [142] / 161 / 186 / 276, 4300 rows [237] / 212 / 226 / 285
//   N 2560: 522 rows 42.0 / 25.9 / [17.9] / 24.4, 2000 rows [49.0] / 54.2 / 51.7 / 59.7, 3000 rows [54.6] / 62.1 / 80 / 103, 3500 rows [93.1] / 84.5 / 90 / 109, 4096 rows [95.4] / 86.2 / 92 / 120
//   N 11264: 522 rows [53.2] / 59.9 / 66.2 / 85.9, 1000 rows 101.5 / [95.4] / 117 / 150, 1500 rows 146.7 / [145.1] / 163 / 219, 2000 rows [165] / 178 / 231 / 299, 3000 rows [283] / 290 / 358 / 451,
//     4096 rows [352] / 400 / 464 / 610
// Parts of K cost the launch that adds their sums; N 2048, K 5632 at 250 rows: 35.9 us whole, 19.7 us and that launch in parts.
struct TileChoice { int shape, k_splits; };
constexpr struct { int bm, bn; float least, start, load; } kShapes[4] = {
    {128, 256, 0.66f, 0.62f, 0.28f}, {128, 128, 0.44f, 0.37f, 0.13f}, {64, 128, 0.28f, 0.25f, 0.05f}, {64, 64, 0.235f, 0.17f, 0.03f}};
// The two large tiles add up all of their part of K in one chain: in small grids they are taken for four parts only (K 2048 is where a chain's error
// shows: 64 steps and more).  The two small tiles, which add up blocks of k, are for small grids and for one row of tiles; past
// that the larger ones are faster (above, 1030 rows), and a row's sums do not depend on how many rows come with it.
TileChoice pick_tile(int M, int n_mats, const int* N, int steps, int num_cus, bool small_grid, bool may_split) {
    TileChoice best{1, may_split && steps >= 64 ? 4 : 1};        // what is left for a small grid of an odd number of steps
    float best_us = 3.0e38f;
    float out_mb = 0.0f;
    for (int i = 0; i < n_mats; ++i) out_mb += (float)M * (float)N[i] * 4e-6f;
    for (int c = 0; c < 4; ++c) {
        if (c >= 2 && (steps % 2 != 0 || !(small_grid || M <= 128))) break;            // the small tiles take two steps a stage
        long long tiles = 0;
        for (int i = 0; i < n_mats; ++i) tiles += (N[i] + kShapes[c].bn - 1) / kShapes[c].bn;
        tiles *= (M + kShapes[c].bm - 1) / kShapes[c].bm;
        for (int s = 1; s <= kMaxSplits; ++s) {
            const int per = s == 1 ? steps : ((steps + s - 1) / s + 1) & ~1;
            if (s > 1 && (!may_split || per < 16 || (long long)per * (s - 1) >= steps || tiles * (s - 1) >= num_cus)) break;
            if (c < 2 && may_split && s < 4 && per >= 32) continue;
            if (c < 2 && small_grid && !may_split && steps >= 64 && steps % 2 == 0) continue;
            const long long units = (tiles * s + num_cus - 1) / num_cus;
            // Past 2048 rows 128 x 128 keeps about the price that it had with four waves, which leaves every choice for the two dense models as it was.  Alone it is the faster one where
            // 128 x 256 has just begun another round (above, 3500, 4096 and 4300 rows).  But thousands of rows run at the part's power, where a tile that reads more bytes a product slows down
            // what comes next, and how much depends on the card.  Whole prompts, ms, with 128 x 128 there / with 128 x 256: TinyLlama on one card, 3300 tokens 17.14 / 16.93, 3500 17.68 /
            // 17.26, 4096 20.15 / 19.69; on another 3300 16.24 / 16.43, 3500 17.06 / 17.30, 4096 19.10 / 19.30, 4300 22.66 / 23.12, 4800 25.26 / 25.49, 5500 28.72 / 28.84, 7600 41.39 / 41.25,
            // Qwen2.5-3B 3300 39.5 / 39.9, 4600 61.2 / 61.9, 5500 72.2 / 71.9, 6700 90.1 / 89.1 (four waves, 128 x 256: TinyLlama 4096 19.96 and 19.54, Qwen2.5-3B 4600 63.3).  From 2049
            // to 3200 rows both prices choose alike there.  Up to 2048 rows the fitted price: gate and up in 128 x 128 tiles, 800 tokens 5.54 ms against 5.65, 1000 5.96 / 6.08, 1500 8.10 / 8.18.
            const float load = c == 1 && M > 2048 ? 0.22f : kShapes[c].load;
            const float a = kShapes[c].start * (float)units + load * (float)(tiles * s) / (float)num_cus;
            float us = (float)per * (a > kShapes[c].least ? a : kShapes[c].least);
            if (s > 1) us += 6.0f + (float)(s + 1) * out_mb / 5.0f;       // MB over TB/s are us
            if (us < best_us) { best_us = us; best = {c, s}; }
        }
    }
    return best;
}

// out[i] = planes[0][i] + planes[1][i] + ... in that order (n4 float4 per plane), then residual[i] + that (residual may be
// out); blockIdx.y = matrix, so the up to three matrices of a launch are summed by one launch as well
struct KPlaneSet {
    const float4* planes[kMaxMats];
    const float4* residual[kMaxMats];
    float4* out[kMaxMats];
    size_t n4[kMaxMats];
};
__global__ __launch_bounds__(256) void add_k_planes_kernel(KPlaneSet set, int k_splits) {
    const int m = blockIdx.y;
    const size_t n4 = set.n4[m];
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    set.out[m][i] = sum_planes(set.planes[m], k_splits, n4, i, set.residual[m]);
}

}  // namespace

bool m40_gemm_tiled_supported(const void* A, const void* B, int M, int N, int K) {
    return M > 32 && N >= 16 && K >= kBK && K % kBK == 0 && m40_aligned16(A) && m40_aligned16(B) &&
           ((long long)((M + 127) / 128) * ((N + 127) / 128)) <= 0x3fffffffll;
}

namespace {

int padded_rows(int M) { return (M + 15) / 16 * 16; }

struct TiledCall {
    int source_kind;
    PackSource source;
    int M, K, n_mats;
    const uint16_t* const* B;
    const int* N;
    float* const* C;
    const float* const* R;
    bool pair;
};
struct TiledPlan {
    TiledMats mats;
    TileChoice choice;
    size_t scale_bytes, need;      // bytes of the row scales; of the packing buffer
};

int plan_tiled(const M40llmCudaContext* ctx, const TiledCall& c, TiledPlan& plan) {
    const PackSource& src = c.source;
    if (c.n_mats < 1 || c.n_mats > kMaxMats || c.source_kind < kPackPlain || (c.source_kind > kPackSwiglu && c.source_kind != kPackDone)) return -2;
    if (c.pair && (c.n_mats != 2 || c.N[0] != c.N[1] || c.N[0] % 16 != 0 || c.N[0] > 0x3fffffff || c.R)) return -2;
    if (c.source_kind == kPackSwiglu && (!src.a2 || !m40_aligned16(src.a2))) return -2;
    if (c.source_kind == kPackNorm && (!src.norm_w || src.norm_dtype > 1u || !m40_aligned16(src.norm_w))) return -2;
    TiledMats& mats = plan.mats = TiledMats{};
    mats.n = c.n_mats;
    long long tiles_128 = 0;
    for (int i = 0; i < c.n_mats; ++i) {
        if (!m40_gemm_tiled_supported(src.a, c.B[i], c.M, c.N[i], c.K) || !(c.C[i] || (c.pair && i == 1))) return -2;
        mats.B[i] = c.B[i];
        mats.C[i] = c.C[i];
        mats.R[i] = c.R ? c.R[i] : nullptr;
        mats.N[i] = c.N[i];
        tiles_128 += (c.N[i] + 127) / 128;
    }
    if ((long long)((c.M + 127) / 128) * tiles_128 > 0x7fffffffll / 8) return -2;
    // Parts of K: partial sums go to planes behind the packed activations and are added in a fixed order by a second launch (every N a
    // multiple of 4 for its float4 accesses) or by the pass that packs them for the next product.  From half a 128 x 128 tile per CU on a split only
    // adds a pass over the sums (1030 rows of N 2048, K 5632, 144 tiles: 77.7 us whole, 78.5 us in the best parts).
    bool n4_ok = true;
    size_t out_floats = 0;
    for (int i = 0; i < c.n_mats; ++i) {
        n4_ok = n4_ok && c.N[i] % 4 == 0 && m40_aligned16(c.C[i]) && m40_aligned16(mats.R[i]);
        out_floats += (size_t)c.M * c.N[i];
    }
    const bool small_grid = (c.M + 127) / 128 * tiles_128 <= ctx->num_cus / 2;
    const int pair_n = c.pair ? 2 * c.N[0] : 0;
    if (c.pair && small_grid && c.K / kBK % 2 != 0) return 1;
    if (c.pair) { mats.pair = 1; mats.n = 1; mats.N[0] = pair_n; }
    plan.choice = pick_tile(c.M, mats.n, c.pair ? &pair_n : c.N, c.K / kBK, ctx->num_cus, small_grid, small_grid && n4_ok && !c.pair);
    plan.scale_bytes = ((size_t)c.M * 4 + 15) & ~(size_t)15;
    plan.need = (size_t)padded_rows(c.M) * c.K * 4 + plan.scale_bytes + (plan.choice.k_splits > 1 ? (size_t)plan.choice.k_splits * out_floats * 4 : 0);
    return 0;
}

// two f16 planes of A (and the partial sums of a K split) in the stream's packing buffer, grown on demand (never while
// the stream is being captured: 1, and the caller uses another kernel)
int provide_pack(M40StreamScratch& sc, hipStream_t stream, size_t need) {
    if (sc.tiled_pack_bytes < need) {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return 1;
        if (hipStreamSynchronize(stream) != hipSuccess) return -2;
        if (sc.tiled_pack) (void)hipFree(sc.tiled_pack);
        sc.tiled_pack = nullptr;
        sc.tiled_pack_bytes = 0;
        const size_t want = need + need / 4;
        if (hipMalloc(&sc.tiled_pack, want) != hipSuccess) {
            (void)hipGetLastError();
            return 1;
        }
        sc.tiled_pack_bytes = want;
    }
    (void)hipGetLastError();
    return 0;
}

// leave: a split product of one matrix leaves its parts for the next call's packing pass, which finds them there
int enqueue_tiled(const M40StreamScratch& sc, hipStream_t stream, const TiledCall& c, const TiledPlan& plan, PackSource* leave) {
    const int M = c.M, K = c.K, k_splits = plan.choice.k_splits;
    _Float16* hi = static_cast<_Float16*>(sc.tiled_pack);
    _Float16* lo = hi + (size_t)padded_rows(M) * K;
    float* row_scale = reinterpret_cast<float*>(static_cast<char*>(sc.tiled_pack) + (size_t)padded_rows(M) * K * 4);
    const PackSource& source = c.source;
    const bool wave_rows = K <= kPackChunks * 64 * 8;
    const auto pack = [&](auto row_threads, auto kind, auto chunks) {
        constexpr int kRowThreads = decltype(row_threads)::value;
        pack_hilo_planes_kernel<kRowThreads, decltype(kind)::value, decltype(chunks)::value>
            <<<(unsigned)(kRowThreads == 64 ? (M + 3) / 4 : M), 256, 0, stream>>>(source, hi, lo, row_scale, M, K);
    };
    const auto pack_norm = [&](auto kind) {
        if (K <= kPackStaged) pack(std::integral_constant<int, 256>(), kind, std::integral_constant<int, kPackStaged / 8 / 256>());
        else pack(std::integral_constant<int, 256>(), kind, std::integral_constant<int, kPackChunks>());
    };
    const auto pack_either = [&](auto kind) {
        if (wave_rows && K <= 4 * 8 * 64) pack(std::integral_constant<int, 64>(), kind, std::integral_constant<int, 4>());
        else if (wave_rows) pack(std::integral_constant<int, 64>(), kind, std::integral_constant<int, kPackChunks>());
        else pack(std::integral_constant<int, 256>(), kind, std::integral_constant<int, kPackChunks>());
    };
    if (c.source_kind == kPackDone) {}
    else if (c.source_kind == kPackNorm && source.planes) pack_norm(std::integral_constant<int, kPackSumNorm>());
    else if (c.source_kind == kPackNorm) pack_norm(std::integral_constant<int, kPackNorm>());
    else if (c.source_kind == kPackSwiglu) pack_either(std::integral_constant<int, kPackSwiglu>());
    else pack_either(std::integral_constant<int, kPackPlain>());
    float* partial = reinterpret_cast<float*>(static_cast<char*>(sc.tiled_pack) + (size_t)padded_rows(M) * K * 4 + plan.scale_bytes);
    TiledMats launch = plan.mats;
    if (k_splits > 1) {
        size_t at = 0;
        for (int i = 0; i < c.n_mats; ++i) {
            launch.C[i] = partial + at;
            at += (size_t)k_splits * M * c.N[i];
        }
    }
    int rc = -2;
    switch (plan.choice.shape) {
        case 0: rc = launch_tiles<4, 4, 2, 4, 1, 4, 3>(stream, hi, lo, row_scale, launch, M, K, k_splits); break;
        case 1: rc = launch_tiles<2, 4, 4, 2, 1, 6, 3>(stream, hi, lo, row_scale, launch, M, K, k_splits); break;
        case 2: rc = M <= 64 ? launch_tiles<2, 2, 2, 4, 2, 5, 5, true>(stream, hi, lo, row_scale, launch, M, K, k_splits) : launch_tiles<2, 2, 2, 4, 2, 5, 5>(stream, hi, lo, row_scale, launch, M, K, k_splits); break;
        case 3: rc = M <= 64 ? launch_tiles<1, 2, 4, 2, 2, 6, 6, true>(stream, hi, lo, row_scale, launch, M, K, k_splits) : launch_tiles<1, 2, 4, 2, 2, 6, 6>(stream, hi, lo, row_scale, launch, M, K, k_splits); break;
    }
    if (rc != 0) return rc;
    if (k_splits > 1 && leave) {
        leave->planes = reinterpret_cast<const float4*>(launch.C[0]);
        leave->residual = reinterpret_cast<const float4*>(plan.mats.R[0]);
        leave->sum = reinterpret_cast<float4*>(c.C[0]);
        leave->k_splits = k_splits;
    } else if (k_splits > 1) {
        KPlaneSet set{};
        size_t blocks = 0;
        for (int i = 0; i < c.n_mats; ++i) {
            set.planes[i] = reinterpret_cast<const float4*>(launch.C[i]);
            set.residual[i] = reinterpret_cast<const float4*>(plan.mats.R[i]);
            set.out[i] = reinterpret_cast<float4*>(c.C[i]);
            set.n4[i] = (size_t)M * c.N[i] / 4;
            blocks = blocks > (set.n4[i] + 255) / 256 ? blocks : (set.n4[i] + 255) / 256;
        }
        add_k_planes_kernel<<<dim3((unsigned)blocks, (unsigned)c.n_mats), 256, 0, stream>>>(set, k_splits);
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace

// Returns 1 when the activations' packing buffer cannot be provided (the stream is being captured and the buffer is
// too small, or the allocation fails): the caller then uses another kernel.
int m40_launch_gemm_tiled_fused(M40llmCudaContext* ctx, hipStream_t stream, uint32_t stream_kind, int source_kind, const float* A,
                                const float* A2, const void* norm_w, uint32_t norm_dtype, float eps, int M, int K, int n_mats,
                                const uint16_t* const* B, const int* N, float* const* C, const float* const* R, bool pair) {
    if (!ctx || stream_kind > 1u) return -2;
    const TiledCall c{source_kind, {A, A2, norm_w, norm_dtype, eps, nullptr, nullptr, nullptr, 0}, M, K, n_mats, B, N, C, R, pair};
    TiledPlan plan;
    int rc = plan_tiled(ctx, c, plan);
    if (rc == 0) rc = provide_pack(ctx->scratch[stream_kind], stream, plan.need);
    return rc != 0 ? rc : enqueue_tiled(ctx->scratch[stream_kind], stream, c, plan, nullptr);
}

// C0 = R0 + A . B0, then the products of RMSNorm(C0): where the first product is cut into parts of K, the pass that norms and packs C0 adds them up (a
// launch and a pass over C0 less: 3.5 us at 101 rows, 4.7 us at 250, 6.5 us at 522 rows of 2048 columns).  The parts lie behind the first
// product's packed rows, K0 >= K1 columns of them, so the second product's packed rows do not reach them.
int m40_launch_gemm_tiled_chain(M40llmCudaContext* ctx, hipStream_t stream, uint32_t stream_kind, const float* A, int M, int K0, const uint16_t* B0, int N0,
                                const float* R0, float* C0, const void* norm_w, uint32_t norm_dtype, float eps, int n_mats, const uint16_t* const* B,
                                const int* N, float* const* C, bool pair, int (*produce)(void*, const M40TiledRows&), void* produce_arg) {
    if (!ctx || stream_kind > 1u) return -2;
    float* const C_first[1] = {C0};
    const float* const R_first[1] = {R0};
    const TiledCall first{produce ? kPackDone : kPackPlain, {produce ? nullptr : A, nullptr, nullptr, 0u, 0.0f, nullptr, nullptr, nullptr, 0}, M, K0, 1, &B0, &N0, C_first, R_first, false};
    TiledCall second{kPackNorm, {C0, nullptr, norm_w, norm_dtype, eps, nullptr, nullptr, nullptr, 0}, M, N0, n_mats, B, N, C, nullptr, pair};
    TiledPlan plan0, plan1;
    int rc = plan_tiled(ctx, first, plan0);
    if (rc == 0) rc = plan_tiled(ctx, second, plan1);
    if (rc == 0) rc = provide_pack(ctx->scratch[stream_kind], stream, plan0.need > plan1.need ? plan0.need : plan1.need);
    if (rc != 0) return rc;
    if (produce) {
        _Float16* hi = static_cast<_Float16*>(ctx->scratch[stream_kind].tiled_pack);
        rc = produce(produce_arg, {hi, hi + (size_t)padded_rows(M) * K0, reinterpret_cast<float*>(hi + 2 * (size_t)padded_rows(M) * K0)});
        if (rc != 0) return rc;
    }
    rc = enqueue_tiled(ctx->scratch[stream_kind], stream, first, plan0, K0 >= N0 ? &second.source : nullptr);
    return rc != 0 ? rc : enqueue_tiled(ctx->scratch[stream_kind], stream, second, plan1, nullptr);
}

int m40_launch_gemm_tiled_multi(M40llmCudaContext* ctx, hipStream_t stream, uint32_t stream_kind, const float* A, int M, int K,
                                int n_mats, const uint16_t* const* B, const int* N, float* const* C) {
    return m40_launch_gemm_tiled_fused(ctx, stream, stream_kind, kPackPlain, A, nullptr, nullptr, 0u, 0.0f, M, K, n_mats, B, N, C, nullptr, false);
}

int m40_launch_gemm_tiled(M40llmCudaContext* ctx, hipStream_t stream, uint32_t stream_kind, const float* A, const uint16_t* B,
                          float* C, int M, int N, int K) {
    return m40_launch_gemm_tiled_multi(ctx, stream, stream_kind, A, M, K, 1, &B, &N, &C);
}
