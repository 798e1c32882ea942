// Packed variable-length causal prefill attention for gfx950, f32 in and out (the step before decode).
//
// Q and Out are [total_q][q_heads][hd], K and V [total_kv][kv_heads][hd]; sequence b owns q_lens[b] query tokens from
// q_offsets[b] and kv_lens[b] keys from kv_offsets[b]; query q_idx attends keys 0 .. kv_len - q_len + q_idx.
//
// The reference walks every key once per (query, head) with one workgroup each (cuda/kernels.cu:3749-3835).  Here a
// workgroup owns 64 or 128 consecutive queries of one q head (four waves x one or two blocks of 16 queries) and streams
// the sequence's keys in tiles of 32 or 64 through LDS, so a key row is fetched once per 64 / 128 queries.  Both products run on v_mfma_f32_16x16x32_f16
// with every f32 operand split exactly into an f16 high and an f16 low part (x = hi + lo to 2^-22): a product is
// three instructions, hi hi + lo hi + hi lo (the lo lo term is below 2^-22 of the operands' magnitudes), which is
// five times the rate of the f32 matrix instruction for the same product at f32-level accuracy:
//   scores  S[query][key] = sum_d Q[query][d] K[key][d]   A = Q (two f16 parts, in registers for the whole kernel),
//           B = K tile (two f16 planes in LDS)
//   output  O[query][d]  += sum_key P[query][key] V[key][d]
// Both are formed transposed (S^T = K Q^T, O^T = V^T P^T) with the tile's keys ordered along the second product's k
// dimension the way the first product's accumulators hold them, so the softmax weights go from one matrix instruction
// into the next inside the lane (no LDS round trip), and maximum, sum and rescaling factor are one value per lane.
// V is stored transposed [d][key slot] so that a lane's eight key slots are one 16-byte read.
// The softmax is online, with a reference point per query in place of the running maximum: weights are
// exp2(x - n) with n within 8 (log2 units) of the largest score so far, moved only when a tile holds a larger one
// (the rows of a lane's accumulators are the same four queries in both products, so the rescaling needs no exchange).
// The result is the same softmax as the reference's three passes (p = exp(s - max) / sum), within f32 rounding.
// Two waves share a SIMD; a wave raises its priority for its matrix-instruction phases, so that the matrix pipe is
// fed first and the other wave's vector work (exponentials, splits) fills the issue slots in between
// (0.283 -> 0.252 ms for one 4096-token sequence at head_dim 64).  Operands beyond the f16 range (|x| > 65504) are not supported by the
// split (none occur after RMSNorm-scaled projections; the decode-side attention has no such limit).
//
// Reference: kernel cuda/kernels.cu:3749-3835; entry points, argument checks and their codes :4834-4977
// (lengths are read back to the host and validated before the launch, also in the _async form).
#include "common.hpp"

#include <type_traits>
#include <vector>

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = 4;
// 16-query blocks per wave: a K / V fragment read from LDS serves every block of the wave.  Two blocks where long
// sequences alone fill the chip four workgroups deep, one otherwise -- two blocks halve the workgroup count and double
// the masked share of a short sequence's diagonal tiles.  One against two blocks, head_dim 128 at 16 / 32 q heads:
// 1 x 4096 tokens 0.30 / 0.33 and 0.63 / 0.53 ms, 4 x 4096 1.17 / 1.02 and 2.13 / 1.85 ms, 16 x 300 0.069 / 0.077 and
// 0.099 / 0.112 ms; head_dim 64 at 32 q heads: 1 x 1024 48 / 52 us, 1 x 2048 94 / 102 us, 16 x 300 59 / 69 us,
// 1 x 4096 0.260 / 0.240 ms, 2 x 4096 0.58 / 0.51 ms.
constexpr float kRefSlack = 8.0f;          // log2 units: weights stay below 256
constexpr uint32_t kTwoBlockMinQueries = 2048;      // a sequence counts as long from here
constexpr int kTwoBlockMinGroupsPerCu = 4;
// keys per LDS tile (KT below): one or two k-steps of the P . V product; 64 where two planes of K and V^T fit the
// static LDS limit (head_dim 64), 32 otherwise
constexpr int key_tile_of(int hd) { return hd == 64 ? 64 : 32; }

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ m40_float4 mfma32(half8 a, half8 b, m40_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// Issue order of a phase of STEPS steps, each two 16-byte LDS fragment reads and PER matrix instructions that use them:
// the reads run AHEAD steps in front of their instructions (left to itself the compiler reuses one register pair and
// waits for every read right after issuing it).
template <int STEPS, int PER, int AHEAD = 1>
__device__ __forceinline__ void fragment_pipeline() {
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * (AHEAD < STEPS ? AHEAD : STEPS), 0);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        if (i + AHEAD < STEPS) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
    }
}
// The rotated value itself goes into the split: without this the compiler folds rotation and conversion into one multiply-add rounded to f16 (m40_f2h)
__device__ __forceinline__ void rounded(float& x) { asm volatile("" : "+v"(x)); }
// x = hi + lo with both parts f16: exact to about 2^-22 relative for values inside the f16 range
__device__ __forceinline__ void split(float x, _Float16* hi, _Float16* lo) {
    const _Float16 h = static_cast<_Float16>(x);
    *hi = h;
    *lo = static_cast<_Float16>(x - static_cast<float>(h));
}

struct PrefillArgs {
    const float* Q; const float* K; const float* V; float* Out;
    const _Float16* planes;     // per padded 32-key tile and kv head: K hi [32][HD], K lo, V^T hi [HD][32], V^T lo
    uint32_t plane_tiles;       // padded tiles in total (sequence b starts at tile kv_offsets[b] / 32 + b ... see pack)
    const uint32_t* q_offsets; const uint32_t* kv_offsets; const uint32_t* q_lens; const uint32_t* kv_lens;
    uint32_t q_heads, kv_heads;
    float *v_max, *v_key;       // per padded tile and kv head: largest finite |V|, of the tile and of each of its keys (with a PrefillRope)
    M40TiledRows rows;          // where the result goes as rows of the next product instead of Out
};

// Prompts that go in unrotated: rows 0 .. of sequence b are its positions 0 ..; queries are rotated where they are loaded, keys where they are
// packed, which also appends them to the dense cache.
struct PrefillRope {
    const float2* angles;       // [rows of the sequences one behind the other][HD / 2] (cos, sin)
    const float *bq, *bk, *bv;  // added before the rotation, or null
    uint32_t layout, max_seq_len;
    uint16_t *k_cache, *v_cache;
    uint32_t* seq_map;
    uint32_t slot[kM40PrefillSeqs];
    uint32_t first[kM40PrefillSeqs];      // row of the angles of a sequence's first row; its rows may lie further on, the offsets may have gaps
};
struct NoRope {};

// Order of a tile's 32 keys along the k dimension of the P . V product: k-slot 8 g + i holds key 4 g + i (i < 4) or
// key 16 + 4 g + (i - 4): exactly the eight keys whose scores lane group g holds after the two score products, so the
// weights go from the score accumulators into the next product's operand without leaving the lane.
__device__ __forceinline__ int key_of_slot(int slot) {
    const int base = slot & ~31, g = (slot & 31) >> 3, i = slot & 7;      // every 32 slots: one k-step over 32 keys
    return base + (i < 4 ? 4 * g + i : 16 + 4 * g + (i - 4));
}

// First padded tile of sequence b in the packed planes: every sequence starts on a tile boundary of its own, so a
// sequence gets one tile of slack (rows_before / 32 rounded down, plus b).
__device__ __forceinline__ uint32_t first_tile_of(uint32_t kv_offset, uint32_t b, uint32_t key_tile) { return kv_offset / key_tile + b; }

// K and V of one 32-key tile and kv head -> two f16 planes each, V transposed, in the order the attention kernel copies
// them to LDS.  Done once per call so that the 64-query workgroups (and the q heads of a group) do not each repeat the
// split.  Keys past the sequence end are written as zeros (they are masked anyway).
// With a PrefillRope the keys are rotated here and both go to the cache as well: the pass that rotated Q and K in place and appended K and V was a
// launch of its own that read and wrote all of Q (4096 rows, 32 + 4 heads of 64: 21.2 us and 5.7 for the packing; one launch).  A thread holds
// quads of columns that rotate with each other.
template <int HD, class ROPE>
__global__ __launch_bounds__(kThreads) void prefill_pack_kv_kernel(PrefillArgs p, ROPE rope) {
    constexpr bool kRope = std::is_same<ROPE, PrefillRope>::value;
    constexpr int kKTile = key_tile_of(HD);
    __shared__ float vt[kKTile][HD + 1];
    __shared__ float wave_max[kWaves];
    const uint32_t b = blockIdx.z, kvh = blockIdx.y, tile = blockIdx.x;
    const uint32_t kv_len = p.kv_lens[b];
    if (tile * kKTile >= kv_len) return;
    const float* Kb = p.K + ((size_t)p.kv_offsets[b] * p.kv_heads + kvh) * HD;
    const float* Vb = p.V + ((size_t)p.kv_offsets[b] * p.kv_heads + kvh) * HD;
    const size_t row_stride = (size_t)p.kv_heads * HD;
    _Float16* out = const_cast<_Float16*>(p.planes) + ((size_t)(first_tile_of(p.kv_offsets[b], b, kKTile) + tile) * p.kv_heads + kvh) * (4 * kKTile * HD);
    _Float16* kh = out, *kl = out + kKTile * HD, *vh = out + 2 * kKTile * HD, *vl = out + 3 * kKTile * HD;
    // All of a thread's elements are requested together, four a load where K and V are aligned for it, and stored four and eight at a time: a tile
    // is one round trip, not one per element (60 tiles of 64 keys x 64: 9.9 us one by one, 4.7 us now)
    constexpr int kQuads = kKTile * HD / 4 / kThreads, kHalf = HD / 2;
    static_assert(kQuads % 2 == 0, "quads come in pairs");
    // where quad u of the thread lies in the tile: quads 2 i and 2 i + 1 hold columns that rotate with each other
    int at[kQuads];
    bool neox = true;
    if constexpr (kRope) neox = rope.layout == M40LLM_ROPE_LAYOUT_NEOX;
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
        const int pair = (int)threadIdx.x + u / 2 * kThreads, key_in = pair / (HD / 8), c = pair % (HD / 8);
        at[u] = kRope ? key_in * HD + (neox ? 4 * c + u % 2 * kHalf : 8 * c + 4 * (u % 2)) : ((int)threadIdx.x + u * kThreads) * 4;
    }
    float4 kx[kQuads], vx[kQuads], cs[kRope ? kQuads : 1];
    auto load = [&](auto quad) {
#pragma unroll
        for (int u = 0; u < kQuads; ++u) {
            const int key_in = at[u] / HD, d = at[u] % HD;
            const uint32_t key = tile * kKTile + key_in, row = key < kv_len ? key : kv_len - 1;
            // the four angles of a pair of quads, two by each
            if constexpr (kRope) {
                const int off = (neox ? at[u & ~1] : at[u & ~1] / 2) % kHalf + 2 * (u % 2);
                cs[u] = *reinterpret_cast<const float4*>(rope.angles + ((size_t)rope.first[b] + row) * kHalf + off);
            }
            kx[u] = quad(Kb + (size_t)row * row_stride + d);
            vx[u] = quad(Vb + (size_t)row * row_stride + d);
        }
    };
    if (m40_aligned16(Kb) && m40_aligned16(Vb)) load([](const float* x) { return *reinterpret_cast<const float4*>(x); });
    else load([](const float* x) { return make_float4(x[0], x[1], x[2], x[3]); });
    if constexpr (kRope) {
        auto add = [](float4& x, const float* bias) { x = make_float4(x.x + bias[0], x.y + bias[1], x.z + bias[2], x.w + bias[3]); };
#pragma unroll
        for (int u = 0; u < kQuads; ++u) {
            const int d = at[u] % HD;
            if (rope.bk) add(kx[u], rope.bk + kvh * HD + d);
            if (rope.bv) add(vx[u], rope.bv + kvh * HD + d);
        }
        const size_t slot_row = (size_t)rope.slot[b] * rope.max_seq_len;
#pragma unroll
        for (int u = 0; u < kQuads; u += 2) {
            float4 &x = kx[u], &y = kx[u + 1];
            const float4 c0 = cs[u], c1 = cs[u + 1];
            if (neox) {
                m40_rope_apply(make_float2(c0.x, c0.y), x.x, y.x, &x.x, &y.x);
                m40_rope_apply(make_float2(c0.z, c0.w), x.y, y.y, &x.y, &y.y);
                m40_rope_apply(make_float2(c1.x, c1.y), x.z, y.z, &x.z, &y.z);
                m40_rope_apply(make_float2(c1.z, c1.w), x.w, y.w, &x.w, &y.w);
            } else {
                m40_rope_apply(make_float2(c0.x, c0.y), x.x, x.y, &x.x, &x.y);
                m40_rope_apply(make_float2(c0.z, c0.w), x.z, x.w, &x.z, &x.w);
                m40_rope_apply(make_float2(c1.x, c1.y), y.x, y.y, &y.x, &y.y);
                m40_rope_apply(make_float2(c1.z, c1.w), y.z, y.w, &y.z, &y.w);
            }
            rounded(x.x); rounded(x.y); rounded(x.z); rounded(x.w);
            rounded(y.x); rounded(y.y); rounded(y.z); rounded(y.w);
        }
#pragma unroll
        for (int u = 0; u < kQuads; ++u) {
            const uint32_t key = tile * kKTile + at[u] / HD;
            if (key >= kv_len) continue;
            const size_t to = (slot_row + key) * row_stride + (size_t)kvh * HD + at[u] % HD;
            *reinterpret_cast<ushort4*>(rope.k_cache + to) = make_ushort4(m40_f2h(kx[u].x), m40_f2h(kx[u].y), m40_f2h(kx[u].z), m40_f2h(kx[u].w));
            *reinterpret_cast<ushort4*>(rope.v_cache + to) = make_ushort4(m40_f2h(vx[u].x), m40_f2h(vx[u].y), m40_f2h(vx[u].z), m40_f2h(vx[u].w));
        }
        if (tile == 0 && kvh == 0 && threadIdx.x == 0) rope.seq_map[rope.slot[b]] = kv_len;
        float mx = 0.0f;
        float* const v_key = p.v_key + ((size_t)(first_tile_of(p.kv_offsets[b], b, kKTile) + tile) * p.kv_heads + kvh) * kKTile;
#pragma unroll
        for (int u = 0; u < kQuads; u += 2) {
            const float v8[8] = {vx[u].x, vx[u].y, vx[u].z, vx[u].w, vx[u + 1].x, vx[u + 1].y, vx[u + 1].z, vx[u + 1].w};
            float of_key = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) of_key = fmaxf(of_key, fabsf(v8[i]) <= 3.402823466e+38f ? fabsf(v8[i]) : 0.0f);      // (keys past the end: the last one's again)
            // HD / 8 neighbouring lanes hold a key
            of_key = fmaxf(of_key, m40_dpp_f<M40_DPP_XOR1>(of_key));
            of_key = fmaxf(of_key, m40_dpp_f<M40_DPP_XOR2>(of_key));
            of_key = fmaxf(of_key, m40_dpp_f<M40_DPP_HALF_MIRROR>(of_key));
            if (HD == 128) of_key = fmaxf(of_key, m40_dpp_f<M40_DPP_ROW_ROR8>(of_key));
            if (threadIdx.x % (HD / 8) == 0) v_key[at[u] / HD] = of_key;
            mx = fmaxf(mx, of_key);
        }
        mx = m40_max64(mx);
        if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = mx;
    }
#pragma unroll
    for (int u = 0; u < kQuads; ++u) {
        const int e = at[u], key_in = e / HD, d = e % HD;
        const bool live = tile * kKTile + key_in < kv_len;
        const float k4[4] = {kx[u].x, kx[u].y, kx[u].z, kx[u].w}, v4[4] = {vx[u].x, vx[u].y, vx[u].z, vx[u].w};
        half4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            _Float16 a, c;
            split(live ? k4[i] : 0.0f, &a, &c);
            hi[i] = a;
            lo[i] = c;
            vt[key_in][d + i] = live ? v4[i] : 0.0f;
        }
        *reinterpret_cast<half4*>(kh + e) = hi;
        *reinterpret_cast<half4*>(kl + e) = lo;
    }
    __syncthreads();
    if constexpr (kRope) {
        if (threadIdx.x == 0) p.v_max[(size_t)(first_tile_of(p.kv_offsets[b], b, kKTile) + tile) * p.kv_heads + kvh] = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
    }
#pragma unroll
    for (int u = 0; u < kKTile * HD / 8 / kThreads; ++u) {
        const int e = ((int)threadIdx.x + u * kThreads) * 8, d = e / kKTile, slot = e % kKTile;
        half8 hi, lo;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            _Float16 a, c;
            split(vt[key_of_slot(slot + i)][d], &a, &c);
            hi[i] = a;
            lo[i] = c;
        }
        *reinterpret_cast<half8*>(vh + e) = hi;
        *reinterpret_cast<half8*>(vl + e) = lo;
    }
}

// QB: 16-query blocks per wave.  With two, every K and V fragment a wave reads from LDS serves 32 queries instead of 16:
// the kernel's LDS traffic (each wave reads the whole K and V tile) was what it spent most of its time on.
// PLANES (with a PrefillRope): the result goes to the rows of the next product, which a packing pass read and wrote again (4096 rows of 2048 12.9 us, 522 rows
// 6.0).  A row's scale must be known to the workgroups of all its heads: it follows from the largest |V| of the keys that the row sees, which no weighted mean of
// those exceeds, brought into [2^14, 2^15): f16 hi + lo keep 22 bits of every value down to 2^-17 of it, and no row depends on what comes behind it (the largest of the
// whole sequence instead took bits from the rows ahead of a large V; a whole prompt of 4096 tokens 21.18 ms
// so, 21.25 now, five of 522 together 4.66 and 4.69, inside their spread).  Below, an error of
// 2^-39 of the largest: for |V| up to 2^14 within the 2^-25 that V's own two parts leave.  A value that is not finite goes in as it is.
template <int HD, int QB, class ROPE, bool PLANES>
__global__ __launch_bounds__(kThreads) void prefill_attn_kernel(PrefillArgs p, ROPE rope) {
    constexpr bool kRope = std::is_same<ROPE, PrefillRope>::value;
    constexpr int kKTile = key_tile_of(HD);
    constexpr int KB = kKTile / 16;        // 16-key score blocks of a tile
    constexpr int KS = HD / 32;            // matrix-instruction k-steps of a score tile
    constexpr int DT = HD / 16;            // 16-column output tiles
    constexpr int KSTR = HD + 8;           // LDS halves per K row: 16-byte fragment reads of 16 keys hit 64 distinct banks
    constexpr int VSTR = kKTile + 8;       // LDS halves per row of the transposed V tile [column][key]
    constexpr int kQWave = 16 * QB;        // queries of a wave
    constexpr int kQGroup = kQWave * kWaves;
    // Two forms of the tile body, by measurement (one 4096-token sequence at 32 heads / eight sequences at 16 heads):
    // head_dim 64 skips a first block that a tile lies wholly behind (branches around its matrix instructions) and
    // leaves the order of fragment reads and matrix instructions to the compiler; head_dim 128 computes such a block
    // masked and orders reads one step ahead of their instructions.  The other way round costs 5-6 % at either size.
    constexpr bool kSkip = QB > 1 && HD == 64, kPipe = HD == 128;
    __shared__ __attribute__((aligned(16))) _Float16 k_lds[2][kKTile * KSTR];   // [hi, lo][key][d]
    __shared__ __attribute__((aligned(16))) _Float16 v_lds[2][HD * VSTR];       // [hi, lo][d][key]

    // Workgroups are dispatched in index order, x fastest: x = q head, y = query tile from the end of the sequence,
    // z = sequence (ordering the tiles of all sequences together by key count measured slower: the sequences' keys
    // then compete for the caches).
    // The tiles with the most keys (the longest workgroups) of every head start first and the short ones fill the
    // tail; with the head as the slow index the last heads' long tiles started near the end of the kernel and the
    // chip ran at a third of its occupancy.  Neighbouring workgroups are the q heads of one kv group on the same keys.
    const uint32_t b = blockIdx.z, h = blockIdx.x;
    const uint32_t q_len = p.q_lens[b], kv_len = p.kv_lens[b];
    const uint32_t q0 = (gridDim.y - 1u - blockIdx.y) * kQGroup;
    if (q0 >= q_len || q_len > kv_len) return;
    const uint32_t kvh = h / (p.q_heads / p.kv_heads);
    const int tid = threadIdx.x, lane = tid & 63;
    // PLANES: the largest |V| of the keys ahead of the workgroup's queries, by tiles, and of the queries' own, a few heads a thread; the rest is looked at at the end
    const uint32_t n_ahead = q0 / kKTile * p.kv_heads, own_key = q0 + (uint32_t)(tid % kQGroup) < q_len ? q0 + (uint32_t)(tid % kQGroup) : q_len - 1;
    const size_t first_max = PLANES ? (size_t)first_tile_of(p.kv_offsets[b], b, kKTile) * p.kv_heads : 0;
    const float* v_key = PLANES ? p.v_key + (first_max + own_key / kKTile * p.kv_heads) * kKTile + own_key % kKTile : nullptr;
    float ahead = PLANES && (uint32_t)tid < n_ahead ? p.v_max[first_max + tid] : 0.0f;
    float own = PLANES && (uint32_t)(tid / kQGroup) < p.kv_heads ? v_key[tid / kQGroup * kKTile] : 0.0f;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);       // as a scalar: tests on it branch without masks
    const int j = lane & 15, g = lane >> 4;
    const float inv_sqrt = HD == 64 ? 0.125f : 0.08838834764831845f;
    const uint32_t shift = kv_len - q_len;                        // query q attends keys 0 .. shift + q
    const uint32_t wg_last_q = q0 + kQGroup - 1 < q_len - 1 ? q0 + kQGroup - 1 : q_len - 1;
    const uint32_t n_tiles = (shift + wg_last_q) / kKTile + 1;    // key tiles this workgroup walks

    // ---- this wave's query blocks: A operand of the score product, lane (query j, k group g) of block qb holds
    //      Q[j][32 s + 8 g .. + 7] as a high and a low f16 part
    const uint32_t wq0 = q0 + (uint32_t)kQWave * wave;            // first query of the wave
    const bool wave_live = wq0 < q_len;
    uint32_t row_end[QB];                                         // last key this lane's query of the block sees
    uint32_t blk_end[QB];                                         // last key any query of the block sees
    half8 qh[QB][KS], ql[QB][KS];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        const uint32_t bq0 = wq0 + 16u * qb;
        const uint32_t my_q = bq0 + j < q_len ? bq0 + j : q_len - 1;      // a query past the end repeats the last one (not stored)
        row_end[qb] = shift + my_q;
        blk_end[qb] = shift + (bq0 + 15u < q_len ? bq0 + 15u : q_len - 1);
        const float* qp = p.Q + ((size_t)(p.q_offsets[b] + my_q) * p.q_heads + h) * HD + 8 * g;
        float x[KS][8];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const float4 x0 = *reinterpret_cast<const float4*>(qp + 32 * s), x1 = *reinterpret_cast<const float4*>(qp + 32 * s + 4);
            x[s][0] = x0.x; x[s][1] = x0.y; x[s][2] = x0.z; x[s][3] = x0.w; x[s][4] = x1.x; x[s][5] = x1.y; x[s][6] = x1.z; x[s][7] = x1.w;
        }
        if constexpr (kRope) {
            // a lane holds both columns of its pairs: neighbours, or 32 s + 8 g + i and half a head further on
            constexpr int kHalf = HD / 2, HS = KS / 2;
            const bool neox = rope.layout == M40LLM_ROPE_LAYOUT_NEOX;
            const float2* angles = rope.angles + ((size_t)rope.first[b] + my_q) * kHalf + (neox ? 8 * g : 4 * g);
            float4 cs[HS][4];
#pragma unroll
            for (int s = 0; s < HS; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i)      // layout of neighbours: two angles of step s, two of step s + HS at a time
                    cs[s][i] = *reinterpret_cast<const float4*>(angles + (neox ? 32 * s + 2 * i : 16 * (s + HS * (i >> 1)) + 2 * (i & 1)));
            if (rope.bq) {
#pragma unroll
                for (int s = 0; s < KS; ++s)
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[s][i] += rope.bq[(size_t)h * HD + 32 * s + 8 * g + i];
            }
#pragma unroll
            for (int s = 0; s < HS; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float2 c0 = make_float2(cs[s][i].x, cs[s][i].y), c1 = make_float2(cs[s][i].z, cs[s][i].w);
                    if (neox) {
                        m40_rope_apply(c0, x[s][2 * i], x[s + HS][2 * i], &x[s][2 * i], &x[s + HS][2 * i]);
                        m40_rope_apply(c1, x[s][2 * i + 1], x[s + HS][2 * i + 1], &x[s][2 * i + 1], &x[s + HS][2 * i + 1]);
                    } else {
                        float(&y)[8] = x[s + HS * (i >> 1)];
                        m40_rope_apply(c0, y[4 * (i & 1)], y[4 * (i & 1) + 1], &y[4 * (i & 1)], &y[4 * (i & 1) + 1]);
                        m40_rope_apply(c1, y[4 * (i & 1) + 2], y[4 * (i & 1) + 3], &y[4 * (i & 1) + 2], &y[4 * (i & 1) + 3]);
                    }
                }
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int i = 0; i < 8; ++i) rounded(x[s][i]);
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                _Float16 a, c;
                split(x[s][i], &a, &c);
                qh[qb][s][i] = a;
                ql[qb][s][i] = c;
            }
        }
    }
    const uint32_t wave_first_end = shift + (wq0 < q_len ? wq0 : q_len - 1);          // last key the wave's first query sees
    const uint32_t wave_end = blk_end[QB - 1];                                        // last key any query of the wave sees

    // ---- K / V tile loads: 16-byte pieces of the packed f16 planes (prefill_pack_kv_kernel), straight into LDS
    constexpr int PIECES = kKTile * HD / 8 / kThreads;           // per plane and thread: 1 (HD 64) or 2 (HD 128)
    const _Float16* tile_base = p.planes + ((size_t)first_tile_of(p.kv_offsets[b], b, kKTile) * p.kv_heads + kvh) * (4 * kKTile * HD);
    const size_t tile_stride = (size_t)p.kv_heads * (4 * kKTile * HD);
    uint4 kreg[2][PIECES], vreg[2][PIECES];
    auto issue = [&](uint32_t tile) {
        const _Float16* t = tile_base + (size_t)tile * tile_stride;
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int c = u * kThreads + tid;
#pragma unroll
            for (int pl = 0; pl < 2; ++pl) {
                kreg[pl][u] = *reinterpret_cast<const uint4*>(t + pl * kKTile * HD + 8 * c);
                vreg[pl][u] = *reinterpret_cast<const uint4*>(t + (2 + pl) * kKTile * HD + 8 * c);
            }
        }
    };
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    auto to_lds = [&]() {
#pragma unroll
        for (int u = 0; u < PIECES; ++u) {
            const int c = u * kThreads + tid;
            const int key_in = c / (HD / 8), kpart = c % (HD / 8);     // K plane [key][HD]
            const int d = c / (kKTile / 8), vpart = c % (kKTile / 8);  // V^T plane [d][32 keys]
#pragma unroll
            for (int pl = 0; pl < 2; ++pl) {
                *reinterpret_cast<u32x4*>(&k_lds[pl][key_in * KSTR + 8 * kpart]) = u32x4{kreg[pl][u].x, kreg[pl][u].y, kreg[pl][u].z, kreg[pl][u].w};
                *reinterpret_cast<u32x4*>(&v_lds[pl][d * VSTR + 8 * vpart]) = u32x4{vreg[pl][u].x, vreg[pl][u].y, vreg[pl][u].z, vreg[pl][u].w};
            }
        }
    };
    issue(0);

    // Products are formed transposed, S^T = K Q^T and O^T = V^T P^T, so that a lane (query j, group g) ends up with the
    // scores of ONE query for keys 4 g .. 4 g + 3 of both 16-key blocks, which are the k-slots 8 g .. 8 g + 7 of the
    // second product (key_of_slot): the weights never pass through LDS, and the running maximum, the sum and the
    // rescaling factor are one value per lane and query block.
    float m_run[QB], l_run[QB];              // maximum over the query's keys so far (equal in its four lanes); this lane's share of the sum
    m40_float4 O[QB][DT];                    // O^T[16 d + 4 g + r][query j] of the block
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        m_run[qb] = -INFINITY;
        l_run[qb] = 0.0f;
#pragma unroll
        for (int d = 0; d < DT; ++d) O[qb][d] = m40_float4{0.f, 0.f, 0.f, 0.f};
    }
    const float scale_log2 = inv_sqrt * 1.4426950408889634f;     // scores in units of log2: weights are exp2(x - max)

    for (uint32_t tile = 0; tile < n_tiles; ++tile) {
        __syncthreads();                  // the previous tile has been read by every wave
        to_lds();
        __syncthreads();
        if (tile + 1 < n_tiles) issue(tile + 1);
        const uint32_t key0 = tile * kKTile;
        if (!wave_live || key0 > wave_end) continue;              // nothing of this tile is visible to the wave
        // a block whose queries all end before this tile (only the first can: later queries see more, and at most one
        // tile per wave).  Computing it all the same changes nothing: every score is masked, and the weights are
        // exp2(-inf - m) = 0 with the finite reference point that tile 0 has left (key 0 is visible to every query).
        bool blk_on[QB];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) blk_on[qb] = !kSkip || key0 <= blk_end[qb];
        // S^T of the tile's 16-key blocks: lane (query j, g) gets keys 16 kb + 4 g + r.  k . q = kh qh + kh ql + kl qh
        // (the kl ql term is below 2^-22 of |q| |k|); a K fragment read serves every query block of the wave
        m40_float4 sc[QB][KB];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) sc[qb][kb] = m40_float4{0.f, 0.f, 0.f, 0.f};
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int off = 32 * s + 8 * g;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const half8 kh = *reinterpret_cast<const half8*>(&k_lds[0][(16 * kb + j) * KSTR + off]);
                const half8 kl = *reinterpret_cast<const half8*>(&k_lds[1][(16 * kb + j) * KSTR + off]);
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) {
                    if (kSkip && !blk_on[qb]) continue;
                    sc[qb][kb] = mfma32(kh, qh[qb][s], sc[qb][kb]);
                    sc[qb][kb] = mfma32(kh, ql[qb][s], sc[qb][kb]);
                    sc[qb][kb] = mfma32(kl, qh[qb][s], sc[qb][kb]);
                }
            }
        }
        if (kPipe) fragment_pipeline<KS * KB, 3 * QB>();
        __builtin_amdgcn_s_setprio(0);
        const bool whole = key0 + (uint32_t)kKTile - 1u <= wave_first_end;      // every key of the tile visible to every query
        half8 ph[QB][KB / 2], pl[QB][KB / 2];       // k-step t: slots 8 g + i = blocks 2 t (i < 4) and 2 t + 1 (i >= 4)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            if (kSkip && !blk_on[qb]) continue;
            float x[4 * KB];
            float mx = -INFINITY;
            if (whole) {                      // the usual tile (a uniform branch): no per-key comparison
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        x[4 * kb + r] = sc[qb][kb][r] * scale_log2;
                        mx = fmaxf(mx, x[4 * kb + r]);
                    }
            } else {
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const bool visible = key0 + 16u * kb + 4u * g + r <= row_end[qb];
                        x[4 * kb + r] = visible ? sc[qb][kb][r] * scale_log2 : -INFINITY;
                        mx = fmaxf(mx, x[4 * kb + r]);
                    }
            }
            // The weights are exp2(x - n) for a reference point n per query that need not be the maximum: any n within
            // kRefSlack of it keeps the weights below 2^kRefSlack, far inside the range of the f16 split, and the softmax
            // is the same.  The reference point moves (cross-lane maximum, rescaling of the sum and the accumulators)
            // only when some lane of the wave sees a score more than kRefSlack above its query's: after the first tiles
            // of a sequence that is rare, and the usual tile has no cross-lane exchange between its two products.
            float n = m_run[qb];
            if (__any(mx > n + kRefSlack)) {
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                mx = fmaxf(mx, __shfl_xor(mx, 32));
                n = fmaxf(n, mx);
                // no reference point yet: the old state weighs nothing
                const float f = m_run[qb] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run[qb] - n);
                l_run[qb] *= f;
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int r = 0; r < 4; ++r) O[qb][d][r] *= f;
                m_run[qb] = n;
            }
            float psum = 0.0f;
#pragma unroll
            for (int i = 0; i < 4 * KB; i += 2) {
                // two weights at a time: the packed f32 -> f16 conversion of gfx950 halves the conversion instructions
                const f32x2 pv = {__builtin_amdgcn_exp2f(x[i] - n), __builtin_amdgcn_exp2f(x[i + 1] - n)};   // a masked key: exp2(-inf) = 0
                psum += pv.x + pv.y;
                const half2v a = __builtin_convertvector(pv, half2v);
                const half2v c = __builtin_convertvector(pv - __builtin_convertvector(a, f32x2), half2v);
                ph[qb][i >> 3][i & 7] = a.x; ph[qb][i >> 3][(i & 7) + 1] = a.y;
                pl[qb][i >> 3][i & 7] = c.x; pl[qb][i >> 3][(i & 7) + 1] = c.y;
            }
            l_run[qb] += psum;
        }
        // O^T += V^T . P^T, 32 keys per k-step: A = V^T[column 16 d + j][k-slots 32 t + 8 g .. + 7], B = this lane's
        // eight weights of the step;  v p = vh ph + vh pl + vl ph; a V fragment read serves every query block
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
#pragma unroll
            for (int t = 0; t < KB / 2; ++t) {
                const half8 vh = *reinterpret_cast<const half8*>(&v_lds[0][(16 * d + j) * VSTR + 32 * t + 8 * g]);
                const half8 vl = *reinterpret_cast<const half8*>(&v_lds[1][(16 * d + j) * VSTR + 32 * t + 8 * g]);
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) {
                    if (kSkip && !blk_on[qb]) continue;
                    O[qb][d] = mfma32(vh, ph[qb][t], O[qb][d]);
                    O[qb][d] = mfma32(vh, pl[qb][t], O[qb][d]);
                    O[qb][d] = mfma32(vl, ph[qb][t], O[qb][d]);
                }
            }
        }
        if (kPipe) fragment_pipeline<DT * (KB / 2), 3 * QB>();
        __builtin_amdgcn_s_setprio(0);
    }

    // ---- out = O / sum: this lane holds columns 16 d + 4 g .. + 3 of its query
    float seen = 0.0f;                 // of the wave's sixty-four queries that hold its own: largest |V| of the keys up to query `lane`
    if constexpr (PLANES) {
        __shared__ float wave_max[kWaves], own_max[kThreads];
        for (uint32_t i = tid + kThreads; i < n_ahead; i += kThreads) ahead = fmaxf(ahead, p.v_max[first_max + i]);
        for (uint32_t i = tid / kQGroup + kThreads / kQGroup; i < p.kv_heads; i += kThreads / kQGroup) own = fmaxf(own, v_key[i * kKTile]);
        ahead = m40_max64(ahead);
        if (lane == 0) wave_max[wave] = ahead;
        own_max[tid] = own;
        __syncthreads();
        ahead = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
        const auto of_query = [&](int q) {
            float m = own_max[q];
#pragma unroll
            for (int i = kQGroup; i < kThreads; i += kQGroup) m = fmaxf(m, own_max[q + i]);
            return m;
        };
        const int half = kQWave * wave / 64;
        seen = of_query(64 * half + lane);
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const float before = __shfl_up(seen, d, 64);
            if (lane >= d) seen = fmaxf(seen, before);
        }
        if (half) ahead = fmaxf(ahead, m40_max64(of_query(lane)));
        seen = fmaxf(seen, ahead);
    }
    if (!wave_live) return;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        float l = l_run[qb] + __shfl_xor(l_run[qb], 16);
        l += __shfl_xor(l, 32);
        const float denom = l > 0.0f ? l : 1.0f;
        const uint32_t q = wq0 + 16u * qb + (uint32_t)j;
        if constexpr (PLANES) {
            const float bound = __shfl(seen, (kQWave * wave + 16 * qb) % 64 + j, 64);
            if (q >= q_len) continue;
            const int row = (int)(p.q_offsets[b] + q), K = (int)p.q_heads * HD;
            const size_t first = m40_tiled_row(row, K);
            int ex;
            (void)frexpf(bound, &ex);
            ex = bound > 0.0f ? (ex < -85 ? -100 : ex - 15) : 0;
            const float row_inv = __uint_as_float((uint32_t)(127 - ex) << 23);
            if (h == 0 && g == 0) p.rows.scale[row] = __uint_as_float((uint32_t)(127 + ex) << 23);
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                half4 hi, lo;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float y = O[qb][d][r] / denom * row_inv;
                    hi[r] = static_cast<_Float16>(y);
                    lo[r] = fabsf(y) <= 3.402823466e+38f ? static_cast<_Float16>(y - static_cast<float>(hi[r])) : static_cast<_Float16>(0.0f);
                }
                const size_t at = first + m40_tiled_col((int)h * HD + 16 * d + 4 * g);
                *reinterpret_cast<half4*>(p.rows.hi + at) = hi;
                *reinterpret_cast<half4*>(p.rows.lo + at) = lo;
            }
        } else if (q < q_len) {
            float* op = p.Out + ((size_t)(p.q_offsets[b] + q) * p.q_heads + h) * HD + 4 * g;
#pragma unroll
            for (int d = 0; d < DT; ++d)
                *reinterpret_cast<float4*>(op + 16 * d) =
                    make_float4(O[qb][d][0] / denom, O[qb][d][1] / denom, O[qb][d][2] / denom, O[qb][d][3] / denom);
        }
    }
}

int prefill_impl(M40llmCudaContext* ctx, const void* q, const void* k, const void* v, const uint32_t* q_offsets,
                 const uint32_t* kv_offsets, const uint32_t* q_lens, const uint32_t* kv_lens, uint32_t batch,
                 uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim, void* out, bool synchronize,
                 const uint32_t* kv_offsets_host = nullptr, const uint32_t* q_lens_host = nullptr,
                 const uint32_t* kv_lens_host = nullptr, const PrefillRope* rope = nullptr, const M40TiledRows* rows = nullptr) {
    if (!ctx || !q || !k || !v || !q_offsets || !kv_offsets || !q_lens || !kv_lens || (!out && !rows)) return -1;
    if (batch == 0) return -2;
    if (q_heads == 0 || kv_heads == 0 || q_heads % kv_heads != 0) return -3;
    if (head_dim != 64 && head_dim != 128) return -9;
    // the lengths are validated on the host before the launch, as the reference does (also in the _async form); a caller
    // that holds the tables on the host passes them and spares the three blocking read-backs (each one drains the device)
    const bool host_tables = kv_offsets_host && q_lens_host && kv_lens_host;
    std::vector<uint32_t> host(2 * (size_t)batch);
    if (host_tables) {
        for (uint32_t i = 0; i < batch; ++i) { host[i] = q_lens_host[i]; host[batch + i] = kv_lens_host[i]; }
    } else {
        if (hipMemcpy(host.data(), q_lens, (size_t)batch * sizeof(uint32_t), hipMemcpyDeviceToHost) != hipSuccess) return -7;
        if (hipMemcpy(host.data() + batch, kv_lens, (size_t)batch * sizeof(uint32_t), hipMemcpyDeviceToHost) != hipSuccess) return -7;
    }
    uint32_t max_q = 0, max_kv = 0;
    for (uint32_t i = 0; i < batch; ++i) {
        const uint32_t ql = host[i], kl = host[batch + i];
        if (ql == 0 || kl == 0 || ql > kl || kl > 8192) return -8;
        max_q = ql > max_q ? ql : max_q;
        max_kv = kl > max_kv ? kl : max_kv;
    }
    if (!m40_aligned16(q) || !m40_aligned16(k) || !m40_aligned16(v) || !m40_aligned16(out)) return -4;
    PrefillArgs a{};
    a.Q = static_cast<const float*>(q); a.K = static_cast<const float*>(k); a.V = static_cast<const float*>(v);
    a.Out = static_cast<float*>(out);
    a.q_offsets = q_offsets; a.kv_offsets = kv_offsets; a.q_lens = q_lens; a.kv_lens = kv_lens;
    a.q_heads = q_heads; a.kv_heads = kv_heads;
    // f16 planes of K and V (prefill_pack_kv_kernel) in the prefill stream's buffer, grown on demand.  The packed
    // layout needs the sequences' key ranges to lie one after the other (offsets non-decreasing with the batch index,
    // no overlap), which is how packed batches are built; anything else is refused.
    std::vector<uint32_t> offs(batch);
    if (host_tables) offs.assign(kv_offsets_host, kv_offsets_host + batch);
    else if (hipMemcpy(offs.data(), kv_offsets, (size_t)batch * sizeof(uint32_t), hipMemcpyDeviceToHost) != hipSuccess) return -7;
    uint64_t end_prev = 0;
    for (uint32_t i = 0; i < batch; ++i) {
        if (offs[i] < end_prev) return -8;
        end_prev = (uint64_t)offs[i] + host[batch + i];
    }
    const uint32_t kKTile = (uint32_t)key_tile_of((int)head_dim);
    const uint64_t plane_tiles = (offs[batch - 1] / kKTile + (batch - 1)) + (host[2 * (size_t)batch - 1] + kKTile - 1) / kKTile;
    const size_t planes_bytes = (size_t)plane_tiles * kv_heads * 4 * kKTile * head_dim * sizeof(_Float16), need = planes_bytes + (size_t)plane_tiles * kv_heads * (1 + kKTile) * sizeof(float);
    M40StreamScratch& sc = ctx->scratch[0];
    if (sc.attn_planes_bytes < need) {
        if (hipStreamSynchronize(ctx->prefill_stream) != hipSuccess) return -5;
        if (sc.attn_planes) (void)hipFree(sc.attn_planes);
        sc.attn_planes = nullptr;
        sc.attn_planes_bytes = 0;
        if (hipMalloc(&sc.attn_planes, need + need / 4) != hipSuccess) {
            (void)hipGetLastError();
            return -4;
        }
        sc.attn_planes_bytes = need + need / 4;
    }
    a.planes = static_cast<const _Float16*>(sc.attn_planes);
    a.plane_tiles = (uint32_t)plane_tiles;
    a.v_max = reinterpret_cast<float*>(static_cast<char*>(sc.attn_planes) + planes_bytes);
    a.v_key = a.v_max + (size_t)plane_tiles * kv_heads;
    if (rows) a.rows = *rows;
    (void)hipGetLastError();
    const dim3 pack_grid((max_kv + kKTile - 1) / kKTile, kv_heads, batch);
    uint64_t long_groups = 0;           // two-block workgroups that the long sequences make
    for (uint32_t i = 0; i < batch; ++i)
        if (host[i] >= kTwoBlockMinQueries) long_groups += (uint64_t)((host[i] + 32u * kWaves - 1) / (32u * kWaves)) * q_heads;
    const uint32_t blocks = long_groups >= (uint64_t)kTwoBlockMinGroupsPerCu * (uint64_t)ctx->num_cus ? 2u : 1u;
    const uint32_t q_group = 16u * kWaves * blocks;     // queries per workgroup
    const dim3 grid(q_heads, (max_q + q_group - 1) / q_group, batch);
    const auto launch = [&](auto hd, auto r) {
        constexpr int HD = decltype(hd)::value;
        using R = decltype(r);
        prefill_pack_kv_kernel<HD, R><<<pack_grid, kThreads, 0, ctx->prefill_stream>>>(a, r);
        if constexpr (std::is_same<R, PrefillRope>::value) {
            if (rows) {
                if (blocks == 2) prefill_attn_kernel<HD, 2, R, true><<<grid, kThreads, 0, ctx->prefill_stream>>>(a, r);
                else prefill_attn_kernel<HD, 1, R, true><<<grid, kThreads, 0, ctx->prefill_stream>>>(a, r);
                return;
            }
        }
        if (blocks == 2) prefill_attn_kernel<HD, 2, R, false><<<grid, kThreads, 0, ctx->prefill_stream>>>(a, r);
        else prefill_attn_kernel<HD, 1, R, false><<<grid, kThreads, 0, ctx->prefill_stream>>>(a, r);
    };
    const auto launch_rope = [&](auto hd) { rope ? launch(hd, *rope) : launch(hd, NoRope{}); };
    if (head_dim == 64) launch_rope(std::integral_constant<int, 64>());
    else launch_rope(std::integral_constant<int, 128>());
    if (hipGetLastError() != hipSuccess) return -4;
    if (synchronize && hipStreamSynchronize(ctx->prefill_stream) != hipSuccess) return -5;
    return 0;
}

}  // namespace

extern "C" {

int m40llm_attention_prefill_f32_gqa_varlen(M40llmCudaContext* ctx, const void* q_dev_f32, const void* k_dev_f32,
                                            const void* v_dev_f32, const uint32_t* q_offsets_dev,
                                            const uint32_t* kv_offsets_dev, const uint32_t* q_lens_dev,
                                            const uint32_t* kv_lens_dev, uint32_t batch_size, uint32_t q_heads,
                                            uint32_t kv_heads, uint32_t head_dim, void* out_dev_f32) {
    return prefill_impl(ctx, q_dev_f32, k_dev_f32, v_dev_f32, q_offsets_dev, kv_offsets_dev, q_lens_dev, kv_lens_dev,
                        batch_size, q_heads, kv_heads, head_dim, out_dev_f32, true);
}

int m40llm_attention_prefill_f32_gqa_varlen_async(M40llmCudaContext* ctx, const void* q_dev_f32, const void* k_dev_f32,
                                                  const void* v_dev_f32, const uint32_t* q_offsets_dev,
                                                  const uint32_t* kv_offsets_dev, const uint32_t* q_lens_dev,
                                                  const uint32_t* kv_lens_dev, uint32_t batch_size, uint32_t q_heads,
                                                  uint32_t kv_heads, uint32_t head_dim, void* out_dev_f32) {
    return prefill_impl(ctx, q_dev_f32, k_dev_f32, v_dev_f32, q_offsets_dev, kv_offsets_dev, q_lens_dev, kv_lens_dev,
                        batch_size, q_heads, kv_heads, head_dim, out_dev_f32, false);
}

int m40llm_ext_attention_prefill_f32_gqa_varlen_host_tables_async(M40llmCudaContext* ctx, const void* q_dev_f32,
                                                                  const void* k_dev_f32, const void* v_dev_f32,
                                                                  const uint32_t* q_offsets_dev, const uint32_t* kv_offsets_dev,
                                                                  const uint32_t* q_lens_dev, const uint32_t* kv_lens_dev,
                                                                  const uint32_t* kv_offsets_host, const uint32_t* q_lens_host,
                                                                  const uint32_t* kv_lens_host, uint32_t batch_size,
                                                                  uint32_t q_heads, uint32_t kv_heads, uint32_t head_dim,
                                                                  void* out_dev_f32) {
    if (!kv_offsets_host || !q_lens_host || !kv_lens_host) return -1;
    return prefill_impl(ctx, q_dev_f32, k_dev_f32, v_dev_f32, q_offsets_dev, kv_offsets_dev, q_lens_dev, kv_lens_dev,
                        batch_size, q_heads, kv_heads, head_dim, out_dev_f32, false, kv_offsets_host, q_lens_host, kv_lens_host);
}

static int rope_append(M40llmCudaContext* ctx, M40llmKVCache* kv, const void* q_dev_f32, const void* k_dev_f32,
                                                   const void* v_dev_f32, const uint32_t* offsets_dev, const uint32_t* lens_dev, uint32_t batch,
                                                   const uint32_t* seq_slots_host, const uint32_t* offsets_host, const uint32_t* lens_host, uint32_t q_heads,
                                                   uint32_t rope_layout, const void* d_angles, const void* d_bq_f32, const void* d_bk_f32,
                                                   const void* d_bv_f32, void* out_dev_f32, const M40TiledRows* rows) {
    if (!ctx || !kv || !q_dev_f32 || !k_dev_f32 || !v_dev_f32 || !offsets_dev || !lens_dev || !seq_slots_host || !offsets_host || !lens_host || !d_angles || (!out_dev_f32 && !rows))
        return -1;
    const int n_bias = (d_bq_f32 != nullptr) + (d_bk_f32 != nullptr) + (d_bv_f32 != nullptr);
    if (batch == 0 || batch > (uint32_t)kM40PrefillSeqs || (n_bias != 0 && n_bias != 3) || rope_layout > M40LLM_ROPE_LAYOUT_NEOX) return -2;
    if (kv->compressed || !kv->d_k || !kv->d_v) return -6;
    PrefillRope r{};
    uint32_t n_rows = 0;
    for (uint32_t i = 0; i < batch; ++i) {
        if (seq_slots_host[i] >= kv->max_batch_size) return -2;
        if (lens_host[i] > kv->max_seq_len) return -5;
        for (uint32_t j = 0; j < i; ++j)
            if (seq_slots_host[j] == seq_slots_host[i]) return -8;   // two sequences of one call would race on a slot
        r.slot[i] = seq_slots_host[i];
        r.first[i] = n_rows;
        n_rows += lens_host[i];              // at most 64 lengths, which the attention refuses above 8192
    }
    if (!m40_aligned16(d_angles)) return -4;
    r.angles = static_cast<const float2*>(d_angles);
    r.bq = static_cast<const float*>(d_bq_f32); r.bk = static_cast<const float*>(d_bk_f32); r.bv = static_cast<const float*>(d_bv_f32);
    r.layout = rope_layout; r.max_seq_len = kv->max_seq_len;
    r.k_cache = kv->d_k; r.v_cache = kv->d_v; r.seq_map = kv->d_seq_map;
    return prefill_impl(ctx, q_dev_f32, k_dev_f32, v_dev_f32, offsets_dev, offsets_dev, lens_dev, lens_dev, batch, q_heads, kv->num_heads, kv->head_dim, out_dev_f32,
                        false, offsets_host, lens_host, lens_host, &r, rows);
}

int m40llm_ext_prefill_attention_rope_append_async(M40llmCudaContext* ctx, M40llmKVCache* kv, const void* q_dev_f32, const void* k_dev_f32,
                                                   const void* v_dev_f32, const uint32_t* offsets_dev, const uint32_t* lens_dev, uint32_t batch,
                                                   const uint32_t* seq_slots_host, const uint32_t* offsets_host, const uint32_t* lens_host, uint32_t q_heads,
                                                   uint32_t rope_layout, const void* d_angles, const void* d_bq_f32, const void* d_bk_f32,
                                                   const void* d_bv_f32, void* out_dev_f32) {
    return rope_append(ctx, kv, q_dev_f32, k_dev_f32, v_dev_f32, offsets_dev, lens_dev, batch, seq_slots_host, offsets_host, lens_host, q_heads, rope_layout, d_angles, d_bq_f32,
                       d_bk_f32, d_bv_f32, out_dev_f32, nullptr);
}

int m40llm_ext_prefill_attention_project_gate_up_async(M40llmCudaContext* ctx, M40llmKVCache* kv, const void* q_dev_f32, const void* k_dev_f32, const void* v_dev_f32,
                                                       const uint32_t* offsets_dev, const uint32_t* lens_dev, uint32_t batch, const uint32_t* seq_slots_host,
                                                       const uint32_t* offsets_host, const uint32_t* lens_host, uint32_t q_heads, uint32_t rope_layout,
                                                       const void* d_angles, const void* d_bq_f32, const void* d_bk_f32, const void* d_bv_f32, uint32_t rows,
                                                       const void* d_wo_f16, int d_model, const void* d_residual_f32, void* d_x_f32, const void* d_norm_weight,
                                                       uint32_t norm_weight_dtype, float eps, const void* d_gate_f16, const void* d_up_f16, int ffn, void* d_hid_f32) {
    if (!ctx || !kv || !lens_host || !offsets_host || !d_wo_f16 || !d_residual_f32 || !d_x_f32 || !d_norm_weight || !d_gate_f16 || !d_up_f16 || !d_hid_f32) return -1;
    if (rows == 0 || d_model <= 0 || ffn <= 0 || norm_weight_dtype > 1u || batch == 0) return -2;
    // the sequences' rows lie one behind the other; what the product has behind them nobody reads
    uint64_t at = 0;
    for (uint32_t i = 0; i < batch; ++i) {
        if (offsets_host[i] != at) return 1;
        at += lens_host[i];
    }
    const uint64_t K = (uint64_t)q_heads * kv->head_dim;
    if (at > rows || rows > 65535u || K == 0 || K > 65536u) return 1;
    const uint16_t *wo = static_cast<const uint16_t*>(d_wo_f16), *B[2] = {static_cast<const uint16_t*>(d_gate_f16), static_cast<const uint16_t*>(d_up_f16)};
    float *x = static_cast<float*>(d_x_f32), *C[2] = {static_cast<float*>(d_hid_f32), nullptr};
    const int N[2] = {ffn, ffn};
    if (!m40_gemm_tiled_supported(nullptr, wo, (int)rows, d_model, (int)K) || !m40_aligned16(d_norm_weight) || ffn % 16 != 0 || ffn > 0x3fffffff ||
        !m40_gemm_tiled_supported(x, B[0], (int)rows, ffn, d_model) || !m40_gemm_tiled_supported(x, B[1], (int)rows, ffn, d_model))
        return 1;
    if (m40_ensure_device(ctx) != 0) return -2;
    auto attend = [&](const M40TiledRows& to) {
        return rope_append(ctx, kv, q_dev_f32, k_dev_f32, v_dev_f32, offsets_dev, lens_dev, batch, seq_slots_host, offsets_host, lens_host, q_heads, rope_layout, d_angles,
                           d_bq_f32, d_bk_f32, d_bv_f32, nullptr, &to);
    };
    return m40_launch_gemm_tiled_chain(ctx, ctx->prefill_stream, 0u, nullptr, (int)rows, (int)K, wo, d_model, static_cast<const float*>(d_residual_f32), x, d_norm_weight,
                                       norm_weight_dtype, eps, 2, B, N, C, true,
                                       [](void* f, const M40TiledRows& to) { return (*static_cast<decltype(attend)*>(f))(to); }, &attend);
}

}  // extern "C"
