// Products of up to 16 bf16 rows with packed weights: decode steps and experts with few rows (packed_gemm.hpp has the layout and the last steps).
//
// Bound by the weights' way from memory, and below some 20 MB by the round trips of a launch (an empty one takes 1.6 us, one that reads what the launch
// before wrote 2.0).  So a workgroup owns one column tile (or one pair of gate and up), its waves share out K and keep few requests each: at two k tiles a
// wave and the next two requested before those are multiplied, 32 waves fit on a CU.  A lane whose row is not there reads the last one's line again: the rows
// come through L2 once a workgroup, as many bytes as its weights if they came whole.  The last step is compiled for its kind: whatever else a general one
// holds would be fetched cold by every launch.  us a launch in a graph of its own kind, weights that no cache holds, one row (the kernel for all kinds
// and 4 to 16 waves that ran these before / this): K 2048, 128 tiles in two parts of K 4.25 / 3.6, 192 tiles 5.1 / 4.3, 528 tiles 10.1 / 8.2, 2000 tiles
// 24.3 / 20.7.
#include "packed_gemm.hpp"

namespace {

struct NoChoices {};
template <int JOBS> struct ChoicesOf { using type = NoChoices; };
template <> struct ChoicesOf<kFewIds> { using type = M40FewChoices; };

// The list of experts in use from the choices of up to 64 (row, choice) pairs, a lane a pair: what few_lists_kernel makes, for the one expert that is number `job` of those in use.
// A row's choices are different experts, so that none has more than 16 rows.  Ids are the caller's memory: of some that repeat an expert, pairs past its 16 slots share the last one.
struct ChosenExpert {
    int jobs, expert, rows;           // experts in use; this one (job < jobs), and how many rows took it
    int pair, row;                    // of the lane's operand row: lane % 16, or its last row
    uint32_t own;                     // the lane's choice (0xffffffff: none)
    unsigned long long hits;          // the pairs that took it
};
__device__ __forceinline__ uint32_t or64(uint32_t v) {
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, M40_DPP_XOR1, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, M40_DPP_XOR2, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, M40_DPP_HALF_MIRROR, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, M40_DPP_MIRROR, 0xf, 0xf, false);
    return (uint32_t)(__builtin_amdgcn_readlane((int)v, 0) | __builtin_amdgcn_readlane((int)v, 16) | __builtin_amdgcn_readlane((int)v, 32) | __builtin_amdgcn_readlane((int)v, 48));
}
__device__ __forceinline__ int bits_below(unsigned long long mask) {          // of the lane
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ ChosenExpert chosen_expert(const uint32_t* ids, int pairs, int top, uint32_t experts, int job, int lane) {
    ChosenExpert c;
    c.own = ids[lane < pairs ? lane : 0];
    if (lane >= pairs) c.own = 0xffffffffu;
    const bool real = c.own < experts;                                     // (experts at most 64)
    const unsigned long long used = (unsigned long long)or64(real && c.own >= 32u ? 1u << (c.own - 32u) : 0u) << 32 | or64(real && c.own < 32u ? 1u << c.own : 0u);
    c.jobs = __popcll(used);
    c.expert = __ffsll(__ballot((used >> lane & 1ull) && bits_below(used) == job)) - 1;
    c.hits = __ballot(real && (int)c.own == c.expert);
    c.rows = min(__popcll(c.hits), 16);
    // pair of the lane's operand row: pairs that took the expert go to the lanes of their rank, the others to one that is not looked at
    const int at = __builtin_amdgcn_ds_permute(4 * ((c.hits >> lane & 1ull) ? bits_below(c.hits) : 63), lane);
    c.pair = __shfl(at, (lane & 15) < c.rows ? lane & 15 : (c.rows > 0 ? c.rows - 1 : 0), 64);
    c.row = c.pair / top;
    return c;
}
// What later launches read of the list: the first expert's job also says how many there are, and where rows go on as they are.
__device__ __forceinline__ void store_list(const M40FewChoices& l, const ChosenExpert& c, int job, int lane) {
    if (job < c.jobs && (c.hits >> lane & 1ull)) l.place[lane] = 16u * (uint32_t)job + (uint32_t)min(bits_below(c.hits), 15);
    if (job == 0 && lane < l.rows * l.top && c.own >= (uint32_t)l.experts) l.place[lane] = M40LLM_PLACE_INPUT;
    if (lane != 0) return;
    if (job < c.jobs) *reinterpret_cast<uint4*>(l.jobs + 4 + 4 * job) = make_uint4((uint32_t)c.expert, 16u * (uint32_t)job, (uint32_t)c.rows, 0u);
    if (job == 0) *reinterpret_cast<uint2*>(l.jobs) = make_uint2((uint32_t)c.jobs, 16u * (uint32_t)c.jobs);
}

// The k tiles of a column tile are added up as PARTS sums (k tile i in sum i % PARTS, the sums in order), PARTS following from K alone, so that WAVES
// changes no bit.  A wave requests U k tiles together, with AHEAD the next U before those are multiplied.  JOBS as in M40FewRows.
//
// All that the first requests need stands in plain arguments, which lie in registers when a wave starts (a structure is read from memory first): count is
// the rows or, with jobs, lda in tiles; p0 the jobs or a_batch in tiles and above it the segment; p1 the gather list or k_total.  kFewIds: p0 the choices, p1 their number, those
// of a row and the experts (16, 16 and 32 bits).
template <int NT, int WAVES, int PARTS, int U, bool AHEAD, int KIND, int JOBS>
__global__ __launch_bounds__(WAVES * 64) void few_rows_kernel(const m40_bf16* rows_a, const m40_bf16* weights, int n_tiles, int k_tiles_in, int count, int k_stride, uint64_t p0, uint64_t p1,
                                                                      long w_batch, M40Epilogue<m40_bf16> e, typename ChoicesOf<JOBS>::type choices) {
    extern __shared__ __align__(16) float red[];       // [PARTS][NT][64][4]
    constexpr int kOwn = PARTS / WAVES;                // sums a wave keeps
    static_assert(PARTS % WAVES == 0 && U % kOwn == 0 && NT <= WAVES);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tile0 = (int)blockIdx.x * NT;
    int batch = blockIdx.z, row0 = 0, rows = count, k_tiles = k_tiles_in;
    constexpr bool kPlain = JOBS == kFewGather || JOBS == kFewIds;       // rows of a that a list names
    float row_scale = 1.0f;
    const m40_bf16* a = rows_a + (lane >> 4) * (kPlain ? 8 : 128);
    if (JOBS == kFewAll) {
        const int segment = (int)(p0 >> 32), k_total = (int)p1;
        a += (long)(segment ? tile0 / segment : batch) * (long)(uint32_t)p0 * kM40Tile + ((lane & 15) < rows ? lane & 15 : rows - 1) * 8;
        if (k_total && k_total - batch * k_tiles < k_tiles) k_tiles = k_total - batch * k_tiles;
    } else if constexpr (JOBS == kFewIds) {
        const ChosenExpert c = chosen_expert(reinterpret_cast<const uint32_t*>(p0), (int)(p1 & 0xffffu), (int)(p1 >> 16 & 0xffffu), (uint32_t)(p1 >> 32), (int)blockIdx.y, lane);
        if (blockIdx.x == 0 && wave == 0) store_list(choices, c, (int)blockIdx.y, lane);
        if ((int)blockIdx.y >= c.jobs) return;
        batch = c.expert;
        row0 = 16 * (int)blockIdx.y;
        rows = c.rows;
        a += (long)c.row * count * 32;
        if (choices.weight_input) row_scale = static_cast<const float*>(choices.weight)[c.pair];
    } else {
        const uint32_t* jobs = reinterpret_cast<const uint32_t*>(p0);
        if (blockIdx.y >= jobs[0]) return;
        const uint32_t* job = jobs + 4 + 4 * blockIdx.y;
        batch = (int)job[0];
        row0 = (int)job[1];
        rows = (int)job[2];
        const int r = (lane & 15) < rows ? lane & 15 : rows - 1;
        if (JOBS == kFewGather) a += (long)reinterpret_cast<const uint32_t*>(p1)[row0 + r] * count * 32;
        else a += (long)(row0 >> 4) * count * kM40Tile + r * 8;
    }
    constexpr long kStep = kPlain ? 32 : kM40Tile;       // elements from k tile to k tile
    const m40_bf16* w[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int t = tile0 + n < n_tiles ? tile0 + n : n_tiles - 1;
        w[n] = weights + batch * w_batch + (long)t * k_stride * kM40Tile + lane * 8;
    }
    m40_float4 acc[kOwn][NT];
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[q][n] = m40_float4{0.f, 0.f, 0.f, 0.f};
    struct Batch { uint4 w[U][NT]; m40_bf16x8 a[U]; };
    auto request = [&](Batch& b, int k) __attribute__((always_inline)) {
        const int left = (k_tiles - k + WAVES - 1) / WAVES;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= left) break;
#pragma unroll
            for (int n = 0; n < NT; ++n) b.w[u][n] = m40_load_stream(reinterpret_cast<const uint4*>(w[n] + (long)(k + u * WAVES) * kM40Tile));
            if (!kPlain) b.a[u] = *reinterpret_cast<const m40_bf16x8*>(a + (long)(k + u * WAVES) * kStep);
        }
        if (kPlain) {          // the rows' numbers are still on their way: all weights first
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (u >= left) break;
                b.a[u] = *reinterpret_cast<const m40_bf16x8*>(a + (long)(k + u * WAVES) * kStep);
            }
        }
    };
    auto multiply = [&](const Batch& b, int k) __attribute__((always_inline)) {
        const int left = (k_tiles - k + WAVES - 1) / WAVES;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= left) break;
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[u % kOwn][n] = M40Act<m40_bf16>::mma(__builtin_bit_cast(m40_bf16x8, b.w[u][n]), b.a[u], acc[u % kOwn][n]);
        }
    };
    if (AHEAD) {
        constexpr int kBatch = U * WAVES;
        Batch b[2];
        if (wave < k_tiles) request(b[0], wave);
        for (int k = wave; k < k_tiles; k += 2 * kBatch) {
            if (k + kBatch < k_tiles) request(b[1], k + kBatch);
            multiply(b[0], k);
            if (k + kBatch >= k_tiles) break;
            if (k + 2 * kBatch < k_tiles) request(b[0], k + 2 * kBatch);
            multiply(b[1], k + kBatch);
        }
    } else {
        for (int k = wave; k < k_tiles; k += U * WAVES) {
            Batch b;
            request(b, k);
            multiply(b, k);
        }
    }
    m40_float4* r4 = reinterpret_cast<m40_float4*>(red);
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
#pragma unroll
        for (int n = 0; n < NT; ++n) r4[((q * WAVES + wave) * NT + n) * 64 + lane] = acc[q][n];
    __syncthreads();
    if (KIND >= 0) e.kind = KIND;
    e.rows = row0 + rows;
    auto sum = [&](int n) __attribute__((always_inline)) {
        m40_float4 s = r4[n * 64 + lane];
#pragma unroll
        for (int i = 1; i < PARTS; ++i) s += r4[(i * NT + n) * 64 + lane];
        return s;
    };
    if (KIND == M40LLM_PACKED_PROJECT && (JOBS != kFewAll || tile0 >= e.plain_tiles)) {
        if (wave == 0) {
            if (JOBS == kFewIds) m40_epilogue_pair(e, row0, (tile0 - e.plain_tiles) / 2, lane, sum(0), sum(NT - 1), row_scale);
            else m40_epilogue_pair(e, row0, (tile0 - e.plain_tiles) / 2, lane, sum(0), sum(NT - 1));
        }
    } else if (wave < NT && tile0 + wave < n_tiles) {      // a wave a tile
        m40_epilogue_tile(e, JOBS == kFewAll ? batch : 0, row0, tile0 + wave, lane, sum(wave));
    }
}

template <int NT, int WAVES, int PARTS, int U, bool AHEAD, int KIND, int JOBS>
int launch(hipStream_t stream, const M40FewRows& g, const M40Epilogue<m40_bf16>& e) {
    const dim3 grid((unsigned)((g.n_tiles + NT - 1) / NT), (unsigned)g.max_jobs, (unsigned)g.batches);
    constexpr size_t lds = (size_t)PARTS * NT * 1024;
    static_assert(lds <= 64 * 1024);
    const bool all = JOBS == kFewAll;
    const uint64_t p0 = all ? (uint64_t)(uint32_t)g.segment << 32 | (uint32_t)(g.a_batch / kM40Tile) : (uint64_t)reinterpret_cast<uintptr_t>(g.jobs);
    const uint64_t p1 = all ? (uint64_t)(uint32_t)g.k_total : (uint64_t)reinterpret_cast<uintptr_t>(g.gather);
    if constexpr (JOBS == kFewIds)
        few_rows_kernel<NT, WAVES, PARTS, U, AHEAD, KIND, JOBS><<<grid, WAVES * 64, lds, stream>>>(
            g.a, g.w, g.n_tiles, g.k_tiles, (int)(g.lda / 32), g.k_stride, (uint64_t) reinterpret_cast<uintptr_t>(g.choices->ids),
            (uint64_t)(g.choices->rows * g.choices->top) | (uint64_t)g.choices->top << 16 | (uint64_t)g.choices->experts << 32, g.w_batch, e, *g.choices);
    else
        few_rows_kernel<NT, WAVES, PARTS, U, AHEAD, KIND, JOBS><<<grid, WAVES * 64, lds, stream>>>(g.a, g.w, g.n_tiles, g.k_tiles, all ? g.rows : (int)(g.lda / 32), g.k_stride, p0, p1, g.w_batch, e, NoChoices{});
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

template <int KIND, int JOBS>
int launch_kind(hipStream_t stream, const M40FewRows& g, const M40Epilogue<m40_bf16>& e, int num_cus) {
    if constexpr (KIND == M40LLM_PACKED_PROJECT) {
        // pairs of tiles, us, 4 waves / 8: 176 pairs 8.3 / 6.3; 352, of which some CUs get one and some two, 9.8 / 10.4; 352 of four experts 10.4 / 11.1; 1056 of
        // twelve 22.4 / 21.4, 2816 of 32 39.7 / 38.4
        const long long pairs = (long long)(g.n_tiles / 2) * (g.jobs || g.choices ? g.max_jobs : g.batches);
        if (pairs > num_cus && pairs <= 2ll * num_cus) return launch<2, 4, 8, 2, true, KIND, JOBS>(stream, g, e);
        return launch<2, 8, 8, 4, false, KIND, JOBS>(stream, g, e);
    } else {
        // The sums' number follows from K.  More than eight rows of many tiles are read once for two tiles: 16 rows, K 2048, 2000 tiles 21.5 us so, 23.8 one by one; 528 tiles 10.0 and 9.4.
        if (g.k_tiles >= 64) {
            if (JOBS == kFewAll && g.rows > 8 && (long long)g.n_tiles * g.batches > 4ll * num_cus) return launch<2, 8, 16, 4, true, KIND, JOBS>(stream, g, e);
            return launch<1, 16, 16, 2, true, KIND, JOBS>(stream, g, e);
        }
        if (g.k_tiles >= 16) return launch<1, 8, 8, 8, false, KIND, JOBS>(stream, g, e);
        return launch<1, 4, 4, 8, false, KIND, JOBS>(stream, g, e);
    }
}

}  // namespace

int m40_few_rows_product(hipStream_t stream, const M40FewRows& g, const M40Epilogue<m40_bf16>& e, int num_cus) {
    if (g.choices) return launch_kind<M40LLM_PACKED_PROJECT, kFewIds>(stream, g, e, num_cus);
    if (g.jobs) return g.gather ? launch_kind<M40LLM_PACKED_PROJECT, kFewGather>(stream, g, e, num_cus) : launch_kind<M40LLM_PACKED_STORE_ACT, kFewSlots>(stream, g, e, num_cus);
    switch (e.kind) {
        case M40LLM_PACKED_STORE: return launch_kind<M40LLM_PACKED_STORE, kFewAll>(stream, g, e, num_cus);
        case M40LLM_PACKED_CAP: return launch_kind<M40LLM_PACKED_CAP, kFewAll>(stream, g, e, num_cus);
        case M40LLM_PACKED_PROJECT: return launch_kind<M40LLM_PACKED_PROJECT, kFewAll>(stream, g, e, num_cus);
        default: return launch_kind<-1, kFewAll>(stream, g, e, num_cus);
    }
}
