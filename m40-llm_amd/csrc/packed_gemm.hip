// Products of tile-packed activations with tile-packed bf16 weights (packed_gemm.hpp has the layout and the last steps).
//
// rows_packed_kernel   a workgroup owns one or two column tiles for up to 64 rows and its waves share out K: weights go
//                      straight from memory into the matrix instruction's operand registers, one contiguous kilobyte a
//                      load, each tile read once per 64 rows; the waves' sums meet in LDS.  17 to 64 rows, and every
//                      product in f32 (up to 16 bf16 rows: few_rows.hip).
// tile_packed_kernel   bf16, more rows: tiles of C of 64 x 64 to 128 x 256, both operands staged through LDS by direct
//                      global-to-LDS loads, five or six stages deep with one barrier a stage.  The buffers hold
//                      operands in instruction order, so LDS reads are contiguous kilobytes as well.
//
// Products per expert: both kernels take a list of jobs (expert, rows of the list sorted by expert) made on the device; the rows are
// gathered from plain rows (few rows, gate and up) or lie packed in list order.
#include "norm_route.hpp"
#include "packed_gemm.hpp"

#include <type_traits>
#include <utility>

namespace {

struct PackedArgs {
    const void* a;
    const m40_bf16* w;
    long lda, a_batch, w_batch;
    int n_tiles, k_tiles, rows;
    int k_stride;                  // k tiles from one row tile of the weights to the next
    int k_total;                   // k tiles of all batches together where the batches are parts of K (else 0)
    // operand rows that lie in cache pages: row tile t is group t % 4 of page pages[t / 4]
    const uint32_t* pages;
    int page_k_tiles;
    const uint32_t *jobs, *gather; // products per expert
    int segment;                   // column tiles that read the same columns of a (0 = all): the next ones read those a_batch further
    __device__ int k_count(int batch) const { return k_total && k_total - batch * k_tiles < k_tiles ? k_total - batch * k_tiles : k_tiles; }
};

enum { kAllRows = 0, kJobSlots = 1, kJobGather = 2 };

constexpr int rows_at_once(int mt, int nt, int waves, int parts) { return parts * mt * nt <= 16 ? parts / waves : 1; }

// The k tiles of a product are added up as PARTS sums (k tile i in sum i % PARTS, the sums in order), PARTS following from K alone: WAVES, which
// follows from the launch's size, divides it and changes no bit of the result.
template <class T, int MT, int NT, int WAVES, int PARTS, int JOBS>
__global__ __launch_bounds__(WAVES * 64) void rows_packed_kernel(PackedArgs g, M40Epilogue<T> e) {
    extern __shared__ __align__(16) float red[];       // [sums at once][MT][NT][64][4]
    constexpr int kOwn = PARTS / WAVES;                // sums a wave keeps
    typedef typename M40Act<T>::vec8 vec8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile0 = (int)blockIdx.x * NT;
    int row0 = (int)blockIdx.y * 16 * MT, batch = blockIdx.z;
    if (JOBS != kAllRows) {
        if (blockIdx.y >= g.jobs[0]) return;
        const uint32_t* job = g.jobs + 4 + 4 * blockIdx.y;
        batch = (int)job[0];
        row0 = (int)job[1];
        g.rows = e.rows = row0 + (int)job[2];
    }
    constexpr long kStep = JOBS == kJobGather ? 32 : kM40Tile;       // elements from k tile to k tile
    const T* a[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int rt = row0 / 16 + m, last = (g.rows - 1) / 16, c = rt < last ? rt : last;
        if (JOBS == kJobGather) a[m] = static_cast<const T*>(g.a) + (long)g.gather[c * 16 + (lane & 15)] * g.lda + (lane >> 4) * 8;
        else a[m] = static_cast<const T*>(g.a) + (JOBS == kAllRows ? (g.segment ? tile0 / g.segment : batch) * g.a_batch : 0) + (long)c * 16 * g.lda + lane * 8;
    }
    const m40_bf16* w[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int t = tile0 + n < g.n_tiles ? tile0 + n : g.n_tiles - 1;
        w[n] = g.w + batch * g.w_batch + (long)t * g.k_stride * kM40Tile + lane * 8;
    }
    const int k_tiles = g.k_count(batch);
    m40_float4 acc[kOwn][MT][NT];
#pragma unroll
    for (int q = 0; q < kOwn; ++q)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[q][m][n] = m40_float4{0.f, 0.f, 0.f, 0.f};
    // A wave's next U k tiles are requested together, also where fewer are left (K 2048 over 16 waves is four): one by one each would cost a
    // round trip to memory.
    constexpr int U = sizeof(T) == 2 ? (MT * NT <= 2 ? 8 : 4) : 1;
    static_assert(PARTS % WAVES == 0 && U % kOwn == 0);
    for (int k = wave; k < k_tiles; k += U * WAVES) {
        uint4 wf[U][NT];
        vec8 af[U][MT];
        const int left = (k_tiles - k + WAVES - 1) / WAVES;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= left) break;
#pragma unroll
            for (int n = 0; n < NT; ++n) wf[u][n] = m40_load_stream(reinterpret_cast<const uint4*>(w[n] + (long)(k + u * WAVES) * kM40Tile));
#pragma unroll
            for (int m = 0; m < MT; ++m) af[u][m] = M40Act<T>::load8(a[m] + (long)(k + u * WAVES) * kStep);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= left) break;
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) acc[u % kOwn][m][n] = M40Act<T>::mma(__builtin_bit_cast(m40_bf16x8, wf[u][n]), af[u][m], acc[u % kOwn][m][n]);
        }
    }
    m40_float4* r4 = reinterpret_cast<m40_float4*>(red);
    static_assert(MT <= WAVES, "a wave adds up one row tile");
    const int mine = wave < MT ? wave : 0;
    m40_float4 s[NT];
    // all sums at once where they take no more memory than eight workgroups a CU have, else a wave's sums one after the other
    constexpr int kAtOnce = rows_at_once(MT, NT, WAVES, PARTS);
#pragma unroll
    for (int q = 0; q < kOwn; q += kAtOnce) {
        if (q > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NT; ++n) r4[(((i * WAVES + wave) * MT + m) * NT + n) * 64 + lane] = acc[q + i][m][n];
        __syncthreads();
        if (wave < MT) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int i = 0; i < kAtOnce * WAVES; ++i) {
                    const m40_float4 v = r4[((i * MT + mine) * NT + n) * 64 + lane];
                    s[n] = q == 0 && i == 0 ? v : s[n] + v;
                }
        }
    }
    if (wave >= MT || row0 + mine * 16 >= g.rows) return;
    if (NT == 2 && e.kind == M40LLM_PACKED_PROJECT && tile0 >= e.plain_tiles) {
        m40_epilogue_pair(e, row0 + mine * 16, (tile0 - e.plain_tiles) / 2, lane, s[0], s[NT - 1]);
    } else {
#pragma unroll
        for (int n = 0; n < NT; ++n)
            if (tile0 + n < g.n_tiles) m40_epilogue_tile(e, JOBS == kAllRows ? batch : 0, row0 + mine * 16, tile0 + n, lane, s[n]);
    }
}

template <class T, int MT, int NT, int WAVES, int PARTS, int JOBS>
int launch_rows(hipStream_t stream, const PackedArgs& g, const M40Epilogue<T>& e, int batches) {
    // g.rows: with jobs, the most jobs there can be
    const dim3 grid((unsigned)((g.n_tiles + NT - 1) / NT), (unsigned)(JOBS == kAllRows ? (g.rows + 16 * MT - 1) / (16 * MT) : g.rows), (unsigned)batches);
    constexpr size_t lds = (size_t)rows_at_once(MT, NT, WAVES, PARTS) * WAVES * MT * NT * 1024;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(rows_packed_kernel<T, MT, NT, WAVES, PARTS, JOBS>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return -2;
    rows_packed_kernel<T, MT, NT, WAVES, PARTS, JOBS><<<grid, WAVES * 64, lds, stream>>>(g, e);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Waves and column tiles of a workgroup, bf16: a launch is mostly the round trips of its requests, so as many waves share out K as let every
// workgroup have its place at once (32 waves a CU); bf16 tiles go in pairs, which read the rows once.  K 2048, weights that no cache
// holds, us:
//   64 rows, 16 waves / pairs and 8 waves / pairs and 4: 192 tiles 8.5 / 11.0 / 12.4, 384 tiles 15.0 / 11.1 / 11.7, 644 tiles 21.8 / 21.1 / 18.8, 2000 tiles
//   57 / 43 / 36
template <class T, int MT, int PARTS, int JOBS>
int launch_rows_parts(hipStream_t stream, const PackedArgs& g, const M40Epilogue<T>& e, int batches, long long tiles, int num_cus) {
    if constexpr (sizeof(T) == 2) {
        if constexpr (JOBS == kAllRows)
            if (MT > 1 && tiles > num_cus) {
                if (tiles <= 2ll * num_cus) return launch_rows<T, MT, 2, 8, PARTS, JOBS>(stream, g, e, batches);
                return launch_rows<T, MT, 2, 4, PARTS, JOBS>(stream, g, e, batches);
            }
        if (tiles > 2ll * num_cus) return launch_rows<T, MT, 1, 4, PARTS, JOBS>(stream, g, e, batches);
        if (tiles > num_cus) return launch_rows<T, MT, 1, 8, PARTS, JOBS>(stream, g, e, batches);
    }
    return launch_rows<T, MT, 1, PARTS, PARTS, JOBS>(stream, g, e, batches);
}
template <class T, int MT, int JOBS>
int launch_rows_m(hipStream_t stream, const PackedArgs& g, const M40Epilogue<T>& e, int batches, int num_cus) {
    // jobs: as many as there can be
    const long long tiles = (long long)g.n_tiles * (JOBS == kAllRows ? (long long)((g.rows + 16 * MT - 1) / (16 * MT)) * batches : g.rows);
    if constexpr (JOBS != kJobSlots)
        if (e.kind == M40LLM_PACKED_PROJECT) {
            if constexpr (sizeof(T) == 2)
                if (tiles > 2ll * num_cus) return launch_rows<T, MT, 2, 4, 8, JOBS>(stream, g, e, batches);
            return launch_rows<T, MT, 2, 8, 8, JOBS>(stream, g, e, batches);
        }
    if constexpr (JOBS != kJobGather) {
        if (g.k_tiles >= 64) return launch_rows_parts<T, MT, 16, JOBS>(stream, g, e, batches, tiles, num_cus);
        if (g.k_tiles >= 16) return launch_rows_parts<T, MT, 8, JOBS>(stream, g, e, batches, tiles, num_cus);
        return launch_rows<T, MT, 1, 4, 4, JOBS>(stream, g, e, batches);
    }
    return -3;
}
template <class T, int JOBS>
int launch_rows_any(hipStream_t stream, const PackedArgs& g, const M40Epilogue<T>& e, int batches, int rows, int num_cus) {
    if constexpr (sizeof(T) == 4)          // (few_rows.hip in bf16)
        if (rows <= 16) return launch_rows_m<T, 1, JOBS>(stream, g, e, batches, num_cus);
    if (rows <= 32) return launch_rows_m<T, 2, JOBS>(stream, g, e, batches, num_cus);
    return launch_rows_m<T, 4, JOBS>(stream, g, e, batches, num_cus);
}

// ---- many rows, bf16 ---------------------------------------------------------------------------------------------------
// Workgroup of WM x WN waves, wave tile 16 MTW x 16 NTW: C tile 16 WM MTW x 16 WN NTW.  A stage is KS k tiles of every operand
// tile: (WM MTW + WN NTW) KS KB, filled by global_load_lds (a wave's instruction moves one 16 x 32 operand tile, a contiguous kilobyte).
//
// Memory instructions are issued under matrix instructions: the fragments of the next step and the loads of a stage kBufs - 1
// ahead go out one at a time between the current step's products (sched_group_barrier), so that no wave waits for an address
// or LDS unit with the matrix pipe idle.  Stage s refills the buffer of stage s - 1, whose fragments every wave had in registers
// before the barrier behind that stage, and ends with stage s + 2 landed.
enum { kPlainRows = 0, kPageKeys = 1, kPageValues = 2, kSlots = 3 };

// s_waitcnt for vector-memory operations only, then the barrier: reads of LDS need no wait of their own here
template <int VM>
__device__ __forceinline__ void landed_and_meet() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0f70 | (VM & 15) | ((VM >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
}
template <int... I, class F>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }

// rows of tiles of a wave whose sums fit into the buffers at a time
constexpr int tile_part(int mtw, int ntw, int wm, int wn, int ks, int bufs) {
    int part = mtw;
    while (wm * wn * part * ntw > (wm * mtw + wn * ntw) * ks * bufs) part /= 2;
    return part;
}

template <int MTW, int NTW, int WM, int WN, int KS, int kBufs, int FORM>
__global__ __launch_bounds__(64 * WM * WN, 1) void tile_packed_kernel(PackedArgs g, M40Epilogue<m40_bf16> e, int band) {
    typedef __attribute__((address_space(3))) void* lds_dst_t;
    typedef const __attribute__((address_space(1))) void* global_src_t;
    extern __shared__ __align__(16) uint8_t stage_lds[];
    constexpr int kWaves = WM * WN, kATiles = WM * MTW, kBTiles = WN * NTW, kRows = 16 * kATiles;      // 16-row operand tiles of the workgroup
    constexpr int kStageBytes = (kATiles + kBTiles) * KS * 1024;
    static_assert(kATiles * KS % kWaves == 0 && kBTiles * KS % kWaves == 0);
    constexpr int kALoads = kATiles * KS / kWaves, kLoads = (kATiles + kBTiles) * KS / kWaves;      // per wave and stage
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr bool kJobs = FORM == kSlots, kPaged = FORM == kPageKeys || FORM == kPageValues;
    const int tiles_n = (g.n_tiles + kBTiles - 1) / kBTiles, tiles_m = kJobs ? (int)g.jobs[0] : (g.rows + kRows - 1) / kRows;
    const int workgroups = kJobs ? tiles_m * tiles_n : (int)gridDim.x;       // the grid is as large as the list of jobs can be
    if (kJobs && (int)blockIdx.x >= workgroups) return;
    // workgroups are dealt to the eight dies in turn: each die gets a contiguous run of tiles, walked in blocks of `band` row
    // tiles so that what runs on a die at one time shares both operands
    const int per_die = workgroups / 8;
    const int logical = (int)blockIdx.x < per_die * 8 ? ((int)blockIdx.x % 8) * per_die + (int)blockIdx.x / 8 : (int)blockIdx.x;
    const int group = logical / (band * tiles_n), in_group = logical - group * band * tiles_n, gm = tiles_m - group * band < band ? tiles_m - group * band : band;
    const int t0 = __builtin_amdgcn_readfirstlane(in_group / gm * kBTiles), row_tile = group * band + in_group % gm;
    int m0 = __builtin_amdgcn_readfirstlane(row_tile * kRows), batch = blockIdx.z;
    if (kJobs) {
        const uint32_t* job = g.jobs + 4 + 4 * row_tile;
        batch = __builtin_amdgcn_readfirstlane((int)job[0]);
        m0 = __builtin_amdgcn_readfirstlane((int)job[1]);
        g.rows = e.rows = m0 + __builtin_amdgcn_readfirstlane((int)job[2]);
    }
    const int stages = g.k_count(batch) / KS;
    // A scalar address that walks k, and per lane a 32-bit offset from it that does not change (cache pages lie anywhere: whole addresses).
    // This wave's pieces of a stage: operand tiles' k tiles wave, wave + kWaves, ... of A, then of the weights.
    const uint8_t* a_base = static_cast<const uint8_t*>(g.a) + ((kJobs ? 0 : (g.segment ? t0 / g.segment : batch) * g.a_batch) + (long)m0 * g.lda) * 2;
    const uint8_t* w_base = reinterpret_cast<const uint8_t*>(g.w + batch * g.w_batch + (long)t0 * g.k_stride * kM40Tile);
    const uint8_t* page[kPaged ? kALoads : 1];
    uint32_t off[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int piece = wave + kWaves * i, sub = piece % KS, t = piece / KS;
        if (i >= kALoads) {
            const int n = t0 + t - kATiles;
            off[i] = (uint32_t)((n < g.n_tiles ? n : g.n_tiles - 1) - t0) * (uint32_t)g.k_stride * 1024u + sub * 1024u + lane * 16u;
        } else if (kPaged) {
            const int rt = m0 / 16 + t, tiles = g.rows / 16, c = rt < tiles ? rt : tiles - 1;
            page[kPaged ? i : 0] = static_cast<const uint8_t*>(g.a) + (((long)g.pages[c >> 2] * 4 + (c & 3)) * g.page_k_tiles + sub) * 1024 + lane * 16;
        } else {
            const int last = (g.rows - 1 - m0) / 16;
            off[i] = (uint32_t)(t < last ? t : last) * (uint32_t)g.lda * 32u + sub * 1024u + lane * 16u;
        }
    }
    auto issue = [&](int buf, int s) __attribute__((always_inline)) {
        uint8_t* base = stage_lds + buf * kStageBytes + wave * 1024;
        int k = (s < stages ? s : stages - 1) * KS * 1024;               // past the end: loaded again, not used
        asm("" : "+s"(k));                                               // keeps it out of the lanes' addresses
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const uint8_t* src = i >= kALoads ? w_base + k + off[i] : kPaged ? page[kPaged ? i : 0] + k : a_base + k + off[i];
            __builtin_amdgcn_global_load_lds((global_src_t)src, (lds_dst_t)(base + i * (kWaves * 1024)), 16, 0, 0);
        }
    };
    const int wm = wave / WN, wn = wave % WN;
    m40_float4 acc[MTW][NTW];
#pragma unroll
    for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) acc[i][j] = m40_float4{0.f, 0.f, 0.f, 0.f};
    struct Frags { m40_bf16x8 a[MTW], b[NTW]; } f[2];
    auto read_frags = [&](Frags& f, int buf, int sub) __attribute__((always_inline)) {
        const uint8_t* a = stage_lds + buf * kStageBytes + (wm * MTW * KS + sub) * 1024 + lane * 16;
        const uint8_t* b = stage_lds + buf * kStageBytes + ((kATiles + wn * NTW) * KS + sub) * 1024 + lane * 16;
#pragma unroll
        for (int i = 0; i < MTW; ++i) f.a[i] = *reinterpret_cast<const m40_bf16x8*>(a + i * KS * 1024);
#pragma unroll
        for (int j = 0; j < NTW; ++j) f.b[j] = *reinterpret_cast<const m40_bf16x8*>(b + j * KS * 1024);
    };
    auto compute = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MTW; ++i)
#pragma unroll
            for (int j = 0; j < NTW; ++j)
                acc[i][j] = FORM == kPageValues ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.a[i], f.b[j], acc[i][j], 0, 0, 0)
                                                : __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < kBufs - 1; ++i) issue(i, i);
    landed_and_meet<(kBufs - 3) * kLoads>();                         // stages 0 and 1 have landed
    read_frags(f[0], 0, 0);
    // ph: the stage's number in a period, after which buffers and fragment sets are back in their order; periods are written out so that
    // addresses are constants and sums stay in their registers
    constexpr int kPeriod = KS == 2 || kBufs % 2 == 0 ? kBufs : 2 * kBufs;
    auto sub_step = [&](auto ph_c, auto sub_c, int s) __attribute__((always_inline)) {
        constexpr int ph = decltype(ph_c)::value, sub = decltype(sub_c)::value, buf = ph % kBufs, set = (ph * KS + sub) & 1;
        read_frags(f[set ^ 1], sub + 1 < KS ? buf : (buf + 1) % kBufs, (sub + 1) % KS);
        if constexpr (sub == 0) issue((buf + kBufs - 1) % kBufs, s + kBufs - 1);
        compute(f[set]);
        // products between two fragment reads, and between two loads
        constexpr int kReads = MTW + NTW, kProducts = MTW * NTW, kPerRead = kProducts >= 2 * kReads + kLoads ? 2 : 1;
        constexpr int kPerLoad = (kProducts - kPerRead * kReads) / kLoads > 0 ? (kProducts - kPerRead * kReads) / kLoads : 1;
#pragma unroll
        for (int i = 0; i < kReads; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, kPerRead, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if constexpr (sub == 0) {
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
        landed_and_meet<(kBufs - 3) * kLoads>();
    };
    int s = 0;
    for (; s + kPeriod <= stages; s += kPeriod)
        unrolled(std::make_integer_sequence<int, kPeriod>(), [&](auto ph_c) __attribute__((always_inline)) { stage(ph_c, s + decltype(ph_c)::value); });
    unrolled(std::make_integer_sequence<int, kPeriod - 1>(), [&](auto ph_c) __attribute__((always_inline)) {
        if (s + decltype(ph_c)::value < stages) stage(ph_c, s + decltype(ph_c)::value);
    });
    m40_wait_and_meet<0>();                                          // every load has landed: the buffers are free
    if (FORM == kPlainRows && e.kind == M40LLM_PACKED_ADD && e.vec_out && e.cols % 16 == 0) {
        // The old values of a row of tiles are requested together, under clamped addresses and ahead of the stores of the row before: loads
        // behind a branch or behind a store that they might alias would be awaited one by one.
        float* o[NTW];
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            const int col = (t0 + wn * NTW + j) * 16;
            o[j] = e.out_f32 + batch * e.out_batch + (col < e.cols ? col : 0) + 4 * (lane >> 4);
        }
        m40_float4 old[2][NTW];
        auto request = [&](auto i_c) __attribute__((always_inline)) {
            constexpr int i = decltype(i_c)::value;
            const int row = m0 + (wm * MTW + i) * 16 + (lane & 15);
            const long at = (long)(row < e.rows ? row : e.rows - 1) * e.ld_out;
#pragma unroll
            for (int j = 0; j < NTW; ++j) old[i & 1][j] = *reinterpret_cast<const m40_float4*>(o[j] + at);
            __builtin_amdgcn_sched_barrier(0);
        };
        request(std::integral_constant<int, 0>());
        unrolled(std::make_integer_sequence<int, MTW>(), [&](auto i_c) __attribute__((always_inline)) {
            constexpr int i = decltype(i_c)::value;
            if constexpr (i + 1 < MTW) request(std::integral_constant<int, i + 1>());
            const int row = m0 + (wm * MTW + i) * 16 + (lane & 15);
            if (row >= e.rows) return;
#pragma unroll
            for (int j = 0; j < NTW; ++j)
                if ((t0 + wn * NTW + j) * 16 < e.cols) *reinterpret_cast<m40_float4*>(o[j] + (long)row * e.ld_out) = old[i & 1][j] + acc[i][j];
        });
        return;
    }
    // The sums go through LDS (each wave its own, as many rows of tiles at a time as fit) so that the last step is a loop of a few instructions
    // and not MTW NTW copies of it: run once per workgroup, those would be fetched cold.
    constexpr int kPart = tile_part(MTW, NTW, WM, WN, KS, kBufs);
    m40_float4* mine = reinterpret_cast<m40_float4*>(stage_lds) + wave * kPart * NTW * 64 + lane;
#pragma unroll 1
    for (int part = 0; part < MTW / kPart; ++part) {
        unrolled(std::make_integer_sequence<int, MTW / kPart>(), [&](auto p_c) __attribute__((always_inline)) {
            if (part != decltype(p_c)::value) return;
#pragma unroll
            for (int i = 0; i < kPart; ++i)
#pragma unroll
                for (int j = 0; j < NTW; ++j) mine[(i * NTW + j) * 64] = acc[decltype(p_c)::value * kPart + i][j];
        });
        const int part_row = m0 + (wm * MTW + part * kPart) * 16;
#pragma unroll 1
        for (int p = 0; p < kPart * NTW / 2; ++p) {
            const int i = p / (NTW / 2), j = p % (NTW / 2) * 2, row0 = part_row + i * 16, tile = t0 + wn * NTW + j;
            if (row0 >= g.rows || tile >= g.n_tiles) continue;
            const m40_float4 v0 = mine[(2 * p) * 64], v1 = mine[(2 * p + 1) * 64];
            const bool second = tile + 1 < g.n_tiles;
            if (FORM == kPageValues) {
                m40_epilogue_values(e, row0, tile, lane, v0);
                if (second) m40_epilogue_values(e, row0, tile + 1, lane, v1);
            } else if (e.kind == M40LLM_PACKED_PROJECT && tile >= e.plain_tiles) {
                if (second) m40_epilogue_pair(e, row0, (tile - e.plain_tiles) / 2, lane, v0, v1);
            } else {
#pragma unroll 1
                for (int k = 0; k < (second ? 2 : 1); ++k) m40_epilogue_tile(e, kJobs ? 0 : batch, row0, tile + k, lane, k ? v1 : v0);
            }
        }
    }
}

template <int MTW, int NTW, int KS, int kBufs, int FORM, int WM, int WN>
int launch_tile(hipStream_t stream, const PackedArgs& g, const M40Epilogue<m40_bf16>& e, int batches) {
    constexpr int lds = (WM * MTW + WN * NTW) * KS * 1024 * kBufs;
    static_assert(lds <= 160 * 1024);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(tile_packed_kernel<MTW, NTW, WM, WN, KS, kBufs, FORM>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (attr != hipSuccess) return -2;
    constexpr bool kJobs = FORM == kSlots;        // g.rows: the most jobs there can be
    const long long tiles_m = kJobs ? g.rows : (g.rows + 16 * WM * MTW - 1) / (16 * WM * MTW), tiles = tiles_m * ((g.n_tiles + WN * NTW - 1) / (WN * NTW));
    // blocks of 5 to 7 rows of tiles measure alike, larger and smaller ones up to a tenth slower (4096 rows, K 2048, N 11264, 128 x 128 tiles, blocks of
    // 4 / 6 / 8 / 16 / 32: 188 / 178 / 185 / 187 / 214 us); few rows are one block
    const int band = kJobs ? 4 : tiles_m <= 9 ? (int)tiles_m : 6;
    tile_packed_kernel<MTW, NTW, WM, WN, KS, kBufs, FORM><<<dim3((unsigned)tiles, 1, (unsigned)batches), 64 * WM * WN, lds, stream>>>(g, e, band);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}
// Which tile: sums are the same whichever it is.  Of the three small ones a launch of t workgroups on c CUs takes, per k tile, about max(least, start + load * t / c): one workgroup
// alone waits for the round trips of a stage, the second on its CU fills those waits.  Tiles of 128 x 128 and 64 x 64 are eight waves, half the wave tile of four: more waves a SIMD that
// fill each other's waits, for more fragment bytes a product (64 x 128 in stages of one k tile has no eight shares of its rows).  us, four waves / eight: 1200 rows, K 2048, N 2048 22.4 /
// 18.9; 2048 rows, K 1408, N 2048 20.4 / 17.1; 4096 rows, K 768, N 3072 29.3 / 27.6; 1500 rows, K 4096, N 2048 35.9 / 30.9; 4096 rows, N 12624 217 / 219; 77 rows, K 2048, N 2048 9.2 / 8.5;
// experts of 2048 x 1408, gate and up / down, 2000 rows 74.5 / 36.1, 73.7 / 34.2, 10 268 rows 168.8 / 85.0, 166.5 / 86.5, of 1024 x 704, 8000 rows 41.6 / 28.1, 38.7 / 26.0.
// The constants were fitted to four waves.  What they choose now, with the two large tiles below (128 x 128 / 64 x 128 / 64 x 64 / 128 x 256 / 256 x 256, the chosen one in brackets; us,
// bf16, weights that no cache holds):
//   K 2048, N 2048:  77 rows 15.7 / 12.7 / [8.5] / 24.7 / 44, 300 rows 16.6 / 13.1 / [9.2] / 25.8 / 46, 700 rows 17.5 / [14.1] / 15.4 / 26.7 / 47, 1200 rows [18.8] / 22.5 / 22.1 / 27.8 / 48,
//     2048 rows [21.1] / 25.0 / 29.8 / 29.5 / 50, 4096 rows 35.7 / 44.8 / 55.5 / [34.9] / 54;  N 4096: 1500 rows 31.8 / 35.0 / 42.5 / [31.9] / 50, 2567 rows [49.0] / 63 / 73 / 58 / 56
//   N 11264: 77 rows 22.8 / [18.4] / 18.8 / 31.7 / 48, 300 rows [31.8] / 30.6 / 35.4 / 32.9 / 52, 700 rows [50.9] / 52.9 / 64 / 58 / 55, 1024 rows 60 / 74 / 88 / 69 / [58], 1300 rows 73 / 91 /
//     109 / [69] / 104, 2048 rows 106 / 130 / 159 / [101] / 112, 2600 rows 137 / 160 / 190 / 127 / [119], 4096 rows 193 / 234 / 284 / 187 / [170]
//   N 12624: 500 rows 40.7 / 49 / 56 / [36.5] / 54, 1300 rows [84] / 102 / 121 / 90 / 103, 1500 rows [90] / - / - / 97 / 103, 4096 rows [218] / - / - / 213 / 212;  N 12048: 2000 rows 107 / - /
//     - / [103] / 113, 3000 rows [164] / - / - / 161 / 163
//   K 5632, N 2048: 77 rows 34.5 / 27.4 / [17.5] / 56 / 99, 700 rows 39.4 / [34.8] / 38.4 / 59 / 103, 1300 rows [41.4] / 52 / 56 / 61 / 104, 4096 rows 90 / 115 / 143 / [82] / 113
//   4096 rows, K 768, N 3072 [27.7] / 35.7 / 43.4 / 34.4 / 33.0; 2048 rows, K 1408, N 2048 [17.2] / 20.3 / 23.4 / 24.1 / 39.4; K 7680, N 2048 [67] / 87 / 105 / 97 / 146; K 4096, N 4096 69.7 /
//     88 / 111 / [62.5] / 91; 1200 rows, K 4096, N 11008 130 / 156 / 182 / 116 / [104]
// Of 80 shapes of 1100 to 2600 rows (N 2048 to 12624, K 2048 to 7680) 128 x 128, the one chosen and the two large ones were timed as well: the chosen one is the fastest or within 3 % of
// it in 70 and at most 8 % behind in the others (128 x 128 where 128 x 256 is faster: 2200 to 2600 rows, K 5632, N 2048 69 to 75 against 64 to 70; 1250 rows, K 4096, N 4096 62 / 58), and
// never more than half a per cent slower than what four waves took.
constexpr struct { int rows, cols; float least, start, load; } kTileShapes[3] = {{128, 128, 0.28f, 0.13f, 0.245f}, {64, 128, 0.20f, 0.10f, 0.165f}, {64, 64, 0.13f, 0.10f, 0.10f}};
// The two large ones are eight waves alone on their CU, and what counts is rounds of the CUs: a k tile of one takes `start` us, a round `fixed` besides, and a round that not all CUs
// have `least` of a full one and more the fuller it is.  Two waves a SIMD fill each other's waits, and of the larger one an operand byte from L2 serves 128 products instead of 64
// (1240 TFLOP/s with every CU busy, more than a large product of the library's).  us, 256 x 256 / 128 x 256 (in brackets: four waves to a tile of 128 x 256):
//   4096 rows, K 2048: N 2048 53 / 36, N 12048 184 / 199, N 12624 217 / 220 (a whole prompt with the former in place of 128 x 128 2235, with 128 x 128 2202); K 7680, N 2048: 148 / 108 [114];
//   K 4096: N 4096 111 / 121, N 11008 292 / 322;  2048 rows, N 11264, K 2048: 113 / 105; N 11008, K 4096: 188 / 175; 1024 rows, N 11008, K 4096: 95 / 116;  3000 rows, K 2048, N 12048 168 / 164
constexpr struct { int rows, cols; float start, fixed, least; } kLargeTiles[2] = {{128, 256, 0.45f, 5.0f, 0.9f}, {256, 256, 0.86f, 7.0f, 0.6f}};
constexpr int kLargeFrom = 48;           // k tiles

template <int FORM>
int launch_tile_any(hipStream_t stream, const PackedArgs& g, const M40Epilogue<m40_bf16>& e, int batches, int num_cus) {
    if constexpr (FORM == kSlots) {
        // A job is one row of tiles.  Long sums take the wider tile, which reads a job's rows half as often (32 experts of 4096 x 2752, gate and up / down, us: 2048 rows 281 / 152, four
        // waves to such a tile 289 / 160; 8192 rows 558 / 298, 571 / 309); of 2048 x 1408 the narrow one's two workgroups a CU are faster (10 268 rows 174, wide 189).
        if (g.k_tiles > 64) return launch_tile<4, 4, 1, 6, FORM, 2, 4>(stream, g, e, batches);
        return launch_tile<2, 4, 1, 5, FORM, 4, 2>(stream, g, e, batches);
    } else {
        const bool pairs = g.k_tiles % 2 == 0 && g.k_total % 2 == 0;          // two k tiles a stage
        const auto count = [&](int rows, int cols) { return (long long)((g.rows + rows - 1) / rows) * ((g.n_tiles * 16 + cols - 1) / cols) * batches; };
        int best = 0;
        float best_cost = 3.0e38f, best_us = 0.0f;
        long long t[3];
        for (int c = 0; c < 3; ++c) {
            t[c] = count(kTileShapes[c].rows, kTileShapes[c].cols);
            if (c == 2 && !pairs) continue;
            const float u = (float)t[c] / (float)num_cus, cost = kTileShapes[c].start + kTileShapes[c].load * u;
            const float at_least = cost > kTileShapes[c].least ? cost : kTileShapes[c].least;
            // (what a tile takes besides its k tiles, which counts beside the large ones)
            if (at_least < best_cost) { best_cost = at_least; best = c; best_us = at_least * (float)g.k_tiles + 1.5f * u * (float)(kTileShapes[c].rows * kTileShapes[c].cols) / 16384.0f; }
        }
        int large = -1;
        for (int c = 0; c < 2 && g.k_tiles >= kLargeFrom; ++c) {
            const long long n = count(kLargeTiles[c].rows, kLargeTiles[c].cols), full = n / num_cus, rest = n % num_cus;
            if (2 * n < num_cus || g.lda > 1 << 23) continue;            // (a tile's operand rows lie within 32-bit offsets)
            const float part = rest ? kLargeTiles[c].least + (1.0f - kLargeTiles[c].least) * (float)rest / (float)num_cus : 0.0f;
            const float us = kLargeTiles[c].start * (float)g.k_tiles * ((float)full + part) + kLargeTiles[c].fixed * (float)(full + (rest != 0));
            if (us < best_us) { best_us = us; large = c; }
        }
        if (large == 0) return launch_tile<4, 4, 1, 6, FORM, 2, 4>(stream, g, e, batches);
        if (large == 1) return launch_tile<4, 8, 1, 4, FORM, 4, 2>(stream, g, e, batches);
        // alone on its CU a workgroup takes the memory of two for deeper buffers: N 2048, K 5632 at 77 rows 21.2 us (64 x 64) against 24.4, at
        // 1300 rows 43.6 us (128 x 128) against 50.7
        const bool alone = pairs && t[best] <= num_cus;
        switch (best) {
            case 0: return alone ? launch_tile<2, 4, 2, 5, FORM, 4, 2>(stream, g, e, batches) : launch_tile<2, 4, 1, 5, FORM, 4, 2>(stream, g, e, batches);
            case 1: return launch_tile<2, 4, 1, 6, FORM, 2, 2>(stream, g, e, batches);
            default: return alone ? launch_tile<1, 2, 2, 6, FORM, 4, 2>(stream, g, e, batches) : launch_tile<1, 2, 2, 5, FORM, 4, 2>(stream, g, e, batches);
        }
    }
}

template <class T>
M40Epilogue<T> make_epilogue(const M40llmPackedGemm& p) {
    M40Epilogue<T> e{};
    e.kind = (int)p.epilogue;
    e.rows = (int)p.rows;
    e.out_f32 = static_cast<float*>(p.out_f32);
    e.out_act = static_cast<T*>(p.out_act);
    e.ld_out = (long)p.ld_out; e.ld_act = (long)p.ld_act;
    e.out_batch = (long)p.out_batch; e.act_batch = (long)p.act_batch;
    e.cols = (int)p.cols;
    auto aligned = [](const void* q, size_t n) { return reinterpret_cast<uintptr_t>(q) % n == 0; };
    e.vec_out = p.ld_out % 4 == 0 && p.out_batch % 4 == 0 && aligned(p.out_f32, 16);
    e.vec_act = p.ld_act % 4 == 0 && p.act_batch % 4 == 0 && aligned(p.out_act, 4 * sizeof(T));
    e.plain_tiles = (int)p.plain_tiles;
    e.activation = (int)p.activation;
    e.act_alpha = p.act_alpha; e.act_limit = p.act_limit;
    e.row_scale = static_cast<const float*>(p.row_scale);
    e.out_scale = p.out_scale; e.out_cap = p.out_cap;
    e.n_tiles = (int)p.n_tiles; e.act_col = (int)p.act_col;
    e.gate = static_cast<const float*>(p.gate);
    e.ld_gate = (long)p.ld_gate;
    e.head_width = (int)p.head_width; e.rot_start = (int)p.rot_start; e.heads = (int)p.heads;
    e.split_row = (int)p.split_row; e.rot_half = (int)p.rot_half;
    e.angles = static_cast<const float2*>(p.angles);
    e.rot_out = static_cast<T*>(p.rot_out);
    e.ld_rot = (long)p.ld_rot;
    return e;
}

int launch_few(hipStream_t stream, const PackedArgs& g, const M40Epilogue<m40_bf16>& e, int batches, int num_cus) {
    const M40FewRows f{static_cast<const m40_bf16*>(g.a), g.w, g.lda, g.a_batch, g.w_batch, g.n_tiles, g.k_tiles, g.rows, g.k_stride, g.k_total, g.segment, batches, g.jobs ? g.rows : 1, g.jobs, g.gather, nullptr};
    return m40_few_rows_product(stream, f, e, num_cus);
}

// gate and up of the experts that a route's ids name; rows = most jobs
int launch_choices(hipStream_t stream, const PackedArgs& g, const M40Epilogue<m40_bf16>& e, const M40llmRoute& q, bool weight_input, int num_cus) {
    const M40FewChoices c{q.ids, q.weight, q.place, q.jobs, (int)q.rows, (int)q.top, (int)q.experts, weight_input};
    const M40FewRows f{static_cast<const m40_bf16*>(g.a), g.w, g.lda, 0, g.w_batch, g.n_tiles, g.k_tiles, 0, g.k_stride, 0, 0, 1, g.rows, nullptr, nullptr, &c};
    return m40_few_rows_product(stream, f, e, num_cus);
}

// one thread per source element
__global__ __launch_bounds__(256) void pack_tiles_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst,
                                                         M40llmPackPlan p, size_t total) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        size_t r = i;
        const uint32_t k = (uint32_t)(r % p.k); r /= p.k;
        const uint32_t kb = (uint32_t)(r % p.k_blocks); r /= p.k_blocks;
        const uint32_t n = (uint32_t)(r % p.n), nb = (uint32_t)(r / p.n);
        const uint32_t row = p.n_offset + nb * p.n_block_pad + n, col = p.k_offset + kb * p.k_block_pad + k;
        const size_t tile = (size_t)(p.tile_first + (row >> 4) * p.tile_stride) * p.k_tiles + (col >> 5);
        dst[tile * kM40Tile + m40_tile_offset(row & 15u, col & 31u)] = src[nb * p.sn_block + n * p.sn + kb * p.sk_block + k * p.sk];
    }
}

__global__ __launch_bounds__(256) void clear_u32_kernel(uint32_t* dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = 0u;
}

__global__ __launch_bounds__(256) void fill_random_bf16_kernel(uint16_t* dst, size_t n, uint64_t seed, float half_range) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        uint64_t z = seed + (i + 1) * 0x9e3779b97f4a7c15ull;        // splitmix64
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        z ^= z >> 31;
        const float u = (float)(uint32_t)(z >> 40) * (2.0f / 16777216.0f) - 1.0f;
        dst[i] = __builtin_bit_cast(uint16_t, static_cast<m40_bf16>(u * half_range));
    }
}

}  // namespace

extern "C" {

int m40llm_ext_fill_random_bf16_async(M40llmCudaContext* ctx, void* d_dst, uint64_t n, uint64_t seed, float std_dev, uint32_t stream_kind) {
    if (!ctx || !d_dst) return -1;
    hipStream_t stream = m40_select_stream(ctx, stream_kind);
    if (!stream || m40_ensure_device(ctx) != 0) return -2;
    if (n == 0) return 0;
    const uint64_t blocks = (n + 255) / 256;
    fill_random_bf16_kernel<<<(unsigned)(blocks < 65536 ? blocks : 65536), 256, 0, stream>>>(static_cast<uint16_t*>(d_dst), (size_t)n, seed,
                                                                                             std_dev * 1.7320508075688772f);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int m40llm_ext_pack_tiles_async(M40llmCudaContext* ctx, const void* d_src, void* d_dst, const M40llmPackPlan* plan, uint32_t stream_kind) {
    if (!ctx || !d_src || !d_dst || !plan) return -1;
    hipStream_t stream = m40_select_stream(ctx, stream_kind);
    if (!stream || m40_ensure_device(ctx) != 0) return -2;
    const M40llmPackPlan& p = *plan;
    const size_t total = (size_t)p.n_blocks * p.n * p.k_blocks * p.k;
    if (total == 0 || p.tile_stride == 0) return -3;
    if (p.k_offset + (uint64_t)(p.k_blocks - 1) * p.k_block_pad + p.k > (uint64_t)p.k_tiles * 32u) return -3;
    const size_t blocks = (total + 255) / 256;
    pack_tiles_kernel<<<(unsigned)(blocks < 65536 ? blocks : 65536), 256, 0, stream>>>(static_cast<const uint16_t*>(d_src),
                                                                                       static_cast<uint16_t*>(d_dst), p, total);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int m40llm_ext_clear_u32_async(M40llmCudaContext* ctx, void* d_dst, size_t n, uint32_t stream_kind) {
    if (!ctx || !d_dst) return -1;
    hipStream_t stream = m40_select_stream(ctx, stream_kind);
    if (!stream || m40_ensure_device(ctx) != 0) return -2;
    if (n == 0) return 0;
    const size_t blocks = (n + 255) / 256;
    clear_u32_kernel<<<(unsigned)(blocks < 4096 ? blocks : 4096), 256, 0, stream>>>(static_cast<uint32_t*>(d_dst), n);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

int m40llm_ext_packed_gemm_async(M40llmCudaContext* ctx, const M40llmPackedGemm* p, uint32_t stream_kind) {
    if (!ctx || !p || !p->a || !p->w) return -1;
    hipStream_t stream = m40_select_stream(ctx, stream_kind);
    if (!stream || m40_ensure_device(ctx) != 0) return -2;
    const bool paged = p->epilogue == M40LLM_PACKED_KEYS || p->epilogue == M40LLM_PACKED_VALUES;
    const M40llmRoute* choices = static_cast<const M40llmRoute*>(p->route);
    if (choices) {
        if (!choices->ids || !choices->weight || !choices->place || !choices->jobs) return -1;
        if (p->jobs || p->gather || p->row_scale || p->act_dtype != M40LLM_ACT_BF16 || p->epilogue != M40LLM_PACKED_PROJECT || p->plain_tiles != 0 || p->batches != 1u || p->k_parts > 1u || p->segment_tiles ||
            m40_route_refused(*choices) || choices->job_rows != 16u || choices->rows * choices->top > 64u || choices->rows > 16u || p->rows < choices->rows || choices->experts > 64u || !m40_aligned16(choices->jobs) ||
            p->w_batch % 8 != 0)
            return -3;
    }
    const uint32_t k_parts = p->k_parts > 1u ? p->k_parts : 1u, part_tiles = (p->k_tiles + k_parts - 1) / k_parts;
    if (p->act_dtype > 1u || p->epilogue > M40LLM_PACKED_CAP || p->activation > M40LLM_LIMITED_GATE || p->rows == 0 || p->batches == 0 || p->batches > 65535u ||
        p->n_tiles == 0 || p->k_tiles == 0 || !m40_aligned16(p->a) || !m40_aligned16(p->w) || p->rows > 0x3fffffffu ||
        (p->batches > 1u && (p->a_batch % 32 != 0 || p->w_batch % 8 != 0)))
        return -3;
    if (p->jobs && (p->batches != 1u || k_parts > 1u || p->max_jobs == 0 || p->max_jobs > 65535u || (p->job_rows != 16u && p->job_rows != 32u && p->job_rows != 64u && p->job_rows != 128u) ||
                    (p->job_rows == 128u && p->act_dtype == M40LLM_ACT_F32) || p->w_batch % 8 != 0 ||
                    !(p->epilogue == M40LLM_PACKED_STORE_ACT ? !p->gather
                                                                  : p->epilogue == M40LLM_PACKED_PROJECT && p->plain_tiles == 0 && (p->job_rows == 128u) == !p->gather)))
        return -3;
    if (!paged && (p->lda % 32 != 0 || p->lda < (uint64_t)p->k_tiles * 32u)) return -3;
    // a workgroup's column tiles lie in one segment
    if (p->segment_tiles && (paged || p->jobs || p->batches != 1u || k_parts > 1u || p->epilogue == M40LLM_PACKED_PROJECT || p->segment_tiles % 16u != 0 || p->a_batch % 32 != 0 ||
                             p->lda < (p->n_tiles - 1u) / p->segment_tiles * p->a_batch + (uint64_t)p->k_tiles * 32u))
        return -3;
    if (k_parts > 1u && (p->epilogue != M40LLM_PACKED_STORE || p->batches != 1u || (k_parts - 1) * part_tiles >= p->k_tiles)) return -3;
    // packed results: whole tiles of columns
    if ((p->epilogue == M40LLM_PACKED_GATED || p->epilogue == M40LLM_PACKED_ROTATE || p->epilogue == M40LLM_PACKED_SILU || p->epilogue == M40LLM_PACKED_SPLIT || p->epilogue == M40LLM_PACKED_TANH ||
         (p->epilogue == M40LLM_PACKED_PROJECT && p->out_act)) &&
        (p->ld_act % 32 != 0 || p->act_col % 4 != 0))
        return -3;
    const bool wide_stores = p->ld_act % 4 == 0 && reinterpret_cast<uintptr_t>(p->out_act) % (p->act_dtype == M40LLM_ACT_F32 ? 16 : 8) == 0;
    switch (p->epilogue) {
        case M40LLM_PACKED_CAP: if (p->batches != 1u || !(p->out_cap >= 0.0f)) return -4; [[fallthrough]];
        case M40LLM_PACKED_STORE: case M40LLM_PACKED_ADD: if (!p->out_f32 || p->cols > p->n_tiles * 16u) return -4; break;
        case M40LLM_PACKED_STORE_ACT: if (!p->out_act || p->cols > p->n_tiles * 16u) return -4; break;
        case M40LLM_PACKED_GATED: if (!p->out_act || !p->gate || p->cols > p->n_tiles * 16u) return -4; break;
        case M40LLM_PACKED_ROTATE:
            if (!p->out_act || !p->angles || p->head_width == 0 || p->head_width % 32 != 0 || p->rot_start % 32 != 0 ||
                p->rot_start >= p->head_width || p->rot_half * 2u != p->head_width - p->rot_start ||
                p->heads * p->head_width != p->n_tiles * 16u || !wide_stores || !m40_aligned16(p->angles) ||
                (p->split_row > 0 && (!p->rot_out || p->ld_rot % 4 != 0 ||
                                      reinterpret_cast<uintptr_t>(p->rot_out) % (p->act_dtype == M40LLM_ACT_F32 ? 16 : 8) != 0)))
                return -4;
            break;
        case M40LLM_PACKED_PROJECT:
            if ((p->plain_tiles > 0 && !p->out_f32) || (p->n_tiles > p->plain_tiles && (!p->out_act || !wide_stores)) ||
                p->plain_tiles % 2 != 0 || p->n_tiles % 2 != 0 || p->plain_tiles > p->n_tiles)
                return -4;
            break;
        case M40LLM_PACKED_SILU: case M40LLM_PACKED_SPLIT: case M40LLM_PACKED_TANH:
            if ((p->plain_tiles > 0 && !p->out_f32) || !p->out_act || !wide_stores || p->plain_tiles > p->n_tiles || p->batches != 1u) return -4;
            break;
        case M40LLM_PACKED_KEYS: case M40LLM_PACKED_VALUES:
            if (!p->out_act || !m40_aligned16(p->out_act) || !p->pages || p->page_k_tiles < p->k_tiles || p->batches != 1u ||
                p->act_dtype != M40LLM_ACT_BF16 || p->rows % M40LLM_PAGE_TOKENS != 0 ||
                (p->epilogue == M40LLM_PACKED_KEYS && p->n_tiles % 2 != 0))
                return -4;
            break;
    }
    PackedArgs g{};
    g.a = p->a;
    g.w = static_cast<const m40_bf16*>(p->w);
    g.lda = (long)p->lda; g.a_batch = (long)p->a_batch * 16; g.w_batch = (long)p->w_batch;
    g.n_tiles = (int)p->n_tiles; g.k_tiles = (int)p->k_tiles; g.rows = (int)p->rows; g.k_stride = (int)p->k_tiles;
    g.pages = p->pages; g.page_k_tiles = (int)p->page_k_tiles;
    g.segment = (int)p->segment_tiles;
    int batches = (int)p->batches;
    if (k_parts > 1u) {
        g.k_total = (int)p->k_tiles; g.k_tiles = (int)part_tiles;
        g.a_batch = (long)part_tiles * kM40Tile; g.w_batch = (long)part_tiles * kM40Tile;
        batches = (int)k_parts;
    }
    (void)hipGetLastError();
    if (choices) {
        g.rows = (int)m40llm_ext_expert_max_jobs(choices->rows, choices->experts, choices->top, 16u);
        return launch_choices(stream, g, make_epilogue<m40_bf16>(*p), *choices, choices->slot_weight != nullptr, ctx->num_cus);
    }
    if (p->jobs) {
        g.jobs = p->jobs; g.gather = p->gather;
        g.rows = (int)p->max_jobs;
        const int rows = (int)p->job_rows;
        if (p->act_dtype == M40LLM_ACT_F32) {
            const M40Epilogue<float> e = make_epilogue<float>(*p);
            return p->gather ? launch_rows_any<float, kJobGather>(stream, g, e, 1, rows, ctx->num_cus) : launch_rows_any<float, kJobSlots>(stream, g, e, 1, rows, ctx->num_cus);
        }
        const M40Epilogue<m40_bf16> e = make_epilogue<m40_bf16>(*p);
        if (rows == 128) return launch_tile_any<kSlots>(stream, g, e, 1, ctx->num_cus);
        if (rows == 16) return launch_few(stream, g, e, 1, ctx->num_cus);
        return p->gather ? launch_rows_any<m40_bf16, kJobGather>(stream, g, e, 1, rows, ctx->num_cus) : launch_rows_any<m40_bf16, kJobSlots>(stream, g, e, 1, rows, ctx->num_cus);
    }
    if (p->act_dtype == M40LLM_ACT_F32) {
        if ((g.rows + 63) / 64 > 65535) return -3;
        return launch_rows_any<float, kAllRows>(stream, g, make_epilogue<float>(*p), batches, g.rows, ctx->num_cus);
    }
    const M40Epilogue<m40_bf16> e = make_epilogue<m40_bf16>(*p);
    if (p->epilogue == M40LLM_PACKED_KEYS) return launch_tile_any<kPageKeys>(stream, g, e, batches, ctx->num_cus);
    if (p->epilogue == M40LLM_PACKED_VALUES) return launch_tile_any<kPageValues>(stream, g, e, batches, ctx->num_cus);
    if (g.rows <= 16) return launch_few(stream, g, e, batches, ctx->num_cus);
    // few columns leave most CUs without a wide tile
    if (g.rows <= 64 || (g.n_tiles <= 8 && batches == 1 && g.rows <= 65535 * 16 && p->epilogue != M40LLM_PACKED_PROJECT)) return launch_rows_any<m40_bf16, kAllRows>(stream, g, e, batches, g.rows, ctx->num_cus);
    return launch_tile_any<kPlainRows>(stream, g, e, batches, ctx->num_cus);
}

}  // extern "C"
