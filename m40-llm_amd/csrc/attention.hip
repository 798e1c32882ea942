// Last-token GQA attention over the dense f16 KV cache for gfx950 (single sequence, device
// length, recent-window and variable-length batched forms share one kernel).
//
// Work split: grid = (kv_head x q-head subgroup, token chunk, batch row).  A workgroup of eight waves
// owns a chunk of 8 * TPW * S token rows (TPW = rows per 64-lane load: 8 at head_dim 64, 4 at 128).
// Every lane issues all of its S K-row and S V-row 128-bit loads before any arithmetic, so a chunk
// costs one memory round trip; the rows serve all G q heads of the subgroup.  Scores stay in
// registers.  With one chunk the kernel writes the output; otherwise it writes the softmax partial
// (max, sum, weighted V) and a second kernel merges the chunks in ascending order.
//
// Reference semantics: three-pass softmax per q head, kv head = qh / (q_heads / kv_heads),
// scale literals for head_dim 64 / 128: cuda/kernels.cu:1367-1655, entry points :3837-4023,
// batched :1740-1823 and :4694-4832.
#include "attention_chunks.hpp"
#include "attention_params.hpp"

#include <atomic>
#include <mutex>
#include <type_traits>

// Fixed chunk-partial buffer of m40llm_ext_attention_last_token_f32_gqa_static_scratch_async: device memory that
// exists from the moment the code object is loaded, so that entry point never allocates.  Every GPU the library
// runs on holds its own copy (at its own address) until the process ends.  In host code the array's name is a
// stand-in, not a device address: host code only ever uses the pointers that hipGetSymbolAddress returned
// (g_static_scratch_ptr), one per device.
constexpr size_t kStaticScratchBytes = 2u << 20;   // 2 MiB
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kStaticScratchMaxDevices = 64;
static std::atomic<float*> g_static_scratch_ptr[kStaticScratchMaxDevices];
static std::mutex g_static_scratch_mutex;
// Who used a device's array last, and an event behind that call's last launch: a call from another context while
// that work is still outstanding is refused (-10) instead of racing.  The event is made with the pointer, at set-up.
struct StaticScratchUse {
    const M40llmCudaContext* owner;
    hipEvent_t done;
    bool have_event, recorded;
};
static StaticScratchUse g_static_scratch_use[kStaticScratchMaxDevices];

int m40_attention_static_scratch_init(int device_id) {
    if (device_id < 0 || device_id >= kStaticScratchMaxDevices) return -2;
    std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
    if (g_static_scratch_ptr[device_id].load(std::memory_order_acquire)) return 0;
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
        (void)hipGetLastError();
        return -4;
    }
    StaticScratchUse& use = g_static_scratch_use[device_id];
    if (!use.have_event) {
        if (hipEventCreateWithFlags(&use.done, hipEventDisableTiming) == hipSuccess) use.have_event = true;
        else (void)hipGetLastError();
    }
    g_static_scratch_ptr[device_id].store(static_cast<float*>(ptr), std::memory_order_release);
    return 0;
}

namespace {

constexpr int kAttnThreads = 512;
constexpr int kWaves = kAttnThreads / 64;


// Steps of a chunk are rows' scores that all lanes of a row hold; lane c goes on with step c % P (P: the steps, rounded up to a power of two), so that a lane works out
// one weight and not all of them, and hands it to the others.  Of eight lanes, step s is in lane s, which quad s / 4 reads itself; in the other quad the mirrored values have it.
template <int... I, class F>
__device__ __forceinline__ void attn_unrolled(std::integer_sequence<int, I...>, F&& f) { (f(std::integral_constant<int, I>{}), ...); }

template <int NS>
__device__ __forceinline__ constexpr int attn_step_mask() { return NS > 4 ? 7 : (NS > 2 ? 3 : NS - 1); }
template <int S, bool EIGHT>
__device__ __forceinline__ float attn_from_step(float own, float mirrored) {
    constexpr int kQuad = (S & 3) * 0x55, kMirror = (3 - (S & 3)) * 0x55, kOther = S & 4 ? 0x5 : 0xa;
    const int here = __builtin_amdgcn_mov_dpp(__float_as_int(own), kQuad, 0xf, 0xf, true);
    return __int_as_float(EIGHT ? __builtin_amdgcn_update_dpp(here, __float_as_int(mirrored), kMirror, 0xf, kOther, false) : here);
}

// HD in {64, 128}; G = q heads per workgroup (<= 4); S = token rows per lane group; PACKED: the result as operands (a launch of one short row has no time to look
// it up: 4.35 us instead of 4.29).
//
// Bound by the vector ALU and a launch's round trips: 32 workgroups of two waves a SIMD, on 32 CUs.  One row of 32 q heads to 4 kv of 64, sized for 512 tokens, us in a
// recorded chain over caches that no cache holds, before / with the kv heads in turn / columns halved in the join, lane groups joined once, clamped loads without a branch /
// and as many steps as there are: 64 tokens 3.73 / 3.73 / 3.9 / 2.55; 128 4.22 / 3.73 / 3.9 / 2.73; 256 4.53 / 3.89 / 3.9 / 3.11; 512 5.23 / 4.97 / 4.49 / 4.50.
// 16 q heads to 2 of 128, 256 tokens 5.05 -> 4.56; 32 to 8 5.11 -> 4.53.
// With a weight worked out by one lane a row instead of by all, and six and three steps beside eight, four, two and one, us a step of 8 tokens, before / now: TinyLlama, one row of 310
// 822 / 812, of 490 836 / 826, four of 310 835 / 823, eight 879 / 844; Qwen2.5-3B, one row of 200 1854 / 1836.  Then with scalar addresses, a third fewer instructions: eight rows of 490
// 878 / 863, others as they were (and 855 instead of 840 with eight of 310 where V's requests may go out between K's, or must be out before the first product).
//
// WIDE: offsets from a step's address in 64 bits, for more kv heads than 32 bits have room for (kMostNarrowHeads).
template <int HD, int G, int S, bool PACKED, bool WIDE = false>
__global__ __launch_bounds__(kAttnThreads, 2) void attn_partial_kernel(AttnParams p) {
    using Offset = std::conditional_t<WIDE, size_t, uint32_t>;
    constexpr int LPT = HD / 8;      // lanes per token row
    constexpr int TPW = 64 / LPT;    // token rows per wave load
    constexpr uint32_t kChunk = kWaves * TPW * S;
    __shared__ __attribute__((aligned(16))) float red[kWaves][G][HD];
    __shared__ float wmax[kWaves][G];
    __shared__ float wsum[kWaves][G];

    // Neighbouring workgroups take the kv heads in turn: with 2, 4 or 8 of them a die of the eight then reads the rows of one, not of all, for its heads
    const uint32_t kvh = blockIdx.x % p.kv_heads, sub = blockIdx.x / p.kv_heads;
    const uint32_t group = p.q_heads / p.kv_heads;
    const uint32_t qh0 = kvh * group + sub * G;          // first q head of this workgroup
    const uint32_t gcount = (sub * G + G <= group) ? G : group - sub * G;
    const uint32_t b = blockIdx.z;
    const uint32_t seq_id = p.seq_ids_dev ? p.seq_ids_dev[b] : p.seq_id;
    const uint32_t len = p.length(b);
    if (len == 0 || len > p.max_seq_len) return;
    if (p.max_batch != 0 && seq_id >= p.max_batch) return;
    const uint32_t t0 = (p.window != 0 && len > p.window) ? len - p.window : 0;
    if (len - t0 > p.span_limit) return;      // longer than the launch was sized for: the row is skipped
    const uint32_t cbeg = t0 + blockIdx.y * kChunk;
    if (cbeg >= len) return;
    const uint32_t cend = cbeg + kChunk < len ? cbeg + kChunk : len;

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int c = lane % LPT, tg = lane / LPT;
    const Offset row_bytes = (Offset)p.kv_heads * (HD * 2u);
    const uint32_t row = (uint32_t)(wave * TPW + tg);
    const size_t base = ((size_t)seq_id * p.max_seq_len + cbeg) * row_bytes + (size_t)kvh * (2 * HD);
    const uint8_t* Kb = reinterpret_cast<const uint8_t*>(p.K) + base;
    const uint8_t* Vb = reinterpret_cast<const uint8_t*>(p.V) + base;
    const float inv_sqrt = HD == 64 ? 0.125f : 0.08838834764831845f;

    float mh[G], lsum[G], acc[G][8];
    // One pass over the chunk's rows, with as many steps as they fill, five and seven rounded up: a recorded step is sized for more tokens than its row has by
    // now, and arithmetic on rows that are not there took 1.1 us of 3.7.  A test at each step instead keeps the steps of a full chunk from overlapping (5.2 -> 5.5).
    const auto pass = [&](auto n_steps) __attribute__((always_inline)) {
        constexpr int NS = decltype(n_steps)::value;
        constexpr int kSure = NS == 8 ? 6 : (NS == 6 ? 4 : NS - 1);      // of fewer steps' rows this pass is not taken
        // every load of this lane, issued before anything waits on memory: scalar addresses that walk the steps, and of a lane an offset that does not change
        float q[G][8];
#pragma unroll
        for (int h = 0; h < G; ++h) {
            const uint32_t qh = qh0 + (h < (int)gcount ? h : 0);
            const float* qp = p.Q + ((size_t)b * p.q_heads + qh) * HD + 8 * c;
            const float4 q0 = *reinterpret_cast<const float4*>(qp);
            const float4 q1 = *reinterpret_cast<const float4*>(qp + 4);
            q[h][0] = q0.x; q[h][1] = q0.y; q[h][2] = q0.z; q[h][3] = q0.w;
            q[h][4] = q1.x; q[h][5] = q1.y; q[h][6] = q1.z; q[h][7] = q1.w;
        }
        __builtin_amdgcn_sched_barrier(0);
        uint4 kw[NS], vw[NS];
        bool valid[NS];
        Offset off[NS];
        const size_t step_bytes = (size_t)(kWaves * TPW) * row_bytes;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint32_t r = (uint32_t)(s * kWaves * TPW) + row, last = cend - 1u - cbeg;
            valid[s] = s < kSure || r <= last;
            off[s] = s < kSure ? row * row_bytes + 16u * c : ((valid[s] ? r : last) - (uint32_t)(kSure * kWaves * TPW)) * row_bytes + 16u * c;
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) kw[s] = *reinterpret_cast<const uint4*>(Kb + (s < kSure ? s : kSure) * step_bytes + off[s]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < NS; ++s) vw[s] = *reinterpret_cast<const uint4*>(Vb + (s < kSure ? s : kSure) * step_bytes + off[s]);

        // ---- scores (every lane of a row group ends up with the row's score) -----------------------
        const int own_step = c & attn_step_mask<NS>();
        const bool own_valid = cbeg + (uint32_t)(own_step * kWaves * TPW) + row < cend && own_step < NS;
        float own[G], mirrored[G];
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float x = 0.0f;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                float kf[8], d = 0.0f;
                m40_unpack8(kw[s], kf);
#pragma unroll
                for (int j = 0; j < 8; ++j) d = fmaf(q[h][j], kf[j], d);
                d = LPT == 8 ? m40_sum8(d) : m40_sum16(d);
                x = s == 0 || own_step == s ? d : x;
            }
            own[h] = own_valid ? x * inv_sqrt : -INFINITY;
        }
#pragma unroll
        for (int h = 0; h < G; ++h) {
            const float m = NS == 1 ? m40_max_lanes_from<LPT>(own[h]) : m40_max64(own[h]);          // (of one step all lanes of a row have the score)
            if (lane == 0) wmax[wave][h] = m;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float m = wmax[0][h];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) m = fmaxf(m, wmax[w][h]);
            mh[h] = m;
        }

        // ---- exp, row sums, weighted V -----------------------------------------------------------
#pragma unroll
        for (int h = 0; h < G; ++h) {
            lsum[h] = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[h][j] = 0.0f;
            own[h] = own_valid ? expf(own[h] - mh[h]) : 0.0f;
            mirrored[h] = m40_dpp_f<M40_DPP_HALF_MIRROR>(own[h]);
        }
        attn_unrolled(std::make_integer_sequence<int, NS>(), [&](auto s_c) __attribute__((always_inline)) {
            constexpr int s = decltype(s_c)::value;
            float vf[8];
            if (s >= kSure) {      // the last row once more: an infinity there counts once
                const uint32_t keep = valid[s] ? ~0u : 0u;
                vw[s] = make_uint4(vw[s].x & keep, vw[s].y & keep, vw[s].z & keep, vw[s].w & keep);
            }
            m40_unpack8(vw[s], vf);
#pragma unroll
            for (int h = 0; h < G; ++h) {
                const float e = NS == 1 ? own[h] : attn_from_step<s, (NS > 4)>(own[h], mirrored[h]);
                lsum[h] += e;
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[h][j] = fmaf(e, vf[j], acc[h][j]);
            }
        });
    };
    const uint32_t steps = (cend - cbeg + kWaves * TPW - 1) / (kWaves * TPW);
    const auto at_most = [&](auto n_steps) __attribute__((always_inline)) {
        constexpr int NS = decltype(n_steps)::value;
        if (NS > S || steps > NS) return false;
        pass(std::integral_constant<int, NS <= S ? NS : S>());
        return true;
    };
    at_most(std::integral_constant<int, 1>()) || at_most(std::integral_constant<int, 2>()) || at_most(std::integral_constant<int, 3>()) || at_most(std::integral_constant<int, 4>()) ||
        at_most(std::integral_constant<int, 6>()) || at_most(std::integral_constant<int, 8>());

    // Join the TPW token rows of the wave (lanes with equal c): each exchange leaves a lane half of the columns to go on with, at the end two of its eight.
#pragma unroll
    for (int h = 0; h < G; ++h) {
        float* a = acc[h];
        if (LPT == 8) {
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] += m40_dpp_f<M40_DPP_ROW_ROR8>(a[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            m40_swap_rows16(a[j], a[j + 4]);
            a[j] += a[j + 4];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            m40_swap_rows32(a[j], a[j + 2]);
            a[j] += a[j + 2];
        }
        const float ssum = m40_sum_lanes_from<LPT>(lsum[h]);
        if (lane == 0) wsum[wave][h] = ssum;
        if (LPT == 16 || (lane & 8) == 0) *reinterpret_cast<float2*>(&red[wave][h][8 * c + ((lane & 16) >> 2) + ((lane & 32) >> 4)]) = make_float2(a[0], a[1]);
    }
    __syncthreads();

    const bool final_out = p.nchunks == 1;
    for (uint32_t e = tid; e < gcount * HD; e += kAttnThreads) {
        const uint32_t h = e / HD, d = e % HD;
        float v = 0.0f, l = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            v += red[w][h][d];
            l += wsum[w][h];
        }
        const uint32_t qh = qh0 + h;
        if (final_out) {
            const float denom = l > 0.0f ? l : 1.0f;
            if constexpr (PACKED) m40_attn_store<HD>(p, b, qh, d, v / denom);
            else static_cast<float*>(p.out)[((size_t)b * p.q_heads + qh) * HD + d] = v / denom;
        } else {
            const size_t at = ((size_t)b * p.q_heads + qh) * p.nchunks + blockIdx.y;
            p.ws[at * HD + d] = v;
            if (d == 0) p.ml()[at] = make_float2(mh[h], l);
        }
    }
}

// Merge chunk partials: grid (q_heads, batch), 256 threads
template <int HD, int PASS>
__global__ __launch_bounds__(256) void attn_combine_kernel(AttnParams p) {
    __shared__ __attribute__((aligned(16))) float sums[4][HD];
    const uint32_t qh = blockIdx.x, b = blockIdx.y;
    const size_t first = ((size_t)b * p.q_heads + qh) * p.nchunks;
    M40ChunkMerge<HD, PASS> merge;
    merge.request(p.ws + first * HD, p.ml() + first, p.nchunks);
    const uint32_t len = p.length(b);
    const uint32_t sid = (p.max_batch != 0 && p.seq_ids_dev) ? p.seq_ids_dev[b] : 0u;
    if (len == 0 || len > p.max_seq_len) return;
    if (p.max_batch != 0 && p.seq_ids_dev && sid >= p.max_batch) return;
    const uint32_t t0 = (p.window != 0 && len > p.window) ? len - p.window : 0;
    if (len - t0 > p.span_limit) return;      // longer than the launch was sized for: the row is skipped
    const float y = merge.finish((len - t0 + p.chunk - 1) / p.chunk, sums);
    if (threadIdx.x < HD) m40_attn_store<HD>(p, b, qh, threadIdx.x, y);
}

// Any head_dim: one thread per output element, the reference's three passes verbatim
// (cuda/kernels.cu:1367-1426).  Used for head_dim other than 64 / 128 only.
__global__ __launch_bounds__(64) void attn_generic_kernel(AttnParams p, uint32_t head_dim) {
    const uint32_t b = blockIdx.z, qh = blockIdx.y;
    const uint32_t d = blockIdx.x * 64 + threadIdx.x;
    if (d >= head_dim) return;
    const uint32_t seq_id = p.seq_ids_dev ? p.seq_ids_dev[b] : p.seq_id;
    const uint32_t len = p.length(b);
    if (len == 0 || len > p.max_seq_len) return;
    const uint32_t t0 = (p.window != 0 && len > p.window) ? len - p.window : 0;
    if (len - t0 > p.span_limit) return;      // longer than the launch was sized for: the row is skipped
    const uint32_t kvh = qh / (p.q_heads / p.kv_heads);
    const size_t ept = (size_t)p.kv_heads * head_dim;
    const float inv_sqrt = m40_inv_sqrt_head_dim(head_dim);
    const float* q = p.Q + ((size_t)b * p.q_heads + qh) * head_dim;
    const uint16_t* Kb = p.K + ((size_t)seq_id * p.max_seq_len) * ept + (size_t)kvh * head_dim;
    const uint16_t* Vb = p.V + ((size_t)seq_id * p.max_seq_len) * ept + (size_t)kvh * head_dim;
    float mx = -1e30f;
    for (uint32_t t = t0; t < len; ++t) {
        float dot = 0.0f;
        for (uint32_t k = 0; k < head_dim; ++k) dot += q[k] * m40_h2f(Kb[(size_t)t * ept + k]);
        mx = fmaxf(mx, dot * inv_sqrt);
    }
    float den = 0.0f, acc = 0.0f;
    for (uint32_t t = t0; t < len; ++t) {
        float dot = 0.0f;
        for (uint32_t k = 0; k < head_dim; ++k) dot += q[k] * m40_h2f(Kb[(size_t)t * ept + k]);
        const float e = expf(dot * inv_sqrt - mx);
        den += e;
        acc += e * m40_h2f(Vb[(size_t)t * ept + d]);
    }
    den = den > 0.0f ? den : 1.0f;
    static_cast<float*>(p.out)[((size_t)b * p.q_heads + qh) * head_dim + d] = acc / den;
}

// The last step of a full chunk (six of eight steps have addresses of their own) reads up to 2 * 8 * 512 / HD - 1 rows past its address: 2^14 bytes a kv head
constexpr uint32_t kMostNarrowHeads = 1u << 18;

template <int HD, int G, int S>
void launch_partial(hipStream_t stream, const AttnParams& p, uint32_t batch) {
    dim3 grid(p.kv_heads * p.subgroups, p.nchunks, batch);
    if (p.packed && p.nchunks == 1) attn_partial_kernel<HD, G, S, true><<<grid, kAttnThreads, 0, stream>>>(p);
    else attn_partial_kernel<HD, G, S, false><<<grid, kAttnThreads, 0, stream>>>(p);
}

template <int HD, int G>
void launch_g(hipStream_t stream, const AttnParams& p, uint32_t batch, int S) {
    switch (S) {
        case 8: launch_partial<HD, G, 8>(stream, p, batch); break;
        case 4: launch_partial<HD, G, 4>(stream, p, batch); break;
        case 2: launch_partial<HD, G, 2>(stream, p, batch); break;
        default: launch_partial<HD, G, 1>(stream, p, batch); break;
    }
}

template <int HD>
void launch_combine(hipStream_t stream, const AttnParams& p, uint32_t batch) {
    // What is asked for beyond the chunks there can be is asked for in vain, 32 KB a head of 128 columns.  us a step, 64 chunks / as many as there can be: Qwen2.5-3B, 8 rows of up
    // to 4000 tokens 2147 / 2133, of 600 2061 / 2045, one of 600 1990 / 1978; TinyLlama, 32 of 900 1273 / 1270
    const dim3 grid(p.q_heads, batch);
    if (p.nchunks <= 16) attn_combine_kernel<HD, 16><<<grid, 256, 0, stream>>>(p);
    else if (p.nchunks <= 32) attn_combine_kernel<HD, 32><<<grid, 256, 0, stream>>>(p);
    else attn_combine_kernel<HD, 64><<<grid, 256, 0, stream>>>(p);
}

// Chooses rows per lane group (S), q heads per workgroup (G) and the chunking for a span of `span` tokens.
template <int HD>
int launch_hd(M40llmCudaContext* ctx, hipStream_t stream, float* partial, size_t partial_bytes, bool fixed_chunking,
              AttnParams& p, uint32_t batch, uint32_t group, uint32_t span) {
    constexpr uint32_t kRowsPerStep = kWaves * (64 / (HD / 8));   // token rows one workgroup covers per S
    // Rows of up to 512 tokens stay on the vector-ALU kernel in batches too.  Its launch grows with the q heads of all rows, the matrix-core kernel's hardly does (us, vector
    // ALU / matrix cores, 512 q heads: 32 to 4 kv of 64, 128 tokens 5.1 / 4.6, 500 tokens 8.8 / 7.8), but q and the weights go into the latter as f16 high and low parts: its
    // errors are 14 to 30 % larger (32 rows of up to 500 tokens 1.16e-7 / 1.36e-7), and an infinite V comes out of it as NaN.
    if (span > 512 && m40_aligned16(p.Q)) {
        // long rows: matrix-core kernel (it reads q with 16-byte loads)
        p.subgroups = (group + 7) / 8;
        const uint64_t groups = (uint64_t)batch * p.kv_heads * p.subgroups;
        // One sequence keeps the larger chunks where its partials of 256 tokens would not fit the fixed buffer: with the context's arena and with that buffer the
        // chunks are the same.
        const size_t need_256 = (size_t)p.q_heads * ((span + 255u) / 256u) * (HD + 2) * sizeof(float);
        uint64_t chunk = m40_attention_chunk(groups, span, (uint32_t)ctx->num_cus, batch > 1 || need_256 <= kStaticScratchBytes);
        for (;;) {
            p.chunk = (uint32_t)chunk;
            p.nchunks = (span + p.chunk - 1) / p.chunk;
            if (p.nchunks == 1 || (size_t)batch * p.q_heads * p.nchunks * (HD + 2) * sizeof(float) <= partial_bytes) break;
            if (fixed_chunking) return -9;   // the caller wants this chunking or none (fixed-size partial buffer)
            chunk *= 2;
        }
        p.ws = partial;
        p.ml_from = (uint32_t)((size_t)batch * p.q_heads * p.nchunks * HD);
        m40_launch_attn_mfma(stream, p, HD, batch);
        if (p.nchunks > 1) {
            launch_combine<HD>(stream, p, batch);
        }
        return 0;
    }
    int G = group >= 4 ? 4 : (group >= 2 ? 2 : 1);
    const uint64_t rows = (uint64_t)batch * p.kv_heads;
    // Short rows are latency-bound, not bandwidth-bound: spread the q heads over more workgroups, down to one head
    // each (K/V of a short row stay in L2, so re-reading them per head costs nothing; measured +3 % on the whole
    // batch-1 token against two heads per workgroup).
    while (span <= 1024 && G > 1 && rows * ((group + G - 1) / G) < 128) G >>= 1;
    p.subgroups = (group + G - 1) / G;
    int S = 8;
    if (span <= kRowsPerStep * 8) {
        // one chunk, no merge launch: the smallest S that covers the span
        S = 1;
        while ((uint32_t)S * kRowsPerStep < span) S <<= 1;
    } else {
        // split until the grid covers the CUs about twice
        while (S > 2 && rows * p.subgroups * ((span + kRowsPerStep * S - 1) / (kRowsPerStep * S)) < 2u * (uint32_t)ctx->num_cus)
            S >>= 1;
    }
    p.chunk = kRowsPerStep * (uint32_t)S;
    p.nchunks = (span + p.chunk - 1) / p.chunk;
    if (p.nchunks > 1) {
        const size_t need = (size_t)batch * p.q_heads * p.nchunks * (HD + 2) * sizeof(float);
        if (need > partial_bytes) {
            if (fixed_chunking) return -9;
            if (S == 8) return -7;
            S = 8;
            p.chunk = kRowsPerStep * 8u;
            p.nchunks = (span + p.chunk - 1) / p.chunk;
            if ((size_t)batch * p.q_heads * p.nchunks * (HD + 2) * sizeof(float) > partial_bytes) return -7;
        }
    }
    p.ws = partial;
    p.ml_from = (uint32_t)((size_t)batch * p.q_heads * p.nchunks * HD);
    if (p.kv_heads > kMostNarrowHeads) {
        const dim3 grid(p.q_heads, p.nchunks, batch);
        if (p.packed && p.nchunks == 1) attn_partial_kernel<HD, 1, 8, true, true><<<grid, kAttnThreads, 0, stream>>>(p);
        else attn_partial_kernel<HD, 1, 8, false, true><<<grid, kAttnThreads, 0, stream>>>(p);
    } else switch (G) {
        case 4: launch_g<HD, 4>(stream, p, batch, S); break;
        case 2: launch_g<HD, 2>(stream, p, batch, S); break;
        default: launch_g<HD, 1>(stream, p, batch, S); break;
    }
    if (p.nchunks > 1) {
        launch_combine<HD>(stream, p, batch);
    }
    return 0;
}

}  // namespace

int m40_launch_dense_attention(M40llmCudaContext* ctx, hipStream_t stream, uint32_t stream_kind,
                               const M40AttnArgs& a) {
    AttnParams p{};
    p.K = a.K; p.V = a.V; p.Q = a.Q;
    p.out = a.packed ? static_cast<void*>(a.packed) : a.Out;
    p.packed = a.packed ? (uint32_t)m40_packed_pad((int)a.batch) : 0u;
    p.seq_ids_dev = a.seq_ids_dev; p.seq_lens_dev = a.seq_lens_dev;
    p.seq_id = a.seq_id; p.len_or_bias = a.seq_lens_dev ? a.len_bias : a.seq_len;
    p.max_seq_len = a.max_seq_len; p.kv_heads = a.kv_heads; p.q_heads = a.q_heads; p.window = a.window;
    p.subgroups = 1;
    p.max_batch = a.max_batch;
    (void)hipGetLastError();
    const uint32_t group = a.q_heads / a.kv_heads;
    uint32_t span = a.max_len_hint;
    if (a.window != 0 && span > a.window) span = a.window;
    if (span == 0) span = 1;
    p.span_limit = span;

    if ((a.head_dim == 64 || a.head_dim == 128) && m40_aligned16(a.Q) && m40_aligned16(a.K) && m40_aligned16(a.V)) {
        M40StreamScratch& scr = ctx->scratch[stream_kind];
        float* partial = a.partial_override ? a.partial_override : static_cast<float*>(scr.attn_partial);
        const size_t partial_bytes = a.partial_override ? a.partial_override_bytes : scr.attn_partial_bytes;
        const bool fixed = a.partial_override != nullptr;
        const int rc = a.head_dim == 64 ? launch_hd<64>(ctx, stream, partial, partial_bytes, fixed, p, a.batch, group, span)
                                        : launch_hd<128>(ctx, stream, partial, partial_bytes, fixed, p, a.batch, group, span);
        if (rc != 0) return rc;
    } else {
        if (a.packed) return -6;
        p.chunk = span; p.nchunks = 1;
        dim3 grid((a.head_dim + 63) / 64, a.q_heads, a.batch);
        attn_generic_kernel<<<grid, 64, 0, stream>>>(p, a.head_dim);
    }
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

// Reads the (ids, lens) pair of a batched call back to the host for validation, as the reference
// does before launching (cuda/kernels.cu:4721-4754); returns the largest length.
// The reference copies both metadata arrays to the host and validates them before it launches (kernels.cu:4723-4754).
// Here the copies are ordered on the decode stream (they see whatever earlier decode-stream work wrote) and land in
// the context's pinned staging words: two asynchronous copies and one wait.
static int validate_batch(M40llmCudaContext* ctx, const M40llmKVCache* kv, const uint32_t* ids_dev,
                          const uint32_t* lens_dev, uint32_t batch, uint32_t* max_len) {
    uint32_t *ids, *lens;
    const bool staged = ctx->host_staging && 2u * batch <= (uint32_t)kM40HostStagingWords;
    if (staged) {
        ids = ctx->host_staging;
        lens = ctx->host_staging + batch;
    } else {
        ids = new uint32_t[batch];
        lens = new uint32_t[batch];
    }
    int rc = 0;
    if (hipMemcpyAsync(lens, lens_dev, (size_t)batch * 4, hipMemcpyDeviceToHost, ctx->decode_stream) != hipSuccess ||
        hipMemcpyAsync(ids, ids_dev, (size_t)batch * 4, hipMemcpyDeviceToHost, ctx->decode_stream) != hipSuccess ||
        hipStreamSynchronize(ctx->decode_stream) != hipSuccess) {
        (void)hipGetLastError();
        rc = -7;
    }
    uint32_t mx = 0;
    for (uint32_t i = 0; rc == 0 && i < batch; ++i) {
        if (ids[i] >= kv->max_batch_size) rc = -8;
        else if (lens[i] == 0 || lens[i] > kv->max_seq_len) rc = -8;
        else if (lens[i] > mx) mx = lens[i];
    }
    if (!staged) { delete[] ids; delete[] lens; }
    *max_len = mx;
    return rc;
}

extern "C" {

int m40llm_attention_last_token_f32_gqa_async(M40llmCudaContext* ctx, const M40llmKVCache* kv, uint32_t seq_id,
                                              const void* q_dev_f32, uint32_t q_heads, uint32_t seq_len,
                                              void* out_dev_f32) {
    if (!ctx || !kv || !q_dev_f32 || !out_dev_f32) return -1;
    if (seq_id >= kv->max_batch_size) return -2;
    if (seq_len == 0 || seq_len > kv->max_seq_len) return -3;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -6;
    if (!kv->d_k || !kv->d_v) return -4;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = 1; a.seq_id = seq_id; a.seq_len = seq_len;
    a.max_len_hint = seq_len;
    return m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a);
}

// m40llm_attention_last_token_f32_gqa_async for callers that cannot allocate (HIP graph capture, serving loops and
// harnesses that forbid hipMalloc): same checks, kernels, chunking and results, but the chunk partials of a long
// row go into this device's copy of the fixed 2 MiB array above instead of the context's arena.  Calls nothing that
// allocates.  -9: the partials of this (q_heads, head_dim, seq_len) do not fit the fixed buffer.  All calls on one
// GPU share that buffer (every partial a call reads it has written itself, so nothing needs clearing between
// calls).  Calls of one context are ordered on its decode stream; a call from another context while the last user's
// work is still outstanding returns -10 (busy) instead of racing.  Under stream capture no event can be queried, so
// captured calls are not guarded: replays that overlap on one GPU race.
int m40llm_ext_attention_last_token_f32_gqa_static_scratch_async(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                                 uint32_t seq_id, const void* q_dev_f32,
                                                                 uint32_t q_heads, uint32_t seq_len,
                                                                 void* out_dev_f32) {
    if (!ctx || !kv || !q_dev_f32 || !out_dev_f32) return -1;
    if (seq_id >= kv->max_batch_size) return -2;
    if (seq_len == 0 || seq_len > kv->max_seq_len) return -3;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -6;
    if (!kv->d_k || !kv->d_v) return -4;
    if (ctx->device_id < 0 || ctx->device_id >= kStaticScratchMaxDevices) return -4;
    float* ptr = g_static_scratch_ptr[ctx->device_id].load(std::memory_order_acquire);
    if (!ptr) {
        // a context made before this translation unit could resolve the symbol: resolve it now, on the context's device
        if (m40_ensure_device(ctx) != 0 || m40_attention_static_scratch_init(ctx->device_id) != 0) return -4;
        ptr = g_static_scratch_ptr[ctx->device_id].load(std::memory_order_acquire);
    }
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->decode_stream, &capture) != hipSuccess) { (void)hipGetLastError(); capture = hipStreamCaptureStatusNone; }
    const bool guarded = capture == hipStreamCaptureStatusNone;
    std::unique_lock<std::mutex> lock(g_static_scratch_mutex, std::defer_lock);
    StaticScratchUse& use = g_static_scratch_use[ctx->device_id];
    if (guarded) {
        lock.lock();
        if (use.owner && use.owner != ctx && use.have_event && use.recorded) {
            const hipError_t q = hipEventQuery(use.done);
            if (q == hipErrorNotReady) return -10;
            if (q != hipSuccess) (void)hipGetLastError();
        }
    }
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = 1; a.seq_id = seq_id; a.seq_len = seq_len;
    a.max_len_hint = seq_len;
    a.partial_override = ptr;
    a.partial_override_bytes = kStaticScratchBytes;
    const int rc = m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a);
    if (guarded && rc == 0 && use.have_event) {
        use.owner = ctx;
        use.recorded = hipEventRecord(use.done, ctx->decode_stream) == hipSuccess;
        if (!use.recorded) (void)hipGetLastError();
    }
    return rc;
}

int m40llm_attention_last_token_f32_gqa(M40llmCudaContext* ctx, const M40llmKVCache* kv, uint32_t seq_id,
                                        const void* q_dev_f32, uint32_t q_heads, uint32_t seq_len,
                                        void* out_dev_f32) {
    int rc = m40llm_attention_last_token_f32_gqa_async(ctx, kv, seq_id, q_dev_f32, q_heads, seq_len, out_dev_f32);
    if (rc != 0) return rc;
    return hipStreamSynchronize(ctx->decode_stream) == hipSuccess ? 0 : -5;
}

// MHA form: q heads == kv heads (cuda/kernels.cu:3837-3861), synchronous.
int m40llm_attention_last_token_f32(M40llmCudaContext* ctx, const M40llmKVCache* kv, uint32_t seq_id,
                                    const void* q_dev_f32, uint32_t seq_len, void* out_dev_f32) {
    if (!ctx || !kv || !q_dev_f32 || !out_dev_f32) return -1;
    if (seq_id >= kv->max_batch_size) return -2;
    if (seq_len == 0 || seq_len > kv->max_seq_len) return -3;
    if (!kv->d_k || !kv->d_v || kv->num_heads == 0) return -4;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = kv->num_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = 1; a.seq_id = seq_id; a.seq_len = seq_len;
    a.max_len_hint = seq_len;
    int rc = m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a);
    if (rc != 0) return -4;
    return hipStreamSynchronize(ctx->decode_stream) == hipSuccess ? 0 : -5;
}

int m40llm_attention_last_token_f32_gqa_seq_len_dev_async(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                          uint32_t seq_id, const void* q_dev_f32,
                                                          uint32_t q_heads, const uint32_t* seq_len_dev,
                                                          void* out_dev_f32) {
    if (!ctx || !kv || !q_dev_f32 || !seq_len_dev || !out_dev_f32) return -1;
    if (seq_id >= kv->max_batch_size) return -2;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -3;
    if (!kv->d_k || !kv->d_v) return -4;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = 1; a.seq_id = seq_id; a.seq_len = 0;
    a.seq_lens_dev = seq_len_dev;            // row 0 of a one-row batch
    a.max_len_hint = kv->max_seq_len;        // the length is unknown on the host: size for the maximum
    return m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a);
}

// Extension: the sequence length is (*position_dev + 1); max_len_hint bounds it and sizes the grid.
int m40llm_ext_attention_last_token_f32_gqa_position_dev_async(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                               uint32_t seq_id, const void* q_dev_f32,
                                                               uint32_t q_heads, const uint32_t* position_dev,
                                                               uint32_t max_len_hint, void* out_dev_f32) {
    if (!ctx || !kv || !q_dev_f32 || !position_dev || !out_dev_f32) return -1;
    if (seq_id >= kv->max_batch_size) return -2;
    if (max_len_hint == 0 || max_len_hint > kv->max_seq_len) return -3;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -6;
    if (!kv->d_k || !kv->d_v) return -4;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = 1; a.seq_id = seq_id; a.seq_len = 0;
    a.seq_lens_dev = position_dev; a.len_bias = 1; a.max_len_hint = max_len_hint;
    return m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a);
}

int m40llm_attention_last_token_f32_gqa_dense_recent_async(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                           uint32_t seq_id, const void* q_dev_f32,
                                                           uint32_t q_heads, uint32_t seq_len,
                                                           uint32_t recent_window, void* out_dev_f32) {
    if (!ctx || !kv || !q_dev_f32 || !out_dev_f32) return -1;
    if (seq_id >= kv->max_batch_size) return -2;
    if (seq_len == 0 || seq_len > kv->max_seq_len) return -3;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -4;
    if (kv->head_dim != 64 && kv->head_dim != 128) return -5;
    if (recent_window == 0) return -6;
    if (!kv->d_k || !kv->d_v) return -7;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = 1; a.seq_id = seq_id; a.seq_len = seq_len;
    a.max_len_hint = seq_len; a.window = recent_window;
    return m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a) == 0 ? 0 : -7;
}

static int batched_impl(M40llmCudaContext* ctx, const M40llmKVCache* kv, const uint32_t* seq_ids_dev,
                        const uint32_t* seq_lens_dev, uint32_t batch_size, const void* q_dev_f32,
                        uint32_t q_heads, void* out_dev_f32, bool synchronize) {
    if (!ctx || !kv || !seq_ids_dev || !seq_lens_dev || !q_dev_f32 || !out_dev_f32) return -1;
    if (batch_size == 0) return -2;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -3;
    if (kv->head_dim != 64 && kv->head_dim != 128) return -6;
    if (!kv->d_k || !kv->d_v) return -6;
    uint32_t max_len = 0;
    int rc = validate_batch(ctx, kv, seq_ids_dev, seq_lens_dev, batch_size, &max_len);
    if (rc != 0) return rc;
    if (max_len == 0) return -8;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = batch_size;
    a.seq_ids_dev = seq_ids_dev; a.seq_lens_dev = seq_lens_dev; a.max_len_hint = max_len;
    rc = m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a);
    if (rc != 0) return -4;
    if (synchronize && hipStreamSynchronize(ctx->decode_stream) != hipSuccess) return -5;
    return 0;
}

// Row-batched attention whose ids / lengths stay on the device: nothing is copied back for validation; rows whose
// id or length (+ len_bias) is out of range are skipped by the kernel.  max_len_hint bounds every row's length.
static int batched_lens_dev(M40llmCudaContext* ctx, const M40llmKVCache* kv, const uint32_t* seq_ids_dev, const uint32_t* seq_lens_dev, uint32_t len_bias,
                            uint32_t batch_size, uint32_t max_len_hint, const void* q_dev_f32, uint32_t q_heads, void* out_dev_f32, void* packed_dev) {
    if (!ctx || !kv || !seq_ids_dev || !seq_lens_dev || !q_dev_f32 || (!out_dev_f32 && !packed_dev)) return -1;
    if (batch_size == 0) return -2;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -3;
    if (kv->head_dim != 64 && kv->head_dim != 128) return -6;
    if (!kv->d_k || !kv->d_v) return -6;
    if (max_len_hint == 0 || max_len_hint > kv->max_seq_len) return -8;
    M40AttnArgs a{};
    a.K = kv->d_k; a.V = kv->d_v; a.max_seq_len = kv->max_seq_len; a.kv_heads = kv->num_heads;
    a.head_dim = kv->head_dim; a.q_heads = q_heads; a.Q = static_cast<const float*>(q_dev_f32);
    a.Out = static_cast<float*>(out_dev_f32); a.batch = batch_size;
    a.packed = static_cast<uint8_t*>(packed_dev);
    a.seq_ids_dev = seq_ids_dev; a.seq_lens_dev = seq_lens_dev; a.len_bias = len_bias; a.max_len_hint = max_len_hint;
    a.max_batch = kv->max_batch_size;
    return m40_launch_dense_attention(ctx, ctx->decode_stream, 1, a) == 0 ? 0 : -4;
}

int m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_async(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                                   const uint32_t* seq_ids_dev,
                                                                   const uint32_t* seq_lens_dev, uint32_t len_bias,
                                                                   uint32_t batch_size, uint32_t max_len_hint,
                                                                   const void* q_dev_f32, uint32_t q_heads,
                                                                   void* out_dev_f32) {
    return batched_lens_dev(ctx, kv, seq_ids_dev, seq_lens_dev, len_bias, batch_size, max_len_hint, q_dev_f32, q_heads, out_dev_f32, nullptr);
}

int m40llm_ext_attention_last_token_f32_gqa_batched_lens_dev_packed_async(M40llmCudaContext* ctx, const M40llmKVCache* kv, const uint32_t* seq_ids_dev,
                                                                          const uint32_t* seq_lens_dev, uint32_t len_bias, uint32_t batch_size,
                                                                          uint32_t max_len_hint, const void* q_dev_f32, uint32_t q_heads, void* packed_dev) {
    if (!ctx || !kv || !seq_ids_dev || !seq_lens_dev || !q_dev_f32 || !packed_dev) return -1;
    if (batch_size == 0) return -2;
    if (q_heads == 0 || kv->num_heads == 0 || q_heads % kv->num_heads != 0) return -3;
    const uint64_t K = (uint64_t)q_heads * kv->head_dim;
    const size_t bytes = K <= 0x7fffffffu ? m40llm_ext_packed_rows_bytes(batch_size, (int)K) : 0;
    if (bytes == 0 || !m40_aligned16(packed_dev) || !m40_aligned16(q_dev_f32) || !m40_apart(q_dev_f32, (size_t)batch_size * K * 4, packed_dev, bytes)) return -6;
    return batched_lens_dev(ctx, kv, seq_ids_dev, seq_lens_dev, len_bias, batch_size, max_len_hint, q_dev_f32, q_heads, nullptr, packed_dev);
}

int m40llm_attention_last_token_f32_gqa_batched(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                const uint32_t* seq_ids_dev, const uint32_t* seq_lens_dev,
                                                uint32_t batch_size, const void* q_dev_f32, uint32_t q_heads,
                                                void* out_dev_f32) {
    return batched_impl(ctx, kv, seq_ids_dev, seq_lens_dev, batch_size, q_dev_f32, q_heads, out_dev_f32, true);
}

int m40llm_attention_last_token_f32_gqa_batched_async(M40llmCudaContext* ctx, const M40llmKVCache* kv,
                                                      const uint32_t* seq_ids_dev, const uint32_t* seq_lens_dev,
                                                      uint32_t batch_size, const void* q_dev_f32,
                                                      uint32_t q_heads, void* out_dev_f32) {
    return batched_impl(ctx, kv, seq_ids_dev, seq_lens_dev, batch_size, q_dev_f32, q_heads, out_dev_f32, false);
}

}  // extern "C"
