// Residual streams: the end of one sublayer and the beginning of the next in one launch.  Every stream becomes a mixture of all old ones plus
// its share of the sublayer's output, and what the next sublayer reads is a weighted sum of the new streams, normed.
#include "norm_route.hpp"
#include "sublayer_rows.hpp"

namespace {

constexpr int kThreads = 256;

template <class T, int S, bool VEC>
__global__ __launch_bounds__(kThreads) void stream_update_kernel(M40llmStreamUpdate a) {
    __shared__ float scratch[kThreads / 64];
    const uint32_t row = a.row_index ? a.row_index[blockIdx.x] : m40_tile_row(blockIdx.x, a.rows);
    m40_stream_update_row<T, S, VEC>(a, row, threadIdx.x, scratch, [&](uint32_t g, const m40_float4& lo, const m40_float4& hi) { m40_store_input<T>(a, row, g, lo, hi); });
}

template <class T, int S>
void launch(hipStream_t stream, const M40llmStreamUpdate& a, bool vec) {
    if (vec) stream_update_kernel<T, S, true><<<a.rows, kThreads, 0, stream>>>(a);
    else stream_update_kernel<T, S, false><<<a.rows, kThreads, 0, stream>>>(a);
}
template <class T>
void launch_any(hipStream_t stream, const M40llmStreamUpdate& a, bool vec) {
    switch (a.streams) {
        case 1: return launch<T, 1>(stream, a, vec);
        case 2: return launch<T, 2>(stream, a, vec);
        case 3: return launch<T, 3>(stream, a, vec);
        case 4: return launch<T, 4>(stream, a, vec);
        default: return a.streams <= 8u ? launch<T, 8>(stream, a, vec) : launch<T, 16>(stream, a, vec);
    }
}

}  // namespace

extern "C" int m40llm_ext_stream_update_async(M40llmCudaContext* ctx, const M40llmStreamUpdate* u, uint32_t stream_kind) {
    if (!ctx || !u || (!u->x0 && !u->streams_x) || (u->w ? !u->h || !u->take : !u->x_out)) return -1;
    hipStream_t stream = m40_select_stream(ctx, stream_kind);
    if (!stream || m40_ensure_device(ctx) != 0) return -2;
    const bool write = u->place || u->n_planes;
    if (u->act_dtype > 1u || u->rows == 0 || u->width == 0 || u->streams == 0 || u->streams > M40LLM_MOST_STREAMS ||
        (u->w && (u->ld_h < u->width || u->ld_h % 32u != 0 || !m40_aligned16(u->h) || (u->h_rows && !m40_aligned16(u->h_rows)))))
        return -3;
    if (u->row_index && u->w) return -4;           // rows of h are those of the step
    if (write && (!u->streams_x || !u->mix || !u->share || (u->place ? !u->expert_out || u->top == 0 : !u->planes))) return -4;
    const bool vec = u->width % 8u == 0 && u->stream_stride % 4u == 0 && m40_aligned16(u->streams_x) && (!u->w || m40_aligned16(u->w)) && (!u->x0 || m40_aligned16(u->x0)) && (!u->x_out || m40_aligned16(u->x_out)) &&
                     (u->place ? u->ld_expert % 8u == 0 && m40_aligned16(u->expert_out) : u->plane_stride % 4u == 0 && (!u->n_planes || m40_aligned16(u->planes)));
    (void)hipGetLastError();
    if (u->route) {
        const M40llmRoute* q = static_cast<const M40llmRoute*>(u->route);
        if (!q->ids || !q->weight || !q->rows_of || !q->place || !q->jobs) return -1;
        if (!vec || !u->w || m40_route_refused(*q)) return -3;
        return m40_stream_update_route(stream, *u);
    }
    if (u->act_dtype == M40LLM_ACT_F32) launch_any<float>(stream, *u, vec);
    else launch_any<m40_bf16>(stream, *u, vec);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}
