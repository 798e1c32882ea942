// The end of one sublayer and the beginning of the next for one row, 256 threads of a workgroup: norm and residual add of layers with the norm on the output
// (sublayer_ops.hip), residual streams (stream_ops.hip); norm_route.hip has the router behind either.
#pragma once

#include "packed_gemm.hpp"

constexpr uint32_t kM40RowThreads = 256;

// Over 256 threads, whose waves' sums are added in order; once a row, which therefore has as many barriers as this has: waves with other work meet a row's at that many (norm_route.hip)
constexpr int kM40RowBarriers = 1;
__device__ __forceinline__ float m40_row_sum(float v, uint32_t tid, float* scratch) {
    v = m40_sum64(v);
    if ((tid & 63u) == 0u) scratch[tid >> 6] = v;
    __syncthreads();
    float s = scratch[0];
#pragma unroll
    for (uint32_t i = 1; i < kM40RowThreads / 64u; ++i) s += scratch[i];
    return s;
}
template <class T, bool VEC>
__device__ __forceinline__ void m40_load_group(const T* src, uint32_t at, uint32_t width, float (&v)[8]) {
    if (VEC) {
        const typename M40Act<T>::vec8 t = M40Act<T>::load8(src + at);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = M40Act<T>::to(t[i]);
    } else {
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) v[i] = at + i < width ? M40Act<T>::to(src[at + i]) : 0.0f;
    }
}
template <bool VEC>
__device__ __forceinline__ void m40_store_group(float* dst, uint32_t at, uint32_t width, const float (&v)[8]) {
    if (VEC) {
        reinterpret_cast<float4*>(dst + at)[0] = make_float4(v[0], v[1], v[2], v[3]);
        reinterpret_cast<float4*>(dst + at)[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i)
            if (at + i < width) dst[at + i] = v[i];
    }
}
// the next sublayer's input: eight columns of a row, packed and (where wanted) plain
template <class T, class A>
__device__ __forceinline__ void m40_store_input(const A& a, uint32_t row, uint32_t g, const m40_float4& lo, const m40_float4& hi) {
    m40_store8<T>(static_cast<T*>(a.h) + m40_packed_at(row, g * 8u, a.ld_h >> 5), lo, hi);
    if (a.h_rows) m40_store8<T>(static_cast<T*>(a.h_rows) + (size_t)row * a.ld_h + g * 8u, lo, hi);
}

// A thread takes groups of eight neighbouring elements and keeps two of them in registers (width up to 4096); beyond, sums are formed again.
// sink(g, low, high): the columns 8 g .. 8 g + 7 of the input.
template <class T, bool VEC, class Sink>
__device__ __forceinline__ void m40_norm_add_row(const M40llmNormAdd& a, uint32_t row, uint32_t tid, float* scratch, const Sink& sink) {
    constexpr uint32_t kGroups = 2;
    const uint32_t width = a.width, groups = a.ld_h / 8u;
    float* x = static_cast<float*>(a.x) + (size_t)row * width;
    const float* w = static_cast<const float*>(a.w);
    // Planes two at a time: one by one each waited for the one before (a row of 2048, planes that the launch before wrote, with that launch: two 4.23 -> 4.00 us, three 4.52 -> 4.31).  Experts' rows one by
    // one: four at a time they are 0.5 to 3 % slower (four of a row of 2048 4.91 / 5.01).
    auto value = [&](uint32_t g, const float (&old)[8], float (&y)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = 0.0f;
        if (g * 8u >= width) return;
        if (a.place) {
            for (uint32_t j = 0; j < a.top; ++j) {
                const uint32_t at = a.place[(size_t)row * a.top + j];
                const float f = static_cast<const float*>(a.weight)[(size_t)row * a.top + j];
                float v[8];
                if (at == M40LLM_PLACE_INPUT) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = old[i];
                } else {
                    m40_load_group<T, VEC>(static_cast<const T*>(a.expert_out) + (size_t)at * a.ld_expert, g * 8u, width, v);
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = fmaf(f, v[i], y[i]);
            }
        } else {
            const float* plane = static_cast<const float*>(a.planes) + (size_t)row * width;
            uint32_t p = 0;
            for (; p + 1u < a.n_planes; p += 2u) {
                float v[2][8];
                m40_load_group<float, VEC>(plane + p * (size_t)a.plane_stride, g * 8u, width, v[0]);
                m40_load_group<float, VEC>(plane + (p + 1u) * (size_t)a.plane_stride, g * 8u, width, v[1]);
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = (y[i] + v[0][i]) + v[1][i];
            }
            if (p < a.n_planes) {
                float v[8];
                m40_load_group<float, VEC>(plane + p * (size_t)a.plane_stride, g * 8u, width, v);
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] += v[i];
            }
        }
    };
    // a row's old values and the weights, requested ahead of the sums
    auto old_and_weights = [&](uint32_t g, float (&v)[8], float (&u)[8]) __attribute__((always_inline)) {
        const uint32_t c = g * 8u < width ? g * 8u : 0u;
        m40_load_group<float, VEC>(x, c, width, v);
        m40_load_group<float, VEC>(w, c, width, u);
    };
    float keep[kGroups][8], keep_x[kGroups][8], keep_w[kGroups][8];
    float q = 0.0f;
    auto sq8 = [&](const float (&y)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) q = fmaf(y[i], y[i], q);
    };
#pragma unroll
    for (uint32_t j = 0; j < kGroups; ++j) {
        old_and_weights(tid + j * kM40RowThreads, keep_x[j], keep_w[j]);
        value(tid + j * kM40RowThreads, keep_x[j], keep[j]);
        sq8(keep[j]);
    }
    for (uint32_t g = tid + kGroups * kM40RowThreads; g < groups; g += kM40RowThreads) {
        float y[8], v[8], u[8];
        old_and_weights(g, v, u);
        value(g, v, y);
        sq8(y);
    }
    const float f = a.mult / sqrtf(m40_row_sum(q, tid, scratch) / (float)width + a.eps);
    auto finish = [&](uint32_t g, const float (&y)[8], const float (&old)[8], const float (&u)[8]) __attribute__((always_inline)) {
        float v[8];
        if (g * 8u < width) {
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) v[i] = VEC || g * 8u + i < width ? fmaf(y[i] * f, u[i], old[i]) : 0.0f;
            m40_store_group<VEC>(x, g * 8u, width, v);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = 0.0f;
        }
        sink(g, m40_float4{v[0], v[1], v[2], v[3]}, m40_float4{v[4], v[5], v[6], v[7]});
    };
#pragma unroll
    for (uint32_t j = 0; j < kGroups; ++j) {
        const uint32_t g = tid + j * kM40RowThreads;
        if (g < groups) finish(g, keep[j], keep_x[j], keep_w[j]);
    }
    for (uint32_t g = tid + kGroups * kM40RowThreads; g < groups; g += kM40RowThreads) {
        float y[8], v[8], u[8];
        old_and_weights(g, v, u);
        value(g, v, y);
        finish(g, y, v, u);
    }
}

// A thread takes groups of eight neighbouring columns in all streams and keeps the sums of two of them in registers (width up to 4096);
// beyond, they are formed again from the streams it has written.  S: streams, or (above four) the most there can be.
// sink as above (without w nothing is sunk, and there is no barrier).
template <class T, int S, bool VEC, class Sink>
__device__ __forceinline__ void m40_stream_update_row(const M40llmStreamUpdate& a, uint32_t row, uint32_t tid, float* scratch, const Sink& sink) {
    constexpr uint32_t kGroups = 2;
    const uint32_t width = a.width, groups = (a.w ? a.ld_h : (width + 7u) & ~7u) / 8u, streams = S <= 4 ? (uint32_t)S : a.streams;
    const float *mix = static_cast<const float*>(a.mix), *share = static_cast<const float*>(a.share), *take = static_cast<const float*>(a.take);
    const float* x0 = a.x0 ? static_cast<const float*>(a.x0) + (size_t)row * width : nullptr;
    float* xs = static_cast<float*>(a.streams_x) + (size_t)row * width;
    const bool write = a.place || a.n_planes;
    // up to four streams: all coefficients in registers before anything is stored
    constexpr bool kFew = S <= 4;
    float mx[kFew ? S : 1][kFew ? S : 1], sh[kFew ? S : 1], tk[kFew ? S : 1];
    if (kFew) {
#pragma unroll
        for (int t = 0; t < S; ++t) {
            tk[kFew ? t : 0] = take ? take[t] : 1.0f;
            sh[kFew ? t : 0] = write ? a.mult * share[t] : 0.0f;
#pragma unroll
            for (int s = 0; s < S; ++s) mx[kFew ? s : 0][kFew ? t : 0] = write ? mix[s * S + t] : 0.0f;
        }
    }
    auto taken = [&](uint32_t t) __attribute__((always_inline)) { return kFew ? tk[kFew ? t : 0] : take ? take[t] : 1.0f; };
    auto old = [&](uint32_t s, uint32_t g, float (&v)[8]) __attribute__((always_inline)) {
        m40_load_group<float, VEC>(x0 ? x0 : xs + s * (size_t)a.stream_stride, g * 8u, width, v);
    };
    auto output = [&](uint32_t g, float (&y)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = 0.0f;
        if (a.place) {
            // places, then rows of four experts at a time; of the last ones (fewer than four) the first again, of which zeros are taken
            const auto rows = [&](uint32_t j0, auto all_c) __attribute__((always_inline)) {
                constexpr bool kAll = decltype(all_c)::value;
                uint32_t at[4];
                float f[4], v[4][8];
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const size_t pick = (size_t)row * a.top + (kAll || j0 + j < a.top ? j0 + j : j0);
                    at[j] = a.place[pick];
                    f[j] = !kAll && j0 + j >= a.top ? 0.0f : a.weight ? static_cast<const float*>(a.weight)[pick] : 1.0f;
                }
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) m40_load_group<T, VEC>(static_cast<const T*>(a.expert_out) + (size_t)at[j] * a.ld_expert, g * 8u, width, v[j]);
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 8; ++i) y[i] = fmaf(f[j], kAll || j == 0 || j0 + j < a.top ? v[j][i] : 0.0f, y[i]);
            };
            uint32_t j0 = 0;
            for (; j0 + 4u <= a.top; j0 += 4u) rows(j0, std::true_type());
            if (j0 < a.top) rows(j0, std::false_type());
        } else {
            const float* plane = static_cast<const float*>(a.planes) + (size_t)row * width;
            uint32_t p = 0;
            for (; p + 1u < a.n_planes; p += 2u) {
                float v[2][8];
                m40_load_group<float, VEC>(plane + p * (size_t)a.plane_stride, g * 8u, width, v[0]);
                m40_load_group<float, VEC>(plane + (p + 1u) * (size_t)a.plane_stride, g * 8u, width, v[1]);
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] += v[0][i] + v[1][i];
            }
            if (p < a.n_planes) {
                float v[8];
                m40_load_group<float, VEC>(plane + p * (size_t)a.plane_stride, g * 8u, width, v);
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] += v[i];
            }
        }
    };
    // the streams' new values are stored (unless nothing reads them any more); their weighted sum in u
    auto turn = [&](uint32_t g, float (&u)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) u[i] = 0.0f;
        if (g * 8u >= width) return;
        float x[S][8], y[8];
#pragma unroll
        for (uint32_t s = 0; s < S; ++s)
            if (s < streams) old(s, g, x[s]);
        if (write) output(g, y);
#pragma unroll
        for (uint32_t t = 0; t < S; ++t) {
            if (t >= streams) continue;
            float z[8];
            if (write) {
                const float f = kFew ? sh[kFew ? t : 0] : a.mult * share[t];
#pragma unroll
                for (int i = 0; i < 8; ++i) z[i] = f * y[i];
#pragma unroll
                for (uint32_t s = 0; s < S; ++s)
                    if (s < streams) {
                        const float m = kFew ? mx[kFew ? s : 0][kFew ? t : 0] : mix[s * streams + t];
#pragma unroll
                        for (int i = 0; i < 8; ++i) z[i] = fmaf(m, x[s][i], z[i]);
                    }
                if (!a.discard) m40_store_group<VEC>(xs + t * (size_t)a.stream_stride, g * 8u, width, z);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) z[i] = x[t][i];
            }
            const float f = taken(t);
#pragma unroll
            for (int i = 0; i < 8; ++i) u[i] = fmaf(f, z[i], u[i]);
        }
    };
    auto again = [&](uint32_t g, float (&u)[8]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) u[i] = 0.0f;
        if (g * 8u >= width) return;
        for (uint32_t t = 0; t < streams; ++t) {
            float z[8];
            m40_load_group<float, VEC>(write || !x0 ? xs + t * (size_t)a.stream_stride : x0, g * 8u, width, z);
            const float f = take ? take[t] : 1.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) u[i] = fmaf(f, z[i], u[i]);
        }
    };
    // the weights' requests go out before the streams', 16 bytes each: behind them, one by one, they held the row's end up
    const float* w = static_cast<const float*>(a.w);
    auto weights = [&](uint32_t g, float (&v)[8]) __attribute__((always_inline)) {
        if (w && g * 8u < width) {
            m40_load_group<float, VEC>(w, g * 8u, width, v);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = 0.0f;
        }
    };
    float kept_w[kGroups][8];
    float keep[kGroups][8], q = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < kGroups; ++j) weights(tid + j * kM40RowThreads, kept_w[j]);
#pragma unroll
    for (uint32_t j = 0; j < kGroups; ++j) {
        turn(tid + j * kM40RowThreads, keep[j]);
#pragma unroll
        for (int i = 0; i < 8; ++i) q = fmaf(keep[j][i], keep[j][i], q);
    }
    for (uint32_t g = tid + kGroups * kM40RowThreads; g < groups; g += kM40RowThreads) {
        float u[8];
        turn(g, u);
#pragma unroll
        for (int i = 0; i < 8; ++i) q = fmaf(u[i], u[i], q);
    }
    const float inv = w ? 1.0f / sqrtf(m40_row_sum(q, tid, scratch) / (float)width + a.eps) : 1.0f;
    auto finish = [&](uint32_t g, const float (&u)[8], const float (&wg)[8]) __attribute__((always_inline)) {
        if (!w) {
            if (g * 8u < width) m40_store_group<VEC>(static_cast<float*>(a.x_out) + (size_t)row * width, g * 8u, width, u);
            return;
        }
        float v[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) v[i] = u[i] * inv * wg[i];          // both zero past the width
        sink(g, m40_float4{v[0], v[1], v[2], v[3]}, m40_float4{v[4], v[5], v[6], v[7]});
    };
#pragma unroll
    for (uint32_t j = 0; j < kGroups; ++j) {
        const uint32_t g = tid + j * kM40RowThreads;
        if (g < groups) finish(g, keep[j], kept_w[j]);
    }
    for (uint32_t g = tid + kGroups * kM40RowThreads; g < groups; g += kM40RowThreads) {
        float u[8], wg[8];
        if (a.discard) turn(g, u);
        else again(g, u);
        weights(g, wg);
        finish(g, u, wg);
    }
}
