// Choice of experts for a row (experts.hip; norm_route.hip makes it behind a norm).
#pragma once

#include "packed_gemm.hpp"

// Experts in groups of `size` neighbours: what is left of `left` when only the `keep` groups whose best choice is largest (the lower group of
// equals) can be chosen from.
template <uint32_t N>
__device__ __forceinline__ uint32_t m40_within_groups(const M40llmRoute& a, uint32_t lane, uint32_t size, const float (&choice)[N], uint32_t left) {
    uint32_t kept = 0, open = left;          // bit i: this lane's expert i is in a group that is taken, in one that still can be
    for (uint32_t k = 0; k < a.keep; ++k) {
        float best = -INFINITY;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) best = open >> i & 1u ? fmaxf(best, choice[i]) : best;
        best = m40_max64(best);
        uint32_t at = 0xffffffffu;           // its lowest expert (of one that is no number: the lowest that is open)
#pragma unroll
        for (uint32_t any = 0; any < 2u; ++any)
#pragma unroll
            for (uint32_t i = 0; i < N; ++i) {
                const unsigned long long hit = __ballot((open >> i & 1u) && (any || choice[i] == best));
                if (at == 0xffffffffu && hit) at = (uint32_t)__ffsll(hit) - 1u + 64u * i;
            }
        if (at == 0xffffffffu) break;
        const uint32_t group = at / size;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i)
            if ((left >> i & 1u) && (lane + 64u * i) / size == group) {
                kept |= 1u << i;
                open &= ~(1u << i);
            }
    }
    return kept;
}

// A wave routes one row: lane l holds the logits z (and corrections c) of experts l, l + 64, ..., N of them.
template <uint32_t N>
__device__ __forceinline__ void m40_route_logits(const M40llmRoute& a, uint32_t lane, const float (&z)[N], const float (&c)[N], uint32_t* ids, float* weight) {
    const uint32_t n = a.experts + a.identity;
    const bool correction = a.correction != nullptr;
    const bool sigmoid = a.score == M40LLM_SCORE_SIGMOID;
    float s[N], choice[N];
    float top = -INFINITY;
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) {
        const uint32_t e = lane + 64u * i;
        s[i] = e < n ? z[i] : -INFINITY;
        choice[i] = c[i];
        top = fmaxf(top, s[i]);
    }
    top = m40_max64(top);
    float sum = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) {
        const float logit = s[i];
        s[i] = lane + 64u * i >= n ? 0.0f : sigmoid ? m40_sigmoid(logit) : expf(logit - top);
        sum += s[i];
        // sigmoids of large logits are equal in f32 where the logits are not: without a correction the logits decide
        if (sigmoid) choice[i] = correction ? choice[i] + s[i] : logit;
    }
    sum = m40_sum64(sum);
    uint32_t left = 0;                       // bit i: this lane's expert i can be chosen
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) {
        const uint32_t e = lane + 64u * i;
        if (!sigmoid) {
            s[i] /= sum;
            choice[i] += s[i];
        }
        if (e < n) left |= 1u << i;
    }
    if (a.groups > 1u) left = m40_within_groups<N>(a, lane, n / a.groups, choice, left);
    uint32_t mine_id = 0;
    float mine_weight = 0.0f;                // choice `lane`
    for (uint32_t j = 0; j < a.top; ++j) {
        float best = -INFINITY;
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) best = left >> i & 1u ? fmaxf(best, choice[i]) : best;
        best = m40_max64(best);
        uint32_t at = 0;
        float w = 0.0f;
        bool found = false;                  // the lowest index of equals: i before lane
#pragma unroll
        for (uint32_t i = 0; i < N; ++i) {
            const unsigned long long hit = __ballot((left >> i & 1u) && choice[i] == best);
            if (!found && hit) {
                const uint32_t l = (uint32_t)__ffsll(hit) - 1u;
                at = l + 64u * i;
                w = __shfl(s[i], (int)l);
                if (lane == l) left &= ~(1u << i);
                found = true;
            }
        }
        if (!found) {                        // nothing comparable is left (not a number): the lowest index that can be chosen
#pragma unroll
            for (uint32_t i = 0; i < N; ++i) {
                const unsigned long long hit = __ballot(left >> i & 1u);
                if (!found && hit) {
                    const uint32_t l = (uint32_t)__ffsll(hit) - 1u;
                    at = l + 64u * i;
                    w = __shfl(s[i], (int)l);
                    if (lane == l) left &= ~(1u << i);
                    found = true;
                }
            }
        }
        if (lane == (j & 63u)) { mine_id = at; mine_weight = w; }
        if ((j & 63u) == 63u || j + 1u == a.top) {
            const uint32_t first = j & ~63u;
            if (first + lane <= j) {
                ids[first + lane] = mine_id;
                weight[first + lane] = mine_weight * a.scale;
            }
        }
    }
}

template <uint32_t N>
__device__ __forceinline__ void m40_route_corrections(const M40llmRoute& a, uint32_t lane, float (&c)[N]) {
#pragma unroll
    for (uint32_t i = 0; i < N; ++i) c[i] = a.correction && lane + 64u * i < a.experts + a.identity ? static_cast<const float*>(a.correction)[lane + 64u * i] : 0.0f;
}
