// Activation rows as matrix operands: what a launch that makes rows leaves for the projection behind it (packed_rows.hip), instead of f32.
//
// Up to 32 rows of K, padded to R = 8, 16 or 32.  Eight consecutive k of a row are one unit with a power-of-two scale of their own: f16 hi + lo
// parts of the value over the scale, the largest magnitude in [2^14, 2^15): a value is exact to 2^-22 of itself and 2^-39 of its unit's largest.  (A unit is what every
// producer holds in eight neighbouring lanes; units that meet in a matrix instruction are brought to one scale by their reader.)  Scale 0: a unit of zeros, or one with
// infinities or NaN, which are left as they are, its finite values as zeros: they add nothing to that.  First the operands, [K / 32][R / 8] KiB, each in the order in which a wave
// reads it: 16 bytes = the eight parts of a unit, of k 32 s + 8 g .. + 7, at lane 16 g + row.  R = 8: one KiB, rows 0-7 of which hold the hi parts and rows
// 8-15 the lo parts.  R = 16, 32: the hi KiB and the lo KiB of each sixteen rows.  Behind them the scales, f32 [K / 8][R].
#pragma once
#include "common.hpp"

static inline __host__ __device__ int m40_packed_pad(int rows) { return rows <= 8 ? 8 : (rows <= 16 ? 16 : 32); }
static inline __host__ __device__ size_t m40_packed_bytes(int rows, int K) { return (size_t)m40_packed_pad(rows) * K * 4 + (size_t)m40_packed_pad(rows) * (K / 8) * 4; }

// Eight neighbouring lanes hold y of row `row`, columns c .. c + 7 with c a multiple of 8 (col = c + the lane's place): all eight store their parts.
__device__ __forceinline__ void m40_store_packed(uint8_t* packed, int pad, int K, int row, int col, float y) {
    const bool finite = fabsf(y) < INFINITY;
    float mx = finite ? fabsf(y) : INFINITY;
    mx = fmaxf(mx, m40_dpp_f<M40_DPP_XOR1>(mx));
    mx = fmaxf(mx, m40_dpp_f<M40_DPP_XOR2>(mx));
    mx = fmaxf(mx, m40_dpp_f<M40_DPP_HALF_MIRROR>(mx));
    int ex;                                  // 2^ex: the unit's scale, at most 2^113
    (void)frexpf(mx, &ex);
    ex = ex < -85 ? -100 : ex - 15;
    const bool scaled = mx > 0.0f && mx < INFINITY;
    const float inv = scaled ? __uint_as_float((uint32_t)(127 - ex) << 23) : (finite ? 0.0f : 1.0f);
    const _Float16 hi = static_cast<_Float16>(y * inv);
    const _Float16 lo = scaled ? static_cast<_Float16>(fmaf(y, inv, -static_cast<float>(hi))) : static_cast<_Float16>(0.0f);
    const int part = pad > 8 ? 1024 : 128, tile = pad > 8 ? 2048 * (row >> 4) : 0, place = pad > 8 ? row & 15 : row;
    uint8_t* at = packed + (size_t)(col >> 5) * (pad * 128) + tile + (16 * ((col >> 3) & 3) + place) * 16 + 2 * (col & 7);
    *reinterpret_cast<_Float16*>(at) = hi;
    *reinterpret_cast<_Float16*>(at + part) = lo;
    if ((col & 7) == 0) reinterpret_cast<float*>(packed + (size_t)pad * K * 4)[(size_t)(col >> 3) * pad + row] = scaled ? __uint_as_float((uint32_t)(127 + ex) << 23) : 0.0f;
}
