// Tokens a workgroup of the matrix-core attention takes (attention_mfma.hip).  Host code alone.
#pragma once

#include <cstdint>

// A multiple of 128 (one 32-token tile per wave and pass), at most 2048, sized for about one workgroup per CU -- measured best at 32 K tokens (256 workgroups of 1024
// tokens: 32 us against 36 us with twice as many half-sized ones) and on the batch-8 step -- rounded to the nearest multiple, and up while more than two workgroups
// would land on a CU and a longer chunk would leave fewer: with more rows and kv heads (`groups`) than that one chunk takes a whole row.
// may_halve: around half a thousand tokens a chunk two workgroups a CU are better: a wave's tiles follow one another, and two is as many as are worth waiting for
// (32 rows of up to 1021 tokens, 4 kv heads of 64: chunks of 512 9.0 us, of 256 7.8 us; 8 rows of up to 4093, 2 kv heads of 128: chunks of 256 8.8 us, of 128
// 9.2 us).
inline uint32_t m40_attention_chunk(uint64_t groups, uint32_t span, uint32_t num_cus, bool may_halve) {
    constexpr uint64_t kMost = 2048;
    uint64_t chunk = (span * groups / num_cus + 64) / 128 * 128;
    if (chunk > 256 && chunk <= 512 && may_halve) chunk = 256;
    if (chunk < 128) chunk = 128;
    while (chunk < span && chunk < kMost && groups * ((span + chunk - 1) / chunk) > 2ull * num_cus) chunk += 128;
    return (uint32_t)(chunk < kMost ? chunk : kMost);
}
