// One peer's anti-replay window (see wg_replay.hip) as a lane reads and moves it.
#pragma once

#include "kernels.hpp"
#include "wg_dev.hpp"

namespace bnk {

constexpr uint64_t WINDOW = (WG_REPLAY_BLOCKS - 1u) * 64u; // 8128

__device__ __forceinline__ bool replay_subject(uint8_t result)
{
    // everything that was authentic: the tag verified
    return result != BNK_WG_BAD_HEADER && result != BNK_WG_UNKNOWN_INDEX && result != BNK_WG_AUTH_FAIL;
}

// Does the packet reach the filter's bit test, given `last` just before it?
__device__ __forceinline__ bool reaches_bit_test(uint64_t c, uint64_t last)
{
    return c < WG_REJECT_AFTER_MESSAGES && (c > last || last - c <= WINDOW);
}

// Was counter c (at or below last0, inside the window) seen before the batch?
__device__ __forceinline__ bool seen_before(const uint64_t *st, uint64_t c)
{
    return (st[1u + ((c >> 6) & (WG_REPLAY_BLOCKS - 1u))] >> (c & 63u)) & 1ull;
}

// Brings one peer's window to `new_last`: clears the blocks passed over.
__device__ __forceinline__ void advance_window(uint64_t *st, uint64_t new_last)
{
    const uint64_t last0 = st[0];
    if (new_last <= last0) return;
    const uint64_t cur = last0 >> 6;
    uint64_t diff = (new_last >> 6) - cur;
    if (diff > WG_REPLAY_BLOCKS) diff = WG_REPLAY_BLOCKS;
    for (uint64_t b = cur + 1; b <= cur + diff; b++) st[1u + (b & (WG_REPLAY_BLOCKS - 1u))] = 0;
    st[0] = new_last;
}

} // namespace bnk
