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

// What the window decides about a packet without looking at other packets'
// counters: turned away outright, ahead of everything before it (fresh for
// certain), inside the window with its bit set before the batch (a repeat for
// certain), or inside the window at or below an earlier counter with the bit
// clear ("late": fresh unless an earlier packet of the batch carried the
// counter too).
enum : uint8_t { RP_NONE = 0, RP_AHEAD = 1, RP_LATE = 2, RP_SEEN = 3 };

// Sets `bit` of `block` in the window of peer `key` for every lane that has one (key 0xFFFFFFFFu:
// none).  A lane whose left neighbour differs gathers the bits of the lanes behind it that
// agree with it in peer and block and issues one atomic for all of them.
__device__ __forceinline__ void mark_bits(uint64_t *state, uint32_t key, uint64_t block, uint64_t bit)
{
    const uint32_t lane = threadIdx.x & 63u;
    // runs of equal (peer, block) among neighbouring lanes
    const uint32_t pkey = (uint32_t)__shfl_up((int)key, 1, 64);
    const uint32_t pblo = (uint32_t)__shfl_up((int)(uint32_t)block, 1, 64);
    const uint32_t pbhi = (uint32_t)__shfl_up((int)(uint32_t)(block >> 32), 1, 64);
    const bool head = lane == 0 || pkey != key || pblo != (uint32_t)block || pbhi != (uint32_t)(block >> 32);
    const unsigned long long heads = __ballot(head);
    // my run ends before the next head after me
    const unsigned long long after = lane == 63u ? 0ull : heads & ~((2ull << lane) - 1ull);
    const uint32_t end = after ? (uint32_t)__ffsll((long long)after) - 1u : 64u;
    uint64_t acc = bit;
    // suffix OR within the run: six doubling steps cover 64 lanes
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t lo = (uint32_t)__shfl_down((int)(uint32_t)acc, off, 64);
        const uint32_t hi = (uint32_t)__shfl_down((int)(uint32_t)(acc >> 32), off, 64);
        if (lane + (uint32_t)off < end) acc |= (uint64_t)hi << 32 | lo;
    }
    if (head && key != 0xFFFFFFFFu && acc != 0)
        atomicOr(reinterpret_cast<unsigned long long *>(
                     &state[(size_t)key * WG_REPLAY_WORDS + 1u + (block & (WG_REPLAY_BLOCKS - 1u))]),
                 (unsigned long long)acc);
}

// Sets the bit of every packet that reached the bit test and still lies in the
// window its peer ends the batch with.  Neighbours in sorted order mostly
// share their peer and their block of 64 counters (small batches come in batch order).  By workgroup `b` of `blocks`, each of
// REPLAY_MARK_THREADS.
//
// The same launch leaves the first-occurrence table empty for the next pass
// (nothing to do when this pass had no late packet, the usual case) and clears
// the flag word the next pass will use (nobody reads that one now).
__device__ __forceinline__ void replay_mark(const ReplayMark &m, uint32_t b, uint32_t blocks)
{
    const uint32_t p = b * REPLAY_MARK_THREADS + threadIdx.x;
    if (m.flags) {
        if (p == 0u) m.flags[m.parity ^ 1u] = 0u;
        if (m.flags[m.parity] != 0u)
            for (uint32_t i = p; i < m.slots; i += blocks * REPLAY_MARK_THREADS) m.table[i] = 0xFFFFFFFFu;
    }
    uint32_t key = 0xFFFFFFFFu;
    uint64_t block = ~0ull, bit = 0;
    if (p < m.n && m.cls[p] != RP_NONE) {
        key = m.skeys[p];
        const uint64_t c = m.sctr[p];
        const uint64_t final_last = m.state[(size_t)key * WG_REPLAY_WORDS];
        if ((final_last >> 6) - (c >> 6) < WG_REPLAY_BLOCKS) { // else its slot now belongs to a later block
            block = c >> 6;
            bit = 1ull << (c & 63u);
        } else {
            key = 0xFFFFFFFFu;
        }
    }
    mark_bits(m.state, key, block, bit);
}

} // namespace bnk
