// Up to 4096 packets by one workgroup, in batch order and without a sort, where the peers' numbers fit
// ROW_DIGITS: each of its 16 waves takes as many rows of 64 packets in a row as the batch needs, keeps what
// its own packets come to per peer in LDS, which only that wave touches, and a thread per peer then
// goes over the waves.  What bounds such a launch is its chain of barriers and trips to LDS and memory; a
// sort is the longest part of it, and what is looked up by a packet's peer or place can be on its way
// from the start here.  3000 packets of 64 peers: send counters 9.0 -> 7.3 us, windows 15.2 -> 6.6;
// 700 packets 5.0 -> 4.2 and 18.5 -> 4.4.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bnk {

constexpr uint32_t ROW_THREADS = 1024, ROW_WAVES = ROW_THREADS / 64u, ROWS_MOST = 4;
constexpr uint32_t ROW_PACKETS = ROW_THREADS * ROWS_MOST;
constexpr uint32_t ROW_DIGITS = 256; // the peers, at most 255, and nobody
constexpr unsigned ROW_BITS = 8;

// Packet of this lane in row j of its wave's, of `rows`.
__device__ __forceinline__ uint32_t row_place(uint32_t rows, uint32_t j)
{
    return ((threadIdx.x >> 6) * rows + j) * 64u + (threadIdx.x & 63u);
}

// The lanes of the wave with this lane's key (below ROW_DIGITS).
__device__ __forceinline__ unsigned long long row_same(uint32_t key, unsigned bits)
{
    unsigned long long same = ~0ull;
    for (unsigned b = 0; b < bits; b++) {
        const bool set = (key >> b) & 1u;
        const unsigned long long m = __ballot(set);
        same &= set ? m : ~m;
    }
    return same;
}

} // namespace bnk
