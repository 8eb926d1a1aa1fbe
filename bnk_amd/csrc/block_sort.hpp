// Sorting 4096 words by a few of their bits within one workgroup, for the launches that do a
// whole batch of up to that many packets themselves (send counters, anti-replay windows).
//
// What bounds such a launch is its chain of barriers and trips to LDS, not its operations: so as
// few passes as the key's bits allow, eight bits at most each (one for up to 254 peers, two for
// up to 65534), and no word-wise traffic but the one exchange per pass.  A pass ranks a row of 64
// words at a time, a ballot per bit, against a count per wave and digit that only that wave
// touches, then scans the counts of all waves at once, four a thread.  Against rocPRIM's sort
// within a workgroup in its place: 3000 packets of 64 peers, counters 9.2 -> 8.2 us and windows
// 15.6 -> 15.1; 4096 of 254 peers 10.9 -> 9.9 and 18.6 -> 18.2, of 1024 peers 14.3 -> 12.5 and
// 22.0 -> 20.6.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bnk {

constexpr uint32_t BLOCK_SORT_THREADS = 1024, BLOCK_SORT_ITEMS = 4;
constexpr uint32_t BLOCK_SORT_WORDS = BLOCK_SORT_THREADS * BLOCK_SORT_ITEMS;
constexpr uint32_t BLOCK_SORT_WAVES = BLOCK_SORT_THREADS / 64u;
constexpr unsigned BLOCK_SORT_DIGIT_BITS = 8;
constexpr uint32_t BLOCK_SORT_DIGITS = 1u << BLOCK_SORT_DIGIT_BITS;
static_assert(BLOCK_SORT_DIGITS * BLOCK_SORT_WAVES == BLOCK_SORT_WORDS, "four counts a thread");

struct BlockSortShared {
    // (a row of counts begins a bank further on than the one before: the scan reads across rows)
    uint32_t count[BLOCK_SORT_WAVES][BLOCK_SORT_DIGITS + 1u];
    uint32_t wave_total[BLOCK_SORT_WAVES];
    uint32_t exchange[BLOCK_SORT_WORDS];
};

// The word that a thread brings as its item j: the batch's 64 of a row, rows of a wave in a row.
__device__ __forceinline__ uint32_t block_sort_place(uint32_t j)
{
    return (threadIdx.x >> 6) * 64u * BLOCK_SORT_ITEMS + j * 64u + (threadIdx.x & 63u);
}

// Sorts by bits [first, first + bits), stably: item j of a thread is the word at
// block_sort_place(j) before, and the one at j * BLOCK_SORT_THREADS + threadIdx.x after.
// Every thread of the workgroup calls it; sh is free to be overwritten, before and (behind a
// barrier) after.
__device__ __forceinline__ void block_sort(uint32_t (&word)[BLOCK_SORT_ITEMS], unsigned first, unsigned bits,
                                           BlockSortShared &sh)
{
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const unsigned passes = (bits + BLOCK_SORT_DIGIT_BITS - 1u) / BLOCK_SORT_DIGIT_BITS;
    const unsigned step = (bits + passes - 1u) / passes;
    uint32_t *const mine = sh.count[wave];
    for (unsigned done = 0; done < bits; done += step) {
        const unsigned shift = first + done, width = bits - done < step ? bits - done : step;
        const uint32_t mask = (1u << width) - 1u;
#pragma unroll
        for (uint32_t k = 0; k < BLOCK_SORT_DIGITS / 64u; k++) mine[k * 64u + lane] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint32_t rank[BLOCK_SORT_ITEMS]; // among the wave's words of the same digit
#pragma unroll
        for (uint32_t j = 0; j < BLOCK_SORT_ITEMS; j++) {
            const uint32_t digit = (word[j] >> shift) & mask;
            unsigned long long same = ~0ull;
            for (unsigned b = 0; b < width; b++) {
                const bool set = (digit >> b) & 1u;
                const unsigned long long m = __ballot(set);
                same &= set ? m : ~m;
            }
            const uint32_t lower = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
            const uint32_t before = mine[digit];
            rank[j] = before + lower;
            // (LDS answers a wave's accesses in order: every lane has read)
            if (lower == 0u) mine[digit] = before + (uint32_t)__popcll(same);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // counts to places: digit after digit, within one wave after wave
        const uint32_t digit = t / (BLOCK_SORT_WAVES / BLOCK_SORT_ITEMS);
        const uint32_t from = t % (BLOCK_SORT_WAVES / BLOCK_SORT_ITEMS) * BLOCK_SORT_ITEMS;
        uint32_t c[BLOCK_SORT_ITEMS], sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < BLOCK_SORT_ITEMS; j++) {
            c[j] = sh.count[from + j][digit];
            sum += c[j];
        }
        uint32_t upto = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)upto, off, 64);
            if ((int)lane >= off) upto += o;
        }
        if (lane == 63u) sh.wave_total[wave] = upto;
        __syncthreads();
        uint32_t at = upto - sum;
#pragma unroll
        for (uint32_t w = 0; w < BLOCK_SORT_WAVES; w++) {
            const uint32_t total = sh.wave_total[w];
            at += w < wave ? total : 0u;
        }
#pragma unroll
        for (uint32_t j = 0; j < BLOCK_SORT_ITEMS; j++) {
            sh.count[from + j][digit] = at;
            at += c[j];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < BLOCK_SORT_ITEMS; j++)
            sh.exchange[mine[(word[j] >> shift) & mask] + rank[j]] = word[j];
        __syncthreads();
        const bool last = done + step >= bits;
#pragma unroll
        for (uint32_t j = 0; j < BLOCK_SORT_ITEMS; j++)
            word[j] = sh.exchange[last ? j * BLOCK_SORT_THREADS + t : block_sort_place(j)];
    }
}

} // namespace bnk
