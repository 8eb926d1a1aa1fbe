// Bookkeeping of the fused relay step open -> filter -> re-seal: verdicts and
// the outbound nonce counters.  A packet that survives takes the next counter
// of its outbound peer in batch order; dropped packets consume none (as in
// wireguard-go, where the nonce is assigned when a packet is queued for
// sending).  That is a segmented exclusive count over the survivors keyed by
// peer: a stable radix sort of (peer, index) pairs puts each peer's survivors
// together in batch order, and a survivor's rank is its distance from the
// first element of its segment.
#include <string.h>

#include <algorithm>

#include <rocprim/rocprim.hpp>

#include "../../include/bnkhip.h"
#include "block_rows.hpp"
#include "block_sort.hpp"
#include "filter_lane.hpp"
#include "kernels.hpp"

namespace bnk {

constexpr uint32_t NO_PEER = 0xFFFFFFFFu;

// What a relayed packet's verdict and key come from, and where they go: keys[] is the outbound peer of each
// survivor and all ones for the rest.  tally: null, or the launch counts the verdicts.
// (With a launch of their own for the verdicts and one that counted them at the end, relayed batches of 1000
// packets with three streams at work took 17.3 us against 12.6, of 4000 22.5 against 18.6, of 100000 76.5
// against 74.4.)
struct RelayIn {
    const uint8_t *auth, *pass;
    const uint32_t *peer_out;
    uint8_t *verdict;
    uint32_t *keys;
    uint32_t *status;
    unsigned long long *tally;
};

// The verdict of a packet of the batch, and its key.
__device__ __forceinline__ uint8_t relay_verdict(const RelayIn &in, uint8_t auth, uint8_t pass, uint32_t n_peers_out, uint32_t &key)
{
    uint8_t v = !auth ? BNK_RELAY_FORGED : !pass ? BNK_RELAY_DENIED : BNK_RELAY_OK;
    if (v == BNK_RELAY_OK && key >= n_peers_out) {
        status_raise(in.status, STATUS_PEER_RANGE);
        v = BNK_RELAY_DENIED;
    }
    if (v != BNK_RELAY_OK) key = NO_PEER;
    return v;
}

// The votes of a wave, one a lane (there: it has one), added to what it has of the three verdicts.
__device__ __forceinline__ void relay_vote(uint8_t v, bool there, uint32_t (&votes)[3])
{
    votes[0] += (uint32_t)__popcll(__ballot(there && v == BNK_RELAY_OK));
    votes[1] += (uint32_t)__popcll(__ballot(there && v == BNK_RELAY_FORGED));
    votes[2] += (uint32_t)__popcll(__ballot(there && v == BNK_RELAY_DENIED));
}
__device__ __forceinline__ void relay_tally(unsigned long long *tally, const uint32_t (&votes)[3])
{
    tally_bump(tally, TALLY_RELAYED, votes[0]);
    tally_bump(tally, TALLY_REJECTED, votes[1]);
    tally_bump(tally, TALLY_DENIED, votes[2]);
}

// Four packets a thread, and each array in one access where they all lie so that it can be (four
// byte loads and stores a packet otherwise: 2^22 packets 20 us against 11.5).  For batches whose counters
// come from a sort; the others' first launch does this along the way (rank_count_tile, peer_rank_rows).
template <bool ALIGNED>
__global__ __launch_bounds__(256) void relay_verdict_kernel(RelayIn in, uint32_t n_peers_out, uint32_t n, uint32_t *idx, uint64_t *ctr_out)
{
    const uint8_t *const auth = in.auth, *const pass = in.pass;
    const uint32_t *const peer_out = in.peer_out;
    uint32_t *const keys = in.keys;
    uint8_t *const verdict = in.verdict;
    const uint32_t first = (blockIdx.x * 256u + threadIdx.x) * 4u;
    if (__ballot(first < n) == 0ull) return;
    const bool whole = ALIGNED && has_from(first, 4u, n);
    alignas(4) uint8_t au[4], pa[4], v[4];
    alignas(16) uint32_t key[4];
    if (whole) {
        *reinterpret_cast<uint32_t *>(au) = *reinterpret_cast<const uint32_t *>(auth + first);
        *reinterpret_cast<uint32_t *>(pa) = *reinterpret_cast<const uint32_t *>(pass + first);
        *reinterpret_cast<uint4 *>(key) = *reinterpret_cast<const uint4 *>(peer_out + first);
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const uint32_t i = min(first + j, n - 1u);
            au[j] = auth[i];
            pa[j] = pass[i];
            key[j] = peer_out[i];
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        v[j] = relay_verdict(in, au[j], pa[j], n_peers_out, key[j]); // (beyond the end: the last packet's again)
    }
    if (in.tally) {
        uint32_t votes[3] = {0, 0, 0};
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) relay_vote(v[j], first < n && first + j < n, votes);
        if ((threadIdx.x & 63u) == 0u) relay_tally(in.tally, votes);
    }
    if (first >= n) return;
    if (whole) {
        *reinterpret_cast<uint32_t *>(verdict + first) = *reinterpret_cast<const uint32_t *>(v);
        *reinterpret_cast<uint4 *>(keys + first) = *reinterpret_cast<const uint4 *>(key);
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        const uint32_t i = first + j;
        if (i >= n) break;
        if (!whole) {
            verdict[i] = v[j];
            keys[i] = key[j];
        }
        idx[i] = i;
        ctr_out[i] = 0;
    }
}

// Where each peer's run starts in the sorted sequence.
__global__ __launch_bounds__(256) void peer_heads_kernel(const uint32_t *skeys, uint32_t n,
                                                         uint32_t *seg_start)
{
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= n) return;
    const uint32_t key = skeys[p];
    if (key == NO_PEER) return;
    if (p == 0u || skeys[p - 1u] != key) seg_start[key] = p;
}

__global__ __launch_bounds__(256) void relay_rank_kernel(const uint32_t *skeys, const uint32_t *sidx,
                                                         const uint32_t *seg_start,
                                                         const uint64_t *ctr_base_out, uint32_t n,
                                                         uint64_t *ctr_out, uint64_t ctr_limit)
{
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= n) return;
    const uint32_t key = skeys[p];
    if (key == NO_PEER) return;
    ctr_out[sidx[p]] = ctr_add(ctr_base_out[key], (uint64_t)(p - seg_start[key]), ctr_limit);
}

// The last element of each peer's segment holds the largest counter handed out.
__global__ __launch_bounds__(256) void peer_advance_kernel(const uint32_t *skeys, const uint32_t *sidx,
                                                           const uint64_t *ctr_out, uint32_t n,
                                                           uint64_t *ctr_base, uint64_t ctr_limit)
{
    const uint32_t p = blockIdx.x * 256u + threadIdx.x;
    if (p >= n) return;
    const uint32_t key = skeys[p];
    if (key == NO_PEER) return;
    if (p + 1u < n && skeys[p + 1u] == key) return;
    ctr_base[key] = ctr_add(ctr_out[sidx[p]], 1u, ctr_limit);
}

// Peer keys are below n_keys and the "no peer" key is all ones, so the low
// bit_width(n_keys) bits order them the same way the full word does.
static unsigned key_bits(uint32_t n_keys)
{
    unsigned bits = 1;
    while (bits < 32 && (n_keys >> bits) != 0) bits++;
    return bits;
}

// A few key bits sort faster in one or two Onesweep passes than in the merge
// sort rocPRIM picks by default for up to 2^20 items.
using SortConfig = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                              rocprim::default_config, 32768>;

constexpr uint32_t RANK_TABLE_MAX_KEYS = 4096;
constexpr uint32_t RANK_ROW_STEP = 256; // 64 lanes x 16 bytes
constexpr uint32_t RANK_ROW_STEPS = RANK_TABLE_MAX_KEYS / RANK_ROW_STEP;
constexpr uint32_t TILE_RUNS_MAX = 32;
constexpr uint32_t TILE_RUNS_FEW = 8; // up to 2^20 packets
constexpr size_t RANK_TABLE_MAX_BYTES = 64u << 20;
// Sorting by peer (launch_peer_sort): up to this many keys.  With 4001 of them a tile's row is
// longer than the tile and it is the library's radix sort or this within 3 % either way.
constexpr uint32_t PEER_SORT_MAX_KEYS = 2048;

struct RankPlan {
    uint32_t runs;  // runs of 64 packets per tile
    uint32_t tiles;
    uint32_t cols;  // entries per row of the table: the keys, rounded up to what a wave moves at once
    size_t bytes;   // the table, then one total per peer, then every peer's counter as the batch found it
    bool fits;
};

static RankPlan rank_plan(uint32_t n, uint32_t n_keys)
{
    RankPlan p{};
    // about 1024 tiles (a wave each: enough to keep every CU busy; with 2048 the table of a
    // thousand peers is longer than the batch: counters and window sort of 2^17 packets 8 us
    // more, of 2^18 6), 2048 for large batches (2^20: 5 us less), as long as a wave
    // can hold its tile's keys in registers
    const uint32_t run_packets = 64u * (n <= 1u << 19 ? 1024u : 2048u);
    p.runs = std::min<uint32_t>(TILE_RUNS_MAX, std::max<uint32_t>(1u, (n + run_packets - 1u) / run_packets));
    p.tiles = (n + 64u * p.runs - 1u) / (64u * p.runs);
    p.cols = (n_keys + RANK_ROW_STEP - 1u) / RANK_ROW_STEP * RANK_ROW_STEP;
    p.bytes = ((size_t)p.tiles + 1u) * p.cols * 4u + (size_t)p.cols * 8u;
    p.fits = n_keys <= RANK_TABLE_MAX_KEYS && p.bytes <= RANK_TABLE_MAX_BYTES;
    return p;
}

size_t relay_sort_tmp_bytes(uint32_t n, uint32_t n_keys)
{
    size_t bytes = 0;
    (void)rocprim::radix_sort_pairs<SortConfig>(nullptr, bytes, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                    (const uint32_t *)nullptr, (uint32_t *)nullptr, (size_t)n, 0,
                                    key_bits(n_keys));
    // once the sort is done the same scratch holds one run start per key
    bytes = std::max(bytes, (size_t)n_keys * 4);
    // the sort-free form's table, for this batch or any part of it (a part is cut
    // into up to 2048 tiles however small it is)
    const RankPlan plan = rank_plan(n, n_keys);
    if (!plan.fits) return bytes;
    const size_t rows = std::max<size_t>(plan.tiles, std::min<size_t>(n / 64u + 1u, 2048u)) + 1u;
    return std::max(bytes, rows * plan.cols * 4u + (size_t)plan.cols * 8u);
}

static hipError_t launch_peer_rank_one_block(const uint32_t *peer, uint32_t n_keys, uint32_t n, uint64_t *ctr_base,
                                             uint64_t *ctr_out, bool advance, bool no_peer_ok, uint64_t ctr_limit,
                                             uint32_t *status, hipStream_t s);

static hipError_t launch_peer_rank_table(const uint32_t *keys, const RankPlan &plan, void *tmp,
                                         uint64_t *ctr_base, uint32_t n_keys, uint32_t n, uint64_t *ctr_out,
                                         bool advance, uint64_t ctr_limit, bool zero_others, uint32_t *status,
                                         const RelayIn *relay, hipStream_t s);
static hipError_t launch_relay_rank_rows(const RelayIn &in, uint32_t n_keys, uint32_t n, uint64_t *ctr_base, uint64_t *ctr_out,
                                         bool advance, hipStream_t s);

// The form for a batch of one workgroup: a packet a thread, four, or rows.
enum RankForm : uint32_t { RANK_SMALL, RANK_BLOCK, RANK_ROWS };
static RankForm rank_form(uint32_t n, uint32_t n_keys)
{
    return n_keys < ROW_DIGITS ? RANK_ROWS : n <= PEER_RANK_SMALL_MAX ? RANK_SMALL : RANK_BLOCK;
}

hipError_t launch_relay_assign(const uint8_t *auth, const uint8_t *pass, const uint32_t *peer_out,
                               const uint64_t *ctr_base_out, uint32_t n_peers_out, uint32_t n,
                               uint32_t *keys, uint32_t *idx, uint32_t *skeys, uint32_t *sidx,
                               void *sort_tmp, size_t sort_tmp_bytes, uint8_t *verdict,
                               uint64_t *ctr_out, uint32_t *status, unsigned long long *tally, bool advance, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    const RankPlan plan = rank_plan(n, n_peers_out);
    const bool one_block = peer_rank_one_block(n, n_peers_out);
    const RelayIn in{auth, pass, peer_out, verdict, keys, status, tally};
    uint64_t *const ctr_base = const_cast<uint64_t *>(ctr_base_out);
    if (one_block && rank_form(n, n_peers_out) == RANK_ROWS) return launch_relay_rank_rows(in, n_peers_out, n, ctr_base, ctr_out, advance, s);
    if (!one_block && plan.fits && plan.bytes <= sort_tmp_bytes)
        return launch_peer_rank_table(keys, plan, sort_tmp, ctr_base, n_peers_out, n, ctr_out, advance, 0ull, true, nullptr, &in, s);
    const bool aligned = (((uintptr_t)auth | (uintptr_t)pass | (uintptr_t)verdict) & 3u) == 0 &&
                         (((uintptr_t)peer_out | (uintptr_t)keys) & 15u) == 0;
    hipLaunchKernelGGL(aligned ? relay_verdict_kernel<true> : relay_verdict_kernel<false>, dim3(n / 1024u + (n % 1024u != 0u)), dim3(256), 0, s,
                       in, n_peers_out, n, idx, ctr_out);
    if (one_block) return launch_peer_rank_one_block(keys, n_peers_out, n, ctr_base, ctr_out, advance, true, 0ull, status, s);
    return launch_peer_rank(keys, idx, skeys, sidx, sort_tmp, sort_tmp_bytes, ctr_base, n_peers_out, n, ctr_out, advance, 0ull, s);
}

// The batch-order counters of a small batch, by one workgroup.
struct RankArgs {
    const uint32_t *peer; // or nullptr: every packet is peer 0
    uint32_t n_keys, n;
    uint64_t *ctr_base, *ctr_out;
    int advance, no_peer_ok;
    unsigned bits; // of a key
    uint64_t ctr_limit;
    uint32_t *status;
};

// Straight from the peer array: a stable block-wide radix sort of (peer, position)
// brings each peer's packets together in batch order; a packet's rank is its
// distance from the head of its run, and the last packet of a run moves the
// peer's base.
BNK_DEV void peer_rank_small(const RankArgs &a)
{
    using Sort = rocprim::block_radix_sort<uint32_t, PEER_RANK_SMALL_MAX, 1, uint32_t>;
    using Scan = rocprim::block_scan<uint32_t, PEER_RANK_SMALL_MAX>;
    __shared__ union {
        typename Sort::storage_type sort;
        typename Scan::storage_type scan;
    } tmp;
    __shared__ uint32_t sk[PEER_RANK_SMALL_MAX + 1];
    const uint32_t t = threadIdx.x;
    uint32_t key[1] = {NO_PEER}, pos[1] = {t};
    if (t < a.n) {
        key[0] = a.peer ? a.peer[t] : 0u;
        if (key[0] >= a.n_keys) {
            if (!(a.no_peer_ok && key[0] == NO_PEER)) status_raise(a.status, STATUS_PEER_RANGE);
            key[0] = NO_PEER;
        }
    }
    // valid keys are below n_keys < 2^bits and "no peer" is all ones, so the low
    // bits order them the way the full word does, "no peer" last
    Sort().sort(key, pos, tmp.sort, 0, a.bits);
    sk[t] = key[0];
    if (t == 0) sk[PEER_RANK_SMALL_MAX] = NO_PEER;
    __syncthreads();
    const bool valid = key[0] != NO_PEER;
    const bool head = t == 0 || sk[t - 1] != key[0];
    const bool last = sk[t + 1] != key[0];
    uint32_t start = 0;
    Scan().inclusive_scan(head ? t : 0u, start, tmp.scan, rocprim::maximum<uint32_t>());
    uint64_t mine = 0;
    if (valid) {
        mine = ctr_add(a.ctr_base[key[0]], t - start, a.ctr_limit);
        a.ctr_out[pos[0]] = mine;
    }
    __syncthreads(); // every base has been read
    if (a.advance && valid && last) a.ctr_base[key[0]] = ctr_add(mine, 1u, a.ctr_limit);
}

// The same for up to PEER_RANK_BLOCK_MAX packets, four a thread, peer and position sorted as
// one word; position p of the sorted batch is thread p % PEER_BLOCK_THREADS's.  (The counting
// form's three launches cost four to six microseconds each at any size: 3000 packets 16 us,
// here 8.)
constexpr uint32_t PEER_BLOCK_THREADS = BLOCK_SORT_THREADS, PEER_BLOCK_ITEMS = BLOCK_SORT_ITEMS;
constexpr unsigned PEER_BLOCK_INDEX_BITS = 12;
static_assert(PEER_RANK_SMALL_MAX == PEER_BLOCK_THREADS, "one launch shape");
static_assert(PEER_RANK_BLOCK_MAX == 1u << PEER_BLOCK_INDEX_BITS && PEER_RANK_BLOCK_MAX == BLOCK_SORT_WORDS, "packed keys");
BNK_DEV void peer_rank_block(const RankArgs &a)
{
    constexpr uint32_t ROWS = PEER_RANK_BLOCK_MAX / 64u;
    static_assert(ROWS == 64u, "a lane per row");
    __shared__ BlockSortShared sort;
    __shared__ uint32_t sk[PEER_RANK_BLOCK_MAX + 1];
    __shared__ uint32_t last_head[ROWS];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t none = (1u << a.bits) - 1u; // above every peer
    uint32_t word[PEER_BLOCK_ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < PEER_BLOCK_ITEMS; j++) {
        const uint32_t i = block_sort_place(j);
        uint32_t key = NO_PEER;
        if (i < a.n) {
            key = a.peer ? a.peer[i] : 0u;
            if (key >= a.n_keys && !(a.no_peer_ok && key == NO_PEER)) status_raise(a.status, STATUS_PEER_RANGE);
        }
        word[j] = (key < a.n_keys ? key : none) << PEER_BLOCK_INDEX_BITS | i;
    }
    block_sort(word, PEER_BLOCK_INDEX_BITS, a.bits, sort);
#pragma unroll
    for (uint32_t j = 0; j < PEER_BLOCK_ITEMS; j++) sk[j * PEER_BLOCK_THREADS + t] = word[j] >> PEER_BLOCK_INDEX_BITS;
    if (t == 0) sk[PEER_RANK_BLOCK_MAX] = NO_PEER;
    __syncthreads();
    // where a position's run begins: the head at or before it in its row of 64, else the last
    // head of the rows before
    uint32_t start[PEER_BLOCK_ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < PEER_BLOCK_ITEMS; j++) {
        const uint32_t p = j * PEER_BLOCK_THREADS + t;
        const unsigned long long heads = __ballot(p == 0u || sk[p - 1u] != sk[p]);
        const unsigned long long upto = heads & (~0ull >> (63u - lane));
        start[j] = upto ? p - lane + 63u - (uint32_t)__clzll((long long)upto) : NO_PEER;
        if (lane == 63u) last_head[p >> 6] = upto ? start[j] : 0u;
    }
    __syncthreads();
    {
        uint32_t back = last_head[lane];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)back, off, 64);
            if ((int)lane >= off) back = max(back, o);
        }
#pragma unroll
        for (uint32_t j = 0; j < PEER_BLOCK_ITEMS; j++) {
            const uint32_t row = j * (PEER_BLOCK_THREADS / 64u) + wave;
            const uint32_t handed = (uint32_t)__shfl((int)back, (int)(row ? row - 1u : 0u), 64);
            if (start[j] == NO_PEER) start[j] = handed; // (the first row begins with a head)
        }
    }
    uint64_t mine[PEER_BLOCK_ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < PEER_BLOCK_ITEMS; j++) {
        const uint32_t p = j * PEER_BLOCK_THREADS + t, key = word[j] >> PEER_BLOCK_INDEX_BITS;
        mine[j] = 0;
        if (key == none) continue;
        mine[j] = ctr_add(a.ctr_base[key], p - start[j], a.ctr_limit);
        a.ctr_out[word[j] & (PEER_RANK_BLOCK_MAX - 1u)] = mine[j];
    }
    __syncthreads(); // every base has been read
#pragma unroll
    for (uint32_t j = 0; j < PEER_BLOCK_ITEMS; j++) {
        const uint32_t p = j * PEER_BLOCK_THREADS + t, key = word[j] >> PEER_BLOCK_INDEX_BITS;
        if (a.advance && key != none && sk[p + 1u] != key) a.ctr_base[key] = ctr_add(mine[j], 1u, a.ctr_limit);
    }
}

// The same without a sort (block_rows.hpp), for tables of fewer than ROW_DIGITS peers.
static_assert(PEER_BLOCK_THREADS == ROW_THREADS && PEER_RANK_BLOCK_MAX == ROW_PACKETS, "one launch shape");
// RELAY: of a relay's batch, whose verdicts come first (a.peer is not read).
template <bool RELAY>
BNK_DEV void peer_rank_rows(const RankArgs &a, const RelayIn &in)
{
    __shared__ uint32_t count[ROW_WAVES][ROW_DIGITS];
    __shared__ uint64_t base[ROW_DIGITS];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
    const uint32_t rows = (a.n + ROW_THREADS - 1u) / ROW_THREADS, none = ROW_DIGITS - 1u;
    uint32_t *const mine = count[wave];
    uint32_t key[ROWS_MOST];
#pragma unroll
    for (uint32_t j = 0; j < ROWS_MOST; j++) {
        const uint32_t i = row_place(rows, j);
        if (!RELAY) key[j] = j < rows && i < a.n ? (a.peer ? a.peer[i] : 0u) : NO_PEER;
    }
    if (RELAY) {
        uint8_t au[ROWS_MOST], pa[ROWS_MOST];
#pragma unroll
        for (uint32_t j = 0; j < ROWS_MOST; j++) {
            const uint32_t i = min(row_place(rows, j), a.n - 1u);
            au[j] = in.auth[i];
            pa[j] = in.pass[i];
            key[j] = in.peer_out[i];
        }
        uint32_t votes[3] = {0, 0, 0};
#pragma unroll
        for (uint32_t j = 0; j < ROWS_MOST; j++) {
            const uint32_t i = row_place(rows, j);
            const bool there = j < rows && i < a.n;
            const uint8_t v = relay_verdict(in, au[j], pa[j], a.n_keys, key[j]); // (elsewhere: the last packet's again)
            if (there) {
                in.verdict[i] = v;
                if (key[j] == NO_PEER) a.ctr_out[i] = 0;
            } else {
                key[j] = NO_PEER;
            }
            if (in.tally) relay_vote(v, there, votes);
        }
        if (in.tally && lane == 0u) relay_tally(in.tally, votes);
    }
    uint64_t was = 0;
    if (t < a.n_keys) was = a.ctr_base[t];
#pragma unroll
    for (uint32_t k = 0; k < ROW_DIGITS / 64u; k++) mine[k * 64u + lane] = 0u;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t rank[ROWS_MOST]; // among the wave's packets of the peer
#pragma unroll
    for (uint32_t j = 0; j < ROWS_MOST; j++) {
        if (j >= rows) break; // (the same for every lane)
        if (key[j] >= a.n_keys) {
            if (!RELAY && row_place(rows, j) < a.n && !(a.no_peer_ok && key[j] == NO_PEER)) status_raise(a.status, STATUS_PEER_RANGE);
            key[j] = none;
        }
        const unsigned long long same = row_same(key[j], ROW_BITS);
        const uint32_t lower = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
        const uint32_t before = mine[key[j]];
        rank[j] = before + lower;
        // (LDS answers a wave's accesses in order: every lane has read)
        if (lower == 0u) mine[key[j]] = before + (uint32_t)__popcll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    if (t < a.n_keys) { // (fewer than ROW_DIGITS)
        uint32_t c[ROW_WAVES], upto = 0;
#pragma unroll
        for (uint32_t w = 0; w < ROW_WAVES; w++) c[w] = count[w][t];
#pragma unroll
        for (uint32_t w = 0; w < ROW_WAVES; w++) {
            count[w][t] = upto;
            upto += c[w];
        }
        base[t] = was;
        if (a.advance && upto != 0u) a.ctr_base[t] = ctr_add(was, upto, a.ctr_limit);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < ROWS_MOST; j++)
        if (j < rows && key[j] != none) a.ctr_out[row_place(rows, j)] = ctr_add(base[key[j]], mine[key[j]] + rank[j], a.ctr_limit);
}

template <uint32_t FORM>
BNK_DEV void peer_rank(const RankArgs &a)
{
    FORM == RANK_ROWS ? peer_rank_rows<false>(a, RelayIn{}) : FORM == RANK_SMALL ? peer_rank_small(a) : peer_rank_block(a);
}

template <uint32_t FORM>
__global__ __launch_bounds__(PEER_BLOCK_THREADS) void peer_rank_kernel(RankArgs a) { peer_rank<FORM>(a); }

__global__ __launch_bounds__(PEER_BLOCK_THREADS) void relay_rank_rows_kernel(RankArgs a, RelayIn in) { peer_rank_rows<true>(a, in); }

// NoteOutbound on the packets of such a batch as well, which has nothing to do with its counters: the
// first workgroup ranks, the second does what a note launch does once, the others note.  In launches of
// their own, one behind the other (4 us each, and 3 for the host to launch one), device-resident tunnel
// passes of 256 packets took 31.7 us in a row against 29.1, of 3000 70.5 against 65.1; 128 packets in
// pinned rings through the tunnel 67.5 against 63.7.
//
// A workgroup notes no more packets than one of its waves has lanes: the packets' headers are a line each,
// and a compute unit has only so many of them in flight.  With 1024 a workgroup device-resident passes of
// 3000 packets took 50.0 us in a row against 47.6; over the link (a ring's packets, as far as no wave of
// their own notes them) a launch for 1024 took 34 us, and a pass 162 against 154.
constexpr uint32_t NOTE_PER_BLOCK = 64;
template <uint32_t FORM>
__global__ __launch_bounds__(PEER_BLOCK_THREADS) void peer_rank_note_kernel(RankArgs a, FilterArgs note)
{
    if (blockIdx.x == 0u) {
        peer_rank<FORM>(a);
    } else if (blockIdx.x == 1u) {
        if (threadIdx.x == 0u) note_once(note);
    } else {
        const uint32_t i = (blockIdx.x - 2u) * NOTE_PER_BLOCK + threadIdx.x;
        if (threadIdx.x < NOTE_PER_BLOCK && i < note.n) note_packet(note, i);
        note_block_done(note);
    }
}

bool peer_rank_one_block(uint32_t n, uint32_t n_keys)
{
    return n <= PEER_RANK_SMALL_MAX || (n <= PEER_RANK_BLOCK_MAX && key_bits(n_keys) + PEER_BLOCK_INDEX_BITS <= 32u);
}

static hipError_t launch_peer_rank_one_block(const uint32_t *peer, uint32_t n_keys, uint32_t n, uint64_t *ctr_base,
                                             uint64_t *ctr_out, bool advance, bool no_peer_ok, uint64_t ctr_limit,
                                             uint32_t *status, hipStream_t s)
{
    const RankArgs a{peer, n_keys, n, ctr_base, ctr_out, advance ? 1 : 0, no_peer_ok ? 1 : 0, key_bits(n_keys), ctr_limit, status};
    void (*const kernels[])(RankArgs) = {peer_rank_kernel<RANK_SMALL>, peer_rank_kernel<RANK_BLOCK>, peer_rank_kernel<RANK_ROWS>};
    hipLaunchKernelGGL(kernels[rank_form(n, n_keys)], dim3(1), dim3(PEER_BLOCK_THREADS), 0, s, a);
    return hipGetLastError();
}

static hipError_t launch_relay_rank_rows(const RelayIn &in, uint32_t n_keys, uint32_t n, uint64_t *ctr_base, uint64_t *ctr_out,
                                         bool advance, hipStream_t s)
{
    const RankArgs a{nullptr, n_keys, n, ctr_base, ctr_out, advance ? 1 : 0, 1, key_bits(n_keys), 0ull, in.status};
    hipLaunchKernelGGL(relay_rank_rows_kernel, dim3(1), dim3(PEER_BLOCK_THREADS), 0, s, a, in);
    return hipGetLastError();
}

hipError_t launch_peer_rank_small(const uint32_t *peer, uint32_t n_keys, uint32_t n, uint64_t *ctr_base,
                                  uint64_t *ctr_out, bool advance, uint64_t ctr_limit, uint32_t *status,
                                  hipStream_t s)
{
    if (n == 0) return hipSuccess;
    if (!peer_rank_one_block(n, n_keys)) return hipErrorInvalidValue;
    return launch_peer_rank_one_block(peer, n_keys, n, ctr_base, ctr_out, advance, false, ctr_limit, status, s);
}

hipError_t launch_peer_rank_small_note(const uint32_t *peer, uint32_t n_keys, uint32_t n, uint64_t *ctr_base,
                                       uint64_t *ctr_out, uint64_t ctr_limit, uint32_t *status, const FilterArgs &note,
                                       uint32_t max_blocks, uint64_t claimed_upper, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    if (!peer_rank_one_block(n, n_keys) || note.n != n) return hipErrorInvalidValue;
    const RankArgs a{peer, n_keys, n, ctr_base, ctr_out, 1, 0, key_bits(n_keys), ctr_limit, status};
    FilterArgs f = note;
    const uint32_t blocks = (n + NOTE_PER_BLOCK - 1u) / NOTE_PER_BLOCK;
    f.record_blocks = f.record && f.record_after ? blocks : 0u;
    void (*const kernels[])(RankArgs, FilterArgs) = {peer_rank_note_kernel<RANK_SMALL>, peer_rank_note_kernel<RANK_BLOCK>,
                                                     peer_rank_note_kernel<RANK_ROWS>};
    hipLaunchKernelGGL(kernels[rank_form(n, n_keys)], dim3(blocks + 2u), dim3(PEER_BLOCK_THREADS), 0, s, a, f);
    return launch_flow_sweep(f, max_blocks, claimed_upper, s);
}

// ---------------------------------------------------------------------------
// The same counters without a sort, for peer tables of at most
// RANK_TABLE_MAX_KEYS rows.  The batch is cut into tiles of TILE_RUNS runs of
// 64 packets, one wave per tile.  rank_count_kernel counts each tile's packets
// per peer into a row of a table; rank_scan_kernel turns every column (a
// peer's counts, tile after tile) into exclusive prefixes and keeps the
// totals; rank_assign_kernel loads its tile's row into LDS and walks the tile
// run by run in batch order: a packet's rank is its peer's entry plus the
// number of lower lanes of the run with the same peer, and one lane per peer
// then moves the entry past the run.  The scan also moves the peers' counters
// past the batch, leaving the values it found for the assigning launch.
// Three launches over the keys, against eight (two of them passes over
// key-index pairs) for the sort.
// ---------------------------------------------------------------------------
// SHIFTED: the key of a packet is keys[i] >> shift, the last key standing for all beyond it.
__device__ __forceinline__ uint32_t rank_key(uint32_t word, unsigned shift, uint32_t n_keys)
{
    return min(word >> shift, n_keys - 1u);
}

// A tile's words, 64 to a run, every load on its way before the first is used: no branch
// around a load (what a branch leaves unloaded the compiler merges with what was loaded, behind a
// wait in each) but the last word again where a lane has none.  RUNS: the runs that a kernel is
// compiled for; so few in most batches that a form of their own pays.  Together with the walks
// below, which wait for LDS at their end instead of in every run: 2^18 packets of 256 peers,
// assigning 10.8 -> 7.1 us, placing 10.6 -> 9.8, counting 6.4 -> 5.6; 2^22 of 4096 peers,
// assigning 41.2 -> 39.7 (the table's rows, longer than the tile), counting 12.8 -> 11.4.
template <uint32_t RUNS>
__device__ __forceinline__ void tile_words(const uint32_t *words, uint32_t first, uint32_t end, uint32_t (&word)[RUNS])
{
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) word[r] = words[min(first + r * 64u + threadIdx.x, end - 1u)];
}

// A row of the table, in as much LDS as its columns take: beside a launch of a lane per packet, which leaves
// a compute unit 21 KiB, room for the longest row would be room for one wave of these.  With other streams at
// work, against 16 KiB for every table: a relay of 2.7 million packets of 5 peers 1346 -> 1340 us, tunnel passes
// of 2^18 packets of 1024 peers 440.7 -> 437.8, the relay of 4096 peers, whose rows are that long, the same.
extern __shared__ __attribute__((aligned(16))) uint32_t rank_row[];

// RELAY: of a relay's batch, whose verdicts come first, and whose keys[] are written here.
template <bool SHIFTED, bool RELAY, uint32_t RUNS>
__device__ __forceinline__ void rank_count_tile(uint32_t tile, const uint32_t *keys, uint32_t n, uint32_t n_keys, uint32_t cols,
                                                uint32_t runs, uint32_t *table, uint32_t *status, unsigned shift, const RelayIn &in)
{
    uint32_t *const cnt = rank_row;
    const uint32_t lane = threadIdx.x;
    uint4 *cnt4 = reinterpret_cast<uint4 *>(cnt);
    for (uint32_t q = lane; q < cols / 4u; q += 64u) cnt4[q] = make_uint4(0, 0, 0, 0);
    const uint32_t first = tile * runs * 64u, end = min(n, first + runs * 64u);
    uint32_t word[RUNS];
    tile_words(RELAY ? in.peer_out : keys, first, end, word);
    if (RELAY) {
        uint8_t au[RUNS], pa[RUNS];
#pragma unroll
        for (uint32_t r = 0; r < RUNS; r++) {
            const uint32_t i = min(first + r * 64u + lane, end - 1u);
            au[r] = in.auth[i];
            pa[r] = in.pass[i];
        }
        uint32_t votes[3] = {0, 0, 0};
#pragma unroll
        for (uint32_t r = 0; r < RUNS; r++) {
            if (first + r * 64u >= end) break; // (the same for every lane)
            const uint32_t i = first + r * 64u + lane;
            const uint8_t v = relay_verdict(in, au[r], pa[r], n_keys, word[r]); // (beyond the end: the last packet's again)
            if (i < end) {
                in.verdict[i] = v;
                in.keys[i] = word[r];
            }
            if (in.tally) relay_vote(v, i < end, votes);
        }
        if (in.tally && lane == 0u) relay_tally(in.tally, votes);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        if (first + r * 64u + lane >= end) break;
        const uint32_t key = SHIFTED ? rank_key(word[r], shift, n_keys) : word[r];
        if (key < n_keys) atomicAdd(&cnt[key], 1u);
        // (keys straight from a caller's peer array: one beyond the table gets no counter and is reported)
        else if (status) status_raise(status, STATUS_PEER_RANGE);
    }
    __syncthreads();
    uint4 *row = reinterpret_cast<uint4 *>(table + (size_t)tile * cols);
    for (uint32_t q = lane; q < cols / 4u; q += 64u) row[q] = cnt4[q];
}

template <bool SHIFTED, uint32_t RUNS>
__global__ __launch_bounds__(64) void rank_count_kernel(const uint32_t *keys, uint32_t n, uint32_t n_keys,
                                                        uint32_t cols, uint32_t runs, uint32_t *table,
                                                        uint32_t *status, unsigned shift)
{
    rank_count_tile<SHIFTED, false, RUNS>(blockIdx.x, keys, n, n_keys, cols, runs, table, status, shift, RelayIn{});
}

template <uint32_t RUNS>
__global__ __launch_bounds__(64) void relay_count_kernel(RelayIn in, uint32_t n, uint32_t n_keys, uint32_t cols, uint32_t runs, uint32_t *table)
{
    rank_count_tile<false, true, RUNS>(blockIdx.x, nullptr, n, n_keys, cols, runs, table, nullptr, 0u, in);
}

// One block per 16 peers: 64 groups of threads share the tiles between them.
constexpr uint32_t SCAN_PEERS = 16, SCAN_PARTS = 64;
constexpr uint32_t SCAN_KEEP = 32; // tiles of a part held in registers between the two passes
__global__ __launch_bounds__(SCAN_PEERS * SCAN_PARTS) void rank_scan_kernel(uint32_t *table, uint32_t tiles,
                                                                             uint32_t n_keys, uint32_t cols,
                                                                             uint32_t *total, uint64_t *ctr_base,
                                                                             uint64_t *base_was, int advance,
                                                                             uint64_t ctr_limit)
{
    __shared__ uint32_t part_sum[SCAN_PARTS][SCAN_PEERS];
    const uint32_t x = threadIdx.x % SCAN_PEERS, y = threadIdx.x / SCAN_PEERS;
    const uint32_t key = blockIdx.x * SCAN_PEERS + x;
    const uint32_t per = (tiles + SCAN_PARTS - 1u) / SCAN_PARTS;
    const uint32_t lo = min(y * per, tiles), hi = min(lo + per, tiles);
    const bool mine = key < n_keys;
    const bool keep = per <= SCAN_KEEP; // (the same for every thread)
    uint32_t c[SCAN_KEEP];
    uint32_t sum = 0;
    if (keep) {
        // every load of the part in flight at once
#pragma unroll
        for (uint32_t j = 0; j < SCAN_KEEP; j++) c[j] = mine && lo + j < hi ? table[(size_t)(lo + j) * cols + key] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < SCAN_KEEP; j++) sum += c[j];
    } else if (mine) {
#pragma unroll 8
        for (uint32_t t = lo; t < hi; t++) sum += table[(size_t)t * cols + key];
    }
    part_sum[y][x] = sum;
    __syncthreads();
    uint32_t run = 0;
    for (uint32_t q = 0; q < y; q++) run += part_sum[q][x];
    if (!mine) return;
    if (keep) {
#pragma unroll
        for (uint32_t j = 0; j < SCAN_KEEP; j++) {
            if (lo + j < hi) table[(size_t)(lo + j) * cols + key] = run;
            run += c[j];
        }
    } else {
        for (uint32_t t = lo; t < hi; t++) {
            uint32_t *e = table + (size_t)t * cols + key;
            const uint32_t v = *e;
            *e = run;
            run += v;
        }
    }
    if (y == SCAN_PARTS - 1u) {
        // the peer's counter as the batch found it stays behind for the assigning launch;
        // the counter itself moves past what the batch takes
        total[key] = run;
        if (ctr_base == nullptr) return;
        const uint64_t was = ctr_base[key];
        base_was[key] = was;
        if (advance && run != 0u) ctr_base[key] = ctr_add(was, run, ctr_limit);
    }
}

// The walk over a tile, by one wave, in batch order: for every packet what stands at its key in
// `before` once the lower runs have moved it (old), and how many lower lanes of its run have the key.
// A key beyond n_keys is nobody's.
template <uint32_t RUNS>
__device__ __forceinline__ void tile_walk(uint32_t *before, const uint32_t (&key)[RUNS], uint32_t first, uint32_t end, uint32_t n_keys,
                                          unsigned bits, uint32_t (&old)[RUNS], uint32_t (&lower)[RUNS])
{
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        old[r] = lower[r] = 0u;
        if (first + r * 64u < end) { // uniform
            const uint32_t kk = key[r];
            const bool valid = kk < n_keys;
            // the lanes of this run with my peer
            unsigned long long same = __ballot(valid);
            for (unsigned b = 0; b < bits; b++) {
                const unsigned long long m = __ballot((kk >> b) & 1u);
                same &= ((kk >> b) & 1u) ? m : ~m;
            }
            lower[r] = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
            // every lane reads its entry before the one lane of each peer moves it: LDS serves a
            // wave's accesses in order, so nothing is waited for from run to run
            old[r] = before[min(kk, n_keys - 1u)];
            if (valid && lower[r] == 0u) atomicAdd(&before[kk], (uint32_t)__popcll(same));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
}

template <uint32_t RUNS>
__global__ __launch_bounds__(64) void rank_assign_kernel(const uint32_t *keys, uint32_t n, uint32_t n_keys,
                                                         uint32_t cols, uint32_t runs, const uint32_t *table,
                                                         unsigned bits,
                                                         const uint64_t *ctr_base, uint64_t *ctr_out,
                                                         uint64_t ctr_limit, int zero_others)
{
    // packets of each peer ahead of the run at hand
    uint32_t *const before = rank_row;
    const uint32_t lane = threadIdx.x;
    const uint32_t first = blockIdx.x * runs * 64u, end = min(n, first + runs * 64u);
    // keys and the peers' bases are fetched up front: nothing inside the walk below waits for memory
    uint32_t key[RUNS];
    tile_words(keys, first, end, key);
    {
        // the tile's row, every load in flight before the first is used
        const uint4 *row = reinterpret_cast<const uint4 *>(table + (size_t)blockIdx.x * cols);
        uint4 v[RANK_ROW_STEPS];
#pragma unroll
        for (uint32_t q = 0; q < RANK_ROW_STEPS; q++)
            v[q] = q * RANK_ROW_STEP < cols ? row[q * 64u + lane] : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (uint32_t q = 0; q < RANK_ROW_STEPS; q++)
            if (q * RANK_ROW_STEP < cols) reinterpret_cast<uint4 *>(before)[q * 64u + lane] = v[q];
    }
    uint64_t base[RUNS];
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        if (first + r * 64u + lane >= end) key[r] = NO_PEER;
        base[r] = ctr_base[min(key[r], n_keys - 1u)];
    }
    __syncthreads();
    uint32_t old[RUNS], lower[RUNS];
    tile_walk(before, key, first, end, n_keys, bits, old, lower);
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        const uint32_t i = first + r * 64u + lane;
        // (a packet without a peer gets no counter)
        const bool valid = key[r] < n_keys;
        if (i < end && (valid || zero_others)) ctr_out[i] = valid ? ctr_add(base[r], old[r] + lower[r], ctr_limit) : 0ull;
    }
}

// The third launch when the batch is to be sorted by key, stably (three launches where the
// library's radix sort takes five to nine with its memsets: a tunnel pass of 16000 packets of
// 100 bytes 100 -> 92 us, 2^17 151 -> 133, 2^18 201 -> 184, 2^20 472 -> 457): a packet's place is where its
// key's packets begin (every tile scans the totals for itself) plus its rank among them.
template <uint32_t RUNS>
__global__ __launch_bounds__(64) void rank_place_kernel(const uint32_t *words, uint32_t n, uint32_t n_keys,
                                                        uint32_t cols, uint32_t runs, const uint32_t *table,
                                                        const uint32_t *total, unsigned bits, unsigned shift,
                                                        uint32_t *sorted)
{
    uint32_t *const before = rank_row;
    const uint32_t lane = threadIdx.x;
    const uint32_t first = blockIdx.x * runs * 64u, end = min(n, first + runs * 64u);
    uint32_t word[RUNS];
    tile_words(words, first, end, word);
    {
        const uint4 *const row = reinterpret_cast<const uint4 *>(table + (size_t)blockIdx.x * cols);
        const uint4 *const tot = reinterpret_cast<const uint4 *>(total);
        uint32_t base = 0;
        for (uint32_t q = 0; q < cols / RANK_ROW_STEP; q++) {
            // (columns beyond the keys hold nothing that was written)
            const uint32_t c = (q * 64u + lane) * 4u;
            uint4 t = tot[q * 64u + lane], v = row[q * 64u + lane];
            if (c >= n_keys) t.x = 0;
            if (c + 1u >= n_keys) t.y = 0;
            if (c + 2u >= n_keys) t.z = 0;
            if (c + 3u >= n_keys) t.w = 0;
            const uint32_t mine = t.x + t.y + t.z + t.w;
            uint32_t inc = mine;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t o = (uint32_t)__shfl_up((int)inc, off, 64);
                if ((int)lane >= off) inc += o;
            }
            const uint32_t s0 = base + inc - mine;
            v.x += s0;
            v.y += s0 + t.x;
            v.z += s0 + t.x + t.y;
            v.w += s0 + t.x + t.y + t.z;
            reinterpret_cast<uint4 *>(before)[q * 64u + lane] = v;
            base += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
        }
    }
    __syncthreads();
    uint32_t key[RUNS], at[RUNS], lower[RUNS];
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) key[r] = first + r * 64u + lane < end ? rank_key(word[r], shift, n_keys) : NO_PEER;
    tile_walk(before, key, first, end, n_keys, bits, at, lower);
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++)
        if (first + r * 64u + lane < end) sorted[at[r] + lower[r]] = word[r];
}

// ---------------------------------------------------------------------------
// The same in two launches, of batches whose table is so short that every tile adds up the rows
// before its own by itself: up to WHOLE_TILES tiles, as long as a wave keeps their packets' words, and
// WHOLE_MAX_KEYS keys.  In batches of this size a launch costs more than what it does (the scan by itself 5
// us and the gap to the next launch 2).  Device-resident tunnel passes of IMIX packets of 64 peers with three
// streams at work, 15 launches -> 10, together with the windows' bits in the filter's launch: 4097 packets
// 50.4 -> 37.8 us, 8192 48.6 -> 38.5, 16384 50.1 -> 40.1, 32768 61.6 -> 54.5.  The counting launch leaves the peers' counters as the batch
// found them, so that the assigning one can move them while it reads; it also takes NoteOutbound of the
// batch along, which nothing of all this needs, and the assigning one the sweep behind that.
// ---------------------------------------------------------------------------
constexpr uint32_t WHOLE_TILES = 64, WHOLE_MAX_KEYS = 1024, WHOLE_THREADS = 256;
static_assert(WHOLE_THREADS == SWEEP_THREADS && WHOLE_THREADS == RANK_ROW_STEP && WHOLE_TILES % 4u == 0u, "one launch; a thread a column");

static bool rank_whole_plan(uint32_t n, uint32_t n_keys, RankPlan &p)
{
    if (n > WHOLE_TILES * 64u * TILE_RUNS_FEW || n_keys > WHOLE_MAX_KEYS) return false;
    p.runs = (n + 64u * WHOLE_TILES - 1u) / (64u * WHOLE_TILES);
    p.tiles = (n + 64u * p.runs - 1u) / (64u * p.runs);
    return true; // (never more tiles than rank_plan has: its scratch holds them)
}

// What stands in the columns of the first `upto` of the table's rows, and in all of them, by the
// workgroup's four waves: a quarter of the rows each, all of a step's loads in flight at once.
template <bool BELOW, bool ALL>
__device__ __forceinline__ void rows_sum(const uint32_t *table, uint32_t cols, uint32_t tiles, uint32_t upto, uint32_t *below, uint32_t *all)
{
    __shared__ __attribute__((aligned(16))) uint32_t part[2][WHOLE_THREADS / 64u][RANK_ROW_STEP];
    constexpr uint32_t WAVES = WHOLE_THREADS / 64u, PER = WHOLE_TILES / WAVES;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, rows = ALL ? tiles : upto;
    for (uint32_t q = 0; q < cols; q += RANK_ROW_STEP) {
        uint4 v[PER];
#pragma unroll
        for (uint32_t j = 0; j < PER; j++)
            v[j] = *reinterpret_cast<const uint4 *>(table + (size_t)min(wave + WAVES * j, tiles - 1u) * cols + q + 4u * lane);
        uint4 b = make_uint4(0, 0, 0, 0), s = b;
#pragma unroll
        for (uint32_t j = 0; j < PER; j++) {
            const uint32_t row = wave + WAVES * j;
            if (row < rows) { s.x += v[j].x; s.y += v[j].y; s.z += v[j].z; s.w += v[j].w; }
            if (BELOW && row < upto) { b.x += v[j].x; b.y += v[j].y; b.z += v[j].z; b.w += v[j].w; }
        }
        if (ALL) *reinterpret_cast<uint4 *>(&part[0][wave][4u * lane]) = s;
        if (BELOW) *reinterpret_cast<uint4 *>(&part[1][wave][4u * lane]) = b;
        __syncthreads();
        const uint32_t t = threadIdx.x;
        if (ALL) all[q + t] = part[0][0][t] + part[0][1][t] + part[0][2][t] + part[0][3][t];
        if (BELOW) below[q + t] = part[1][0][t] + part[1][1][t] + part[1][2][t] + part[1][3][t];
        __syncthreads();
    }
}

struct WholeArgs {
    const uint32_t *keys;
    uint32_t n, n_keys, cols, runs, tiles;
    uint32_t *table;
    uint64_t *ctr_base, *base_was;
    uint32_t *status;
};

// Workgroups: the tiles, the peers' counters, then those of NoteOutbound (note_once, and a packet a lane).
template <uint32_t RUNS>
__global__ __launch_bounds__(64) void rank_count_whole_kernel(WholeArgs a, FilterArgs note)
{
    const uint32_t b = blockIdx.x;
    if (b < a.tiles) {
        rank_count_tile<false, false, RUNS>(b, a.keys, a.n, a.n_keys, a.cols, a.runs, a.table, a.status, 0u, RelayIn{});
    } else if (b == a.tiles) {
        for (uint32_t k = threadIdx.x; k < a.n_keys; k += 64u) a.base_was[k] = a.ctr_base[k];
    } else if (b == a.tiles + 1u) {
        if (threadIdx.x == 0u) note_once(note);
    } else {
        const uint32_t i = (b - a.tiles - 2u) * 64u + threadIdx.x;
        if (i < note.n) note_packet(note, i);
        note_block_done(note);
    }
}

// The same of a relay's batch, with its verdicts.
template <uint32_t RUNS>
__global__ __launch_bounds__(64) void relay_count_whole_kernel(WholeArgs a, RelayIn in)
{
    if (blockIdx.x < a.tiles) rank_count_tile<false, true, RUNS>(blockIdx.x, nullptr, a.n, a.n_keys, a.cols, a.runs, a.table, nullptr, 0u, in);
    else
        for (uint32_t k = threadIdx.x; k < a.n_keys; k += 64u) a.base_was[k] = a.ctr_base[k];
}

// Workgroups: the tiles, one that moves the peers' counters (with advance), the sweep's.
template <uint32_t RUNS>
__global__ __launch_bounds__(WHOLE_THREADS) void rank_assign_whole_kernel(WholeArgs a, unsigned bits, uint64_t *ctr_out, uint64_t ctr_limit,
                                                                          int zero_others, int advance, SweepArgs sweep)
{
    __shared__ uint32_t before[WHOLE_MAX_KEYS];
    const uint32_t b = blockIdx.x;
    if (b > a.tiles) {
        flow_sweep(sweep, b - a.tiles - 1u);
        return;
    }
    if (b == a.tiles) {
        if (!advance) return;
        rows_sum<false, true>(a.table, a.cols, a.tiles, 0u, nullptr, before);
        for (uint32_t k = threadIdx.x; k < a.n_keys; k += WHOLE_THREADS)
            if (before[k] != 0u) a.ctr_base[k] = ctr_add(a.base_was[k], before[k], ctr_limit);
        return;
    }
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t first = b * a.runs * 64u, end = min(a.n, first + a.runs * 64u);
    uint32_t key[RUNS];
    uint64_t base[RUNS];
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        const uint32_t i = first + r * 64u + lane, k = a.keys[min(i, end - 1u)];
        key[r] = i < end ? k : NO_PEER;
    }
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) base[r] = a.base_was[min(key[r], a.n_keys - 1u)];
    rows_sum<true, false>(a.table, a.cols, a.tiles, b, before, nullptr);
    if (threadIdx.x >= 64u) return;
    uint32_t old[RUNS], lower[RUNS];
    tile_walk(before, key, first, end, a.n_keys, bits, old, lower);
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) {
        const uint32_t i = first + r * 64u + lane;
        const bool valid = key[r] < a.n_keys;
        if (i < end && (valid || zero_others)) ctr_out[i] = valid ? ctr_add(base[r], old[r] + lower[r], ctr_limit) : 0ull;
    }
}

// The second launch when the batch is to be sorted (rank_place_kernel).
template <uint32_t RUNS>
__global__ __launch_bounds__(WHOLE_THREADS) void rank_place_whole_kernel(const uint32_t *words, uint32_t n, uint32_t n_keys, uint32_t cols,
                                                                         uint32_t runs, uint32_t tiles, const uint32_t *table,
                                                                         unsigned bits, unsigned shift, uint32_t *sorted)
{
    __shared__ uint32_t before[WHOLE_MAX_KEYS], total[WHOLE_MAX_KEYS];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t first = blockIdx.x * runs * 64u, end = min(n, first + runs * 64u);
    uint32_t word[RUNS];
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) word[r] = words[min(first + r * 64u + lane, end - 1u)];
    rows_sum<true, true>(table, cols, tiles, blockIdx.x, before, total);
    if (threadIdx.x >= 64u) return;
    // where each key's packets begin
    uint32_t base = 0;
    for (uint32_t q = 0; q < cols; q += RANK_ROW_STEP) {
        const uint32_t c = q + 4u * lane; // (columns beyond the keys are all 0)
        const uint32_t t0 = total[c], t1 = total[c + 1u], t2 = total[c + 2u], t3 = total[c + 3u], mine = t0 + t1 + t2 + t3;
        uint32_t inc = mine;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)inc, off, 64);
            if ((int)lane >= off) inc += o;
        }
        const uint32_t s0 = base + inc - mine;
        before[c] += s0;
        before[c + 1u] += s0 + t0;
        before[c + 2u] += s0 + t0 + t1;
        before[c + 3u] += s0 + t0 + t1 + t2;
        base += (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t key[RUNS], at[RUNS], lower[RUNS];
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++) key[r] = first + r * 64u + lane < end ? rank_key(word[r], shift, n_keys) : NO_PEER;
    tile_walk(before, key, first, end, n_keys, bits, at, lower);
#pragma unroll
    for (uint32_t r = 0; r < RUNS; r++)
        if (first + r * 64u + lane < end) sorted[at[r] + lower[r]] = word[r];
}

// One key more than there are peers: the packets without one, last.
static RankPlan sort_plan(uint32_t n, uint32_t n_peers)
{
    RankPlan p = rank_plan(n, n_peers + 1u);
    p.fits = p.fits && n_peers + 1u <= PEER_SORT_MAX_KEYS;
    return p;
}

size_t peer_sort_tmp_bytes(uint32_t n, uint32_t n_peers)
{
    const RankPlan p = sort_plan(n, n_peers);
    return p.fits ? p.bytes : 0;
}

hipError_t launch_peer_sort(const uint32_t *words, uint32_t *sorted, uint32_t n, uint32_t n_peers, unsigned shift,
                            void *tmp, hipStream_t s)
{
    RankPlan plan = sort_plan(n, n_peers);
    const uint32_t n_keys = n_peers + 1u;
    if (rank_whole_plan(n, n_keys, plan)) {
        uint32_t *const table = static_cast<uint32_t *>(tmp);
        hipLaunchKernelGGL((rank_count_kernel<true, TILE_RUNS_FEW>), dim3(plan.tiles), dim3(64), plan.cols * 4u, s, words, n, n_keys, plan.cols, plan.runs,
                           table, (uint32_t *)nullptr, shift);
        hipLaunchKernelGGL(rank_place_whole_kernel<TILE_RUNS_FEW>, dim3(plan.tiles), dim3(WHOLE_THREADS), 0, s, words, n, n_keys, plan.cols,
                           plan.runs, plan.tiles, table, key_bits(n_keys), shift, sorted);
        return hipGetLastError();
    }
    uint32_t *table = static_cast<uint32_t *>(tmp), *total = table + (size_t)plan.tiles * plan.cols;
    const auto count = plan.runs <= TILE_RUNS_FEW ? rank_count_kernel<true, TILE_RUNS_FEW> : rank_count_kernel<true, TILE_RUNS_MAX>;
    const auto place = plan.runs <= TILE_RUNS_FEW ? rank_place_kernel<TILE_RUNS_FEW> : rank_place_kernel<TILE_RUNS_MAX>;
    hipLaunchKernelGGL(count, dim3(plan.tiles), dim3(64), plan.cols * 4u, s, words, n, n_keys, plan.cols, plan.runs, table,
                       (uint32_t *)nullptr, shift);
    hipLaunchKernelGGL(rank_scan_kernel, dim3((n_keys + SCAN_PEERS - 1u) / SCAN_PEERS), dim3(SCAN_PEERS * SCAN_PARTS), 0, s,
                       table, plan.tiles, n_keys, plan.cols, total, (uint64_t *)nullptr, (uint64_t *)nullptr, 0, 0ull);
    hipLaunchKernelGGL(place, dim3(plan.tiles), dim3(64), plan.cols * 4u, s, words, n, n_keys, plan.cols, plan.runs, table,
                       total, key_bits(n_keys), shift, sorted);
    return hipGetLastError();
}

// note: null, or the batch's NoteOutbound, with the sweep behind it.
static hipError_t launch_peer_rank_whole(const uint32_t *keys, const RankPlan &plan, void *tmp, uint64_t *ctr_base, uint32_t n_keys,
                                         uint32_t n, uint64_t *ctr_out, bool advance, uint64_t ctr_limit, bool zero_others,
                                         uint32_t *status, const FilterArgs *note, const SweepArgs &sweep, const RelayIn *relay,
                                         hipStream_t s)
{
    uint32_t *const table = static_cast<uint32_t *>(tmp);
    uint64_t *const base_was = reinterpret_cast<uint64_t *>(table + (size_t)plan.tiles * plan.cols);
    const WholeArgs a{keys, n, n_keys, plan.cols, plan.runs, plan.tiles, table, ctr_base, base_was, status};
    const uint32_t noting = note ? 1u + (note->n + 63u) / 64u : 0u;
    if (relay) hipLaunchKernelGGL(relay_count_whole_kernel<TILE_RUNS_FEW>, dim3(plan.tiles + 1u), dim3(64), plan.cols * 4u, s, a, *relay);
    else hipLaunchKernelGGL(rank_count_whole_kernel<TILE_RUNS_FEW>, dim3(plan.tiles + 1u + noting), dim3(64), plan.cols * 4u, s, a, note ? *note : FilterArgs{});
    hipLaunchKernelGGL(rank_assign_whole_kernel<TILE_RUNS_FEW>, dim3(plan.tiles + 1u + sweep.blocks), dim3(WHOLE_THREADS), 0, s, a,
                       key_bits(n_keys), ctr_out, ctr_limit, zero_others ? 1 : 0, advance ? 1 : 0, sweep);
    return hipGetLastError();
}

bool peer_rank_whole(uint32_t n, uint32_t n_keys)
{
    RankPlan p{};
    return rank_whole_plan(n, n_keys, p);
}

hipError_t launch_peer_rank_counting_note(const uint32_t *peer, void *tmp, uint64_t *ctr_base, uint32_t n_keys, uint32_t n,
                                          uint64_t *ctr_out, uint64_t ctr_limit, uint32_t *status, const FilterArgs &note,
                                          uint32_t max_blocks, uint64_t claimed_upper, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    RankPlan plan = rank_plan(n, n_keys);
    if (!rank_whole_plan(n, n_keys, plan) || note.n != n) return hipErrorInvalidValue;
    FilterArgs f = note;
    const SweepArgs sweep = flow_sweep_args(f, max_blocks, claimed_upper);
    f.record_blocks = f.record && f.record_after && sweep.blocks == 0u ? (n + 63u) / 64u : 0u;
    return launch_peer_rank_whole(peer, plan, tmp, ctr_base, n_keys, n, ctr_out, true, ctr_limit, true, status, &f, sweep, nullptr, s);
}

static hipError_t launch_peer_rank_table(const uint32_t *keys, const RankPlan &plan, void *tmp,
                                         uint64_t *ctr_base, uint32_t n_keys, uint32_t n, uint64_t *ctr_out,
                                         bool advance, uint64_t ctr_limit, bool zero_others, uint32_t *status,
                                         const RelayIn *relay, hipStream_t s)
{
    RankPlan whole = plan;
    if (rank_whole_plan(n, n_keys, whole))
        return launch_peer_rank_whole(keys, whole, tmp, ctr_base, n_keys, n, ctr_out, advance, ctr_limit, zero_others, status, nullptr,
                                      SweepArgs{}, relay, s);
    uint32_t *table = static_cast<uint32_t *>(tmp);
    uint32_t *total = table + (size_t)plan.tiles * plan.cols;
    uint64_t *base_was = reinterpret_cast<uint64_t *>(total + plan.cols);
    const auto count = plan.runs <= TILE_RUNS_FEW ? rank_count_kernel<false, TILE_RUNS_FEW> : rank_count_kernel<false, TILE_RUNS_MAX>;
    const auto assign = plan.runs <= TILE_RUNS_FEW ? rank_assign_kernel<TILE_RUNS_FEW> : rank_assign_kernel<TILE_RUNS_MAX>;
    if (relay)
        hipLaunchKernelGGL((plan.runs <= TILE_RUNS_FEW ? relay_count_kernel<TILE_RUNS_FEW> : relay_count_kernel<TILE_RUNS_MAX>), dim3(plan.tiles),
                           dim3(64), plan.cols * 4u, s, *relay, n, n_keys, plan.cols, plan.runs, table);
    else
        hipLaunchKernelGGL(count, dim3(plan.tiles), dim3(64), plan.cols * 4u, s, keys, n, n_keys, plan.cols, plan.runs, table, status, 0u);
    hipLaunchKernelGGL(rank_scan_kernel, dim3((n_keys + SCAN_PEERS - 1u) / SCAN_PEERS),
                       dim3(SCAN_PEERS * SCAN_PARTS), 0, s, table, plan.tiles, n_keys, plan.cols, total, ctr_base,
                       base_was, advance ? 1 : 0, ctr_limit);
    hipLaunchKernelGGL(assign, dim3(plan.tiles), dim3(64), plan.cols * 4u, s, keys, n, n_keys, plan.cols, plan.runs,
                       table, key_bits(n_keys), base_was, ctr_out, ctr_limit, zero_others ? 1 : 0);
    return hipGetLastError();
}

bool peer_rank_counts(uint32_t n, uint32_t n_keys, size_t tmp_bytes)
{
    const RankPlan plan = rank_plan(n, n_keys);
    return !peer_rank_one_block(n, n_keys) && plan.fits && plan.bytes <= tmp_bytes;
}

hipError_t launch_peer_rank_counting(const uint32_t *peer, void *tmp, uint64_t *ctr_base, uint32_t n_keys, uint32_t n,
                                     uint64_t *ctr_out, bool advance, uint64_t ctr_limit, uint32_t *status,
                                     hipStream_t s)
{
    if (n == 0) return hipSuccess;
    // (a packet whose peer lies beyond the table gets counter 0, as one without a peer does)
    return launch_peer_rank_table(peer, rank_plan(n, n_keys), tmp, ctr_base, n_keys, n, ctr_out, advance, ctr_limit,
                                  true, status, nullptr, s);
}

hipError_t launch_peer_rank(uint32_t *keys, uint32_t *idx, uint32_t *skeys, uint32_t *sidx,
                            void *sort_tmp, size_t sort_tmp_bytes, uint64_t *ctr_base, uint32_t n_keys,
                            uint32_t n, uint64_t *ctr_out, bool advance, uint64_t ctr_limit, hipStream_t s)
{
    if (n == 0) return hipSuccess;
    const RankPlan plan = rank_plan(n, n_keys);
    if (plan.fits && plan.bytes <= sort_tmp_bytes)
        return launch_peer_rank_table(keys, plan, sort_tmp, ctr_base, n_keys, n, ctr_out, advance, ctr_limit, false,
                                      nullptr, nullptr, s);
    const dim3 grid((n + 255u) / 256u);
    hipError_t e = rocprim::radix_sort_pairs<SortConfig>(sort_tmp, sort_tmp_bytes, keys, skeys, idx, sidx, (size_t)n,
                                             0, key_bits(n_keys), s);
    if (e != hipSuccess) return e;
    uint32_t *seg_start = static_cast<uint32_t *>(sort_tmp);
    hipLaunchKernelGGL(peer_heads_kernel, grid, dim3(256), 0, s, skeys, n, seg_start);
    hipLaunchKernelGGL(relay_rank_kernel, grid, dim3(256), 0, s, skeys, sidx, seg_start, ctr_base, n, ctr_out,
                       ctr_limit);
    if (advance)
        hipLaunchKernelGGL(peer_advance_kernel, grid, dim3(256), 0, s, skeys, sidx, ctr_out, n, ctr_base,
                           ctr_limit);
    return hipGetLastError();
}

} // namespace bnk
