// Device-side views of the filter's tables, shared by kernels and host code.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wg_dev.hpp"

namespace bnk {

constexpr uint32_t FLOW_REGIONS = 6;     // protocol class (3) x top address bit (2)
constexpr int64_t FLOW_TOMB = INT64_MIN; // expiry of a deleted (or never used) slot
// Words of FlowTableDev::counters: entries in the map, slots ever claimed; since the last note
// launch, whether a sweep ran and how many entries it deleted (FLOW_LIVE still counts those);
// and two int64, no entry of the map expires before FLOW_MIN_EXP (0: nothing known), or before
// FLOW_NEXT_EXP if a sweep ran.  FLOW_NOTE_BLOCKS: see FilterArgs::record_blocks (0 between launches).
enum : uint32_t {
    FLOW_LIVE = 0, FLOW_CLAIMED = 1, FLOW_SWEPT = 2, FLOW_GONE = 3, FLOW_MIN_EXP = 4, FLOW_NEXT_EXP = 6, FLOW_NOTE_BLOCKS = 8,
    FLOW_COUNTERS = 10
};
constexpr uint32_t FLOW_SWEEP_ABOVE = 4096; // filter.go:202: no sweep while the map holds at most so many entries
constexpr int64_t FLOW_TTL_LEAST = 30000000000LL; // filter.go:108-117: nothing is stored for less

// One 16-byte slot, so a probe is a single memory transaction.
struct FlowSlotMem {
    uint64_t key; // 0 = empty
    int64_t exp;  // expiry in Unix ns, FLOW_TOMB = not in the map
};

struct FlowTableDev {
    FlowSlotMem *slots; // [FLOW_REGIONS * cap]
    uint32_t *counters; // [FLOW_COUNTERS]
    uint32_t *list;     // [cap / 2] the slots ever claimed, in the order they were: what walks the
                        // whole map walks this instead of FLOW_REGIONS * cap slots
    uint32_t *present;  // [present_bits / 32] one hashed bit per key ever stored in this table:
                        // small enough to stay in L2, it answers most misses without a probe
    uint32_t *present_small; // [SMALL_BITS / 32] two hashed bits per key (a Bloom filter) in a
                             // size a workgroup can hold in LDS beside the cut points: with
                             // few enough keys the check kernel asks this one and never
                             // leaves the CU for a packet without a flow
    uint32_t cap;       // slots per region, a power of two
    uint32_t present_mask; // present_bits - 1 (a power of two)
};

constexpr uint32_t SMALL_BITS = 44u * 1024u * 8u; // 44 KiB: leaves 36 KiB of a workgroup's 80 for cut points
constexpr uint32_t SMALL_KEYS_MAX = 3u << 16;     // beyond this a clear answer gets too rare (false
                                                  // positives pass 43 %) and the large bitmap is asked

// A range of ports in a word, first | (0xFFFF - last) << 16, with first <= last; so these two are none,
// and have no port.
constexpr uint32_t RANGE_PAD = 0xFFFFFFFFu;
constexpr uint32_t RANGE_LONG = 0xFFFEFFFFu; // first word of a block that only points on
constexpr uint32_t RANGE_BLOCK = 16;         // entries per 64-byte block
constexpr uint32_t RANGE_CLASSES = 3;        // icmp, tcp, udp
constexpr uint32_t JUMP_BUCKETS = 1024;

struct RuleIndexDev {
    const uint32_t *bounds; // [n_bounds] ascending starts of the elementary source intervals
    const uint32_t *ranges; // 64-byte blocks of RANGE_BLOCK one-word ranges of ports, sorted,
                            // disjoint, padded with RANGE_PAD.  Block RANGE_CLASSES * j + c is
                            // interval j's list for class c, so finding the interval finds the
                            // list.  A list of more than RANGE_BLOCK ranges lives in blocks past
                            // the first RANGE_CLASSES * n_bounds, and its block is {RANGE_LONG,
                            // first block, blocks}
    const uint4 *wide;      // [n_wide] (net, mask, key_lo, key_hi) scanned by every packet
    const uint16_t *jump;   // [JUMP_BUCKETS + 1] when n_bounds fits 16 bits, else null: the cut
                            // points from bounds[1] up are spread over equal address buckets
                            // and jump[b] is the last cut point at or below bucket b's start,
                            // so a search only has to look between jump[b] and jump[b + 1]
    uint32_t jump_lo;       // bounds[1]
    uint32_t jump_shift;    // bucket of src = (src - jump_lo) >> jump_shift
    uint32_t n_bounds;
    uint32_t top_step;      // largest power of two < n_bounds (0 when n_bounds == 1)
    uint32_t n_wide;
    bool long_lists;        // some interval's list is longer than a block
};

struct FilterArgs {
    const uint8_t *pkts;
    const uint64_t *off;  // or nullptr: i * stride
    const uint32_t *lens; // or nullptr: len
    const uint8_t *gate;  // or nullptr; gate[i] == 0 skips packet i (verdict 0)
    const uint8_t *heads; // check only, or nullptr: the records AeadArgs::heads describes.  With
                          // them the kernel goes through the records (record t is packet
                          // order[t], or t), takes length and authenticity from them (lens
                          // and gate are not read) and looks at the packet itself only for
                          // an IP header with options
    const uint32_t *order; // with heads, or nullptr
    uint8_t *verdict;     // check only
    uint8_t *wg_result;   // check only, or nullptr: the BNK_WG_* results of the decapsulation that
                          // delivered these packets; a denied packet's BNK_WG_OK becomes BNK_WG_FILTERED
    unsigned long long *tally; // check only, or nullptr: the launch counts its verdicts here
                          // (TALLY_ALLOWED / TALLY_DENIED, see tally_bump)
    unsigned long long *wg_tally; // with wg_result, or nullptr: the launch counts the results here as
                          // it leaves them (decap_slot, and TALLY_ALLOWED for what was delivered)
    uint32_t *status;
    int64_t now;
    uint32_t n, stride, len;
    uint64_t limit;       // arena size for device-resident batches with per-packet arrays: a
                          // packet reaching beyond it is not read, fails the parse and
                          // raises STATUS_BOUNDS.  0: the host has checked the layout
    uint32_t ahead;       // note only: bytes of the arena that lie ahead of pkts (with limit)
    uint32_t trim;        // bytes at the end of each packet that are not payload
    uint32_t small_in_lds; // set by the launcher: there is LDS for present_small (a launch reads it
                          // while the table has seen at most SMALL_KEYS_MAX keys)
    uint64_t *record;     // note only: pinned host word that receives record_seq - 1 << 32 | slots
    uint32_t record_seq;  // claimed by the batches up to that number, or more (see flows_reserve)
    bool record_after;    // note only: and record_seq << 32 | slots once this launch, the last of its
                          // batch, has ended
    uint32_t record_blocks; // set by the launcher: the launch has that many workgroups with packets, and the
                          // last of them to be done leaves that record (0: it does not)
    ReplayMark mark; // check only: bits of the batch's windows that are still to be set (n 0: none)
    RuleIndexDev rules;
    FlowTableDev flows;
};

hipError_t launch_fill_u64(uint64_t *p, uint32_t n, uint64_t v, hipStream_t s);
hipError_t launch_flow_clear(FlowSlotMem *p, uint32_t n, hipStream_t s);
hipError_t launch_fill_u8(uint8_t *p, uint32_t n, uint8_t v, hipStream_t s);
hipError_t launch_filter_check(const FilterArgs &a, uint32_t max_blocks, hipStream_t s);
// inserts, then the reference's conditional expiry sweep
// claimed_upper: the host's upper bound on claimed slots.  Up to 4096 the
// sweep cannot fire and its launch is left out.
hipError_t launch_filter_note(const FilterArgs &a, uint32_t max_blocks, uint64_t claimed_upper, hipStream_t s);
// The sweep alone, behind a launch that has noted the batch; or what it does, for a launch of other work
// with that many workgroups of SWEEP_THREADS more (flow_sweep in filter_lane.hpp; 0: nothing to do).
struct SweepArgs {
    FlowTableDev ft;
    int64_t now;
    uint64_t *record; // or nullptr
    uint32_t seq, blocks;
};
constexpr uint32_t SWEEP_THREADS = 256;
SweepArgs flow_sweep_args(const FilterArgs &a, uint32_t max_blocks, uint64_t claimed_upper);
hipError_t launch_flow_sweep(const FilterArgs &a, uint32_t max_blocks, uint64_t claimed_upper, hipStream_t s);
// launch_peer_rank_small (kernels.hpp), advancing, and launch_filter_note on the same batch in one launch.
hipError_t launch_peer_rank_small_note(const uint32_t *peer, uint32_t n_keys, uint32_t n, uint64_t *ctr_base,
                                       uint64_t *ctr_out, uint64_t ctr_limit, uint32_t *status, const FilterArgs &note,
                                       uint32_t max_blocks, uint64_t claimed_upper, hipStream_t s);
// launch_peer_rank_counting (kernels.hpp), advancing, with launch_filter_note on the same batch in its two
// launches, where peer_rank_whole says so.
bool peer_rank_whole(uint32_t n, uint32_t n_keys);
hipError_t launch_peer_rank_counting_note(const uint32_t *peer, void *tmp, uint64_t *ctr_base, uint32_t n_keys, uint32_t n,
                                          uint64_t *ctr_out, uint64_t ctr_limit, uint32_t *status, const FilterArgs &note,
                                          uint32_t max_blocks, uint64_t claimed_upper, hipStream_t s);
hipError_t launch_flow_rehash(const FlowTableDev &from, const FlowTableDev &to, uint32_t *status,
                              uint32_t max_blocks, hipStream_t s);

} // namespace bnk
