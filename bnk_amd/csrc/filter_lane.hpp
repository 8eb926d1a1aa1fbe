// What a lane does with one packet header, for the kernels of the packet filter: the IPv4 5-tuple
// parse, the flow table's slots, and recording an outgoing packet's flow.
#pragma once

#include "filter_dev.hpp"
#include "kernels.hpp"

#ifndef BNK_DEV
#define BNK_DEV __device__ __forceinline__
#endif

namespace bnk {

BNK_DEV uint32_t ld32u(const uint8_t *p)
{
    uint32_t v;
    __builtin_memcpy(&v, p, 4);
    return v;
}

struct Parsed {
    uint32_t src, dst;
    uint32_t sport, dport;
    uint32_t proto;
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 __attribute__((aligned(1))) u32x4_unaligned;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef u32x2 __attribute__((aligned(1))) u32x2_unaligned;

// filter.go:71-106.  Bytes 0-15 come in one load and bytes 16-23 (destination
// and, without IP options, the ports) in a second when the packet has them:
// every load instruction here reads 64 different lines, so their number is
// what the kernel pays for.
// Where packet i lies in its arena, worked out only when somebody asks.
struct PacketAt {
    const uint8_t *pkts;
    const uint64_t *off;
    uint32_t stride, i;
    BNK_DEV const uint8_t *get() const { return pkts + (off ? off[i] : (uint64_t)i * stride); }
};

// `p`: the packet's first 24 bytes (as many as it has); `full`: the packet
// where it lies, looked at only for a header with options.
BNK_DEV bool parse_words(const u32x4 a, uint32_t dst_w, uint32_t l4_w, bool wide, uint32_t len, Parsed &o,
                         const PacketAt &full)
{
    const uint32_t w0 = a.x;
    if (((w0 >> 4) & 0xFu) != 4u) return false;
    const uint32_t ihl = (w0 & 0xFu) * 4u;
    if (ihl < 20u || len < ihl) return false;
    o.proto = (a.z >> 8) & 0xFFu;
    o.src = __builtin_bswap32(a.w);
    o.dst = __builtin_bswap32(dst_w);
    const uint32_t body = len - ihl;
    if (o.proto == 6u || o.proto == 17u) {
        if (body < 4u) return false;
        const uint32_t w = __builtin_bswap32(wide && ihl == 20u ? l4_w : ld32u(full.get() + ihl));
        o.sport = w >> 16;
        o.dport = w & 0xFFFFu;
        return true;
    }
    if (o.proto == 1u) {
        if (body < 1u) return false;
        o.sport = 0;
        o.dport = 0;
        return true;
    }
    return false;
}

BNK_DEV bool parse_packet(const uint8_t *p, uint32_t len, Parsed &o, const PacketAt &full)
{
    if (len < 20u) return false;
    const u32x4 a = *reinterpret_cast<const u32x4_unaligned *>(p);
    uint32_t dst_w, l4_w = 0;
    const bool wide = len >= 24u;
    if (wide) {
        const u32x2 b = *reinterpret_cast<const u32x2_unaligned *>(p + 16);
        dst_w = b.x;
        l4_w = b.y;
    } else {
        dst_w = ld32u(p + 16);
    }
    return parse_words(a, dst_w, l4_w, wide, len, o, full);
}

BNK_DEV uint32_t proto_class(uint32_t proto) { return proto == 1u ? 0u : proto == 6u ? 1u : 2u; }

// filter.go:108-117
BNK_DEV int64_t flow_ttl_ns(uint32_t proto)
{
    return proto == 6u ? 120000000000LL : 30000000000LL;
}

// Where a key word of a region goes: the first slot to look at, its bit of the presence bitmap, and
// its two of the small one (a Bloom filter).  The products are what it costs, a wide one as much as
// four other instructions: three of them here (a 64-bit finaliser and the small one's bits took nine).
// 65,536 keys spread as they did with that one, random or in sequence in any of their parts: found
// 0.165 slots on, 9.3 % of others pass the small bitmap and 0.3 % both.
struct FlowHash {
    uint32_t start, bit, small0, small1;
};
BNK_DEV FlowHash flow_hash(uint64_t word, uint32_t region)
{
    const uint64_t x = (uint64_t)((uint32_t)(word >> 32) ^ region << 27) * 0x9E3779B1u + (uint32_t)word;
    const uint32_t f = (uint32_t)x ^ (uint32_t)(x >> 32);
    const uint64_t y = (uint64_t)(f ^ f >> 15) * 0xC2B2AE3Du + x;
    const uint32_t y0 = (uint32_t)y, y1 = (uint32_t)(y >> 32);
    const uint64_t z = (uint64_t)(y0 ^ y1) * 0x85EBCA6Bu;
    const uint32_t z0 = (uint32_t)z, z1 = (uint32_t)(z >> 32);
    return FlowHash{z1 ^ z0, z1, y1 ^ z0, z1 ^ y0};
}
// The small bitmap's word and bit for small0 or small1: 24 of its bits choose one of the words, which
// are no power of two, and the lowest five the bit.
BNK_DEV uint32_t small_word(uint32_t h) { return (uint32_t)((uint64_t)(h & 0xFFFFFFu) * (SMALL_BITS / 32u << 8) >> 32); }
static_assert((SMALL_BITS / 32u << 8) < 1u << 24, "a product of 24 bits");

struct FlowSlot {
    uint64_t word;   // stored key word (never 0)
    uint32_t base;   // first slot of the region
    uint32_t start;  // probe start within the region
    uint32_t bit;    // this key's bit in the presence bitmap
    uint32_t small0, small1; // and those of the small one (small_word)
};

BNK_DEV FlowSlot flow_slot(const FlowTableDev &ft, uint32_t remote, uint32_t rport, uint32_t lport,
                           uint32_t proto)
{
    FlowSlot s;
    const uint32_t region = proto_class(proto) * 2u + (remote >> 31);
    s.word = (1ULL << 63) | ((uint64_t)(remote & 0x7FFFFFFFu) << 32) | ((uint64_t)rport << 16) | lport;
    s.base = region * ft.cap;
    const FlowHash h = flow_hash(s.word, region);
    s.start = h.start & (ft.cap - 1u);
    s.bit = h.bit & ft.present_mask;
    s.small0 = h.small0;
    s.small1 = h.small1;
    return s;
}

// One word holds a range of ports, the first below the complement of the last; a packet's port is
// brought into the same form once.  The range has it where neither half lies above the port's: 0 then.
// (One instruction for both halves, where a range of class and port in one word, first << 14 | span,
// took four.)
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
BNK_DEV uint32_t range_key(uint32_t port) { return (port | port << 16) ^ 0xFFFF0000u; }
BNK_DEV uint32_t range_miss(uint32_t e, uint32_t range_key)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, e), __builtin_bit_cast(u16x2, range_key)));
}
// The block of the ranges that interval iv has for a class.
BNK_DEV uint32_t range_block(uint32_t iv, uint32_t cls) { return iv * RANGE_CLASSES + cls; }

// filter.go:195-201 for one packet of a batch (the sweep of :202-208 follows as its own
// kernel because it depends on the entry count after every insert).
//
// A packet of a flow that the table has (nearly all of them, on a link that is
// in use) costs one 16-byte read and at most a plain store: every lane of the
// batch writes the same expiry for the key, and nothing is deleted in this
// launch, so a lane may see the old expiry or the new one.  Only a slot that
// looks empty or deleted is claimed with atomics, whose answers count; such a
// look may be out of date (the L2s of the eight XCDs are not coherent), then the
// atomic says so.  2^18 headers of 65,536 flows: 10.6 us (the slots' lines), with a
// compare-and-swap and an exchange per packet instead 29.1; behind transport headers
// in a tunnel's slots, 16,384 flows, 11.9 and 32.1.
BNK_DEV void note_flow(const FilterArgs &a, const Parsed &h)
{
    // remote = dst, remotePort = dstPort, localPort = srcPort
    const FlowSlot s = flow_slot(a.flows, h.dst, h.dport, h.sport, h.proto);
    const unsigned long long expiry = (unsigned long long)(a.now + flow_ttl_ns(h.proto));
    bool placed = false;
    for (uint32_t probe = 0; probe < a.flows.cap; probe++) {
        const uint32_t at_slot = s.base + ((s.start + probe) & (a.flows.cap - 1u));
        FlowSlotMem *slot = a.flows.slots + at_slot;
        unsigned long long *kp = reinterpret_cast<unsigned long long *>(&slot->key);
        unsigned long long *ep = reinterpret_cast<unsigned long long *>(&slot->exp);
        const ulonglong2 cur = *reinterpret_cast<const ulonglong2 *>(slot);
        if (cur.x != 0ULL && cur.x != s.word) continue; // (a key stays where it is)
        if (cur.x == s.word && (int64_t)cur.y != FLOW_TOMB) {
            if (cur.y != expiry) *ep = expiry;
            placed = true;
            break;
        }
        const unsigned long long old = cur.x ? cur.x : atomicCAS(kp, 0ULL, (unsigned long long)s.word);
        if (old == 0ULL) {
            const uint32_t pos = atomicAdd(&a.flows.counters[FLOW_CLAIMED], 1u);
            if (pos < a.flows.cap / 2u) a.flows.list[pos] = at_slot; // (flows_reserve keeps it below)
            atomicOr(&a.flows.present[s.bit >> 5], 1u << (s.bit & 31u));
            atomicOr(&a.flows.present_small[small_word(s.small0)], 1u << (s.small0 & 31u));
            atomicOr(&a.flows.present_small[small_word(s.small1)], 1u << (s.small1 & 31u));
        }
        if (old == 0ULL || old == s.word) {
            // the lane that replaces a tombstone (fresh slots start as
            // tombstones) brings the entry into the map
            const int64_t prev = (int64_t)atomicExch(ep, expiry);
            if (prev == FLOW_TOMB) atomicAdd(&a.flows.counters[FLOW_LIVE], 1u);
            placed = true;
            break;
        }
    }
    if (!placed) status_raise(a.status, STATUS_FLOWS_FULL);
}

// filter.go:189-201 for packet i of a batch.
BNK_DEV void note_packet(const FilterArgs &a, uint32_t i)
{
    const uint64_t at = a.off ? a.off[i] : (uint64_t)i * a.stride;
    const uint32_t len = a.lens ? a.lens[i] : a.len;
    if (beyond_arena(at, a.ahead, len, a.limit)) {
        status_raise(a.status, STATUS_BOUNDS);
        return;
    }
    const uint8_t *p = a.pkts + at;
    Parsed h;
    if (!parse_packet(p, len, h, PacketAt{a.pkts, a.off, a.stride, i})) return;
    note_flow(a, h);
}

// What a note launch does once, by one thread of a workgroup that has no packets: its few
// dependent reads, an atomic and a store to the host would otherwise be one wave's way to its
// first packet, and the whole launch waits for the slowest wave.
BNK_DEV void note_once(const FilterArgs &a)
{
    // What the last sweep left behind is folded in here, so that the next one can read the
    // entry count and the bound without anybody changing them meanwhile.
    uint32_t *c = a.flows.counters;
    int64_t *least = reinterpret_cast<int64_t *>(c + FLOW_MIN_EXP), *next = reinterpret_cast<int64_t *>(c + FLOW_NEXT_EXP);
    int64_t bound = *least;
    if (c[FLOW_SWEPT] != 0u) {
        bound = *next;
        if (c[FLOW_GONE]) atomicSub(&c[FLOW_LIVE], c[FLOW_GONE]);
        c[FLOW_GONE] = 0u;
        c[FLOW_SWEPT] = 0u;
    }
    *next = INT64_MAX;
    *least = a.now + FLOW_TTL_LEAST < bound ? a.now + FLOW_TTL_LEAST : bound;
    // (at least what the batches before this one claimed; the launch's own last workgroup knows better)
    if (a.record && !a.record_blocks)
        __hip_atomic_store(a.record, (uint64_t)(a.record_seq - 1u) << 32 | atomicAdd(&c[FLOW_CLAIMED], 0u),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// FilterArgs::record_blocks, by every thread of a workgroup with packets once it is through with them.
// (Claims are atomics whose answers have come back, so the workgroup that counts itself last reads
// what all of them have claimed.)
BNK_DEV void note_block_done(const FilterArgs &a)
{
    if (!a.record_blocks) return;
    __syncthreads();
    if (threadIdx.x != 0u) return;
    uint32_t *c = a.flows.counters;
    if (atomicAdd(&c[FLOW_NOTE_BLOCKS], 1u) + 1u != a.record_blocks) return;
    __hip_atomic_store(&c[FLOW_NOTE_BLOCKS], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(a.record, (uint64_t)a.record_seq << 32 | atomicAdd(&c[FLOW_CLAIMED], 0u), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// filter.go:202-207: above 4096 entries, delete those with now.After(exp); there
// is nothing to delete while no entry can have expired.  Nothing this launch
// decides by changes while it runs: what it deletes and the bound it finds over
// what it leaves go into words of their own until the next note launch.  (A
// counter of finished note blocks in their place costs 23 ns per block.)
//
// Over the list of claimed slots: 14.4 us for 65,536, a gather each, where going through the
// table they live in (200 MB, sized for batches of 2^18 packets) took 31 us behind every
// batch.  The host cannot tell that nothing has expired, so the launch is made behind every
// batch above 4096 entries; it returns at once then (2 to 5 us).  Being made, it leaves the record of
// the batch ahead of it (FilterArgs::record_after; record null: not), which a launch for it alone did.
// By workgroup `block` of SweepArgs::blocks.
BNK_DEV void flow_sweep(const SweepArgs &a, uint32_t block)
{
    const FlowTableDev &ft = a.ft;
    const int64_t now = a.now;
    if (a.record && block == 0u && threadIdx.x == 0u)
        __hip_atomic_store(a.record, (uint64_t)a.seq << 32 | ft.counters[FLOW_CLAIMED], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (ft.counters[FLOW_LIVE] <= FLOW_SWEEP_ABOVE || now <= *reinterpret_cast<const int64_t *>(ft.counters + FLOW_MIN_EXP)) return;
    if (block == 0u && threadIdx.x == 0u) ft.counters[FLOW_SWEPT] = 1u;
    const uint32_t claimed = ft.counters[FLOW_CLAIMED];
    const uint32_t total = claimed < ft.cap / 2u ? claimed : ft.cap / 2u;
    const uint32_t stride = a.blocks * SWEEP_THREADS;
    int64_t least = INT64_MAX;
    uint32_t gone = 0;
    for (uint32_t idx = block * SWEEP_THREADS + threadIdx.x; idx < total; idx += stride) {
        FlowSlotMem *slot = ft.slots + ft.list[idx];
        const int64_t e = slot->exp;
        if (e == FLOW_TOMB) continue;
        if (now > e) {
            slot->exp = FLOW_TOMB;
            gone++;
        } else if (e < least) {
            least = e;
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        gone += (uint32_t)__shfl_xor((int)gone, off, 64);
        const int64_t o = (int64_t)((uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)((uint64_t)least >> 32), off, 64) << 32 |
                                    (uint32_t)__shfl_xor((int)(uint32_t)least, off, 64));
        if (o < least) least = o;
    }
    if ((threadIdx.x & 63u) != 0u) return;
    if (gone) atomicAdd(&ft.counters[FLOW_GONE], gone);
    if (least != INT64_MAX)
        (void)__hip_atomic_fetch_min(reinterpret_cast<int64_t *>(ft.counters + FLOW_NEXT_EXP), least, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace bnk
