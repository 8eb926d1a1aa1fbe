// Which AEAD launch a batch gets: a wave per packet, a few lanes per packet or a lane per packet.
// Host code, of sizes and kinds of memory only (tests/cpp/route_test.cpp runs it without a GPU).
#pragma once
#include <math.h>

#include <algorithm>

#include "kernels.hpp"

namespace bnk {

// Which launch?  Packets in GPU memory (us per launch of n packets in a row, all of
// them resident at once; seal and open within 2 us of each other):
//   a wave per packet   4.5 + 2.7 per 1000 packets at 1420 bytes, 1.8 at 60
//   split over lanes    6.5 + 9.2 q, q = pieces per run (n = 16384 x 1420: q = 2), 3 less than
//                       with q = 1 where every block gets a lane of its own
//   a lane per packet   5 + 2.75 per ChaCha20 block of the longest packet, and 20 more
//                       for the grouping where lengths vary
// so 4096 packets x 1420 take 15 / 17 / 71 us, 16384 50 / 26 / 71, and 24000 packets of 1
// to 1420 bytes - / 35 / 97.
//
// Packets in host memory (over_link): a wave per packet reads them where they are, the
// others fetch the whole span first: about 17 us + 2.7 to 3.3 ns per packet (200 to 1420
// bytes) against a lane per packet: measured crossovers 3,000 packets of 60 bytes, 4,800 of
// 200, 16,400 of 1420.  With the common length known the rule stays just under them;
// without it the caller's threshold stands alone.
//
// True when the launch will run one wave per packet (then order[] is not used and callers need
// not build it).
inline bool aead_runs_spread(const AeadArgs &a)
{
    // (the wave-per-packet kernel does the framing of whole slots and datagrams, not behind a header)
    if (a.wg.mode != WG_FUSE_OFF && a.in_skip != 0u) return false;
    if (a.over_link) {
        if (a.lens) return a.n <= a.spread_max;
        const uint64_t by_len = 12ull * a.len + a.spread_max / 2;
        return a.n <= std::min<uint64_t>(4ull * a.spread_max, by_len);
    }
    // 2560 by default.  Pairs of launches, us alone with a wait behind each / in a row / with three streams
    // at work, a wave per packet against split, packets of 1 to 1420 bytes: 1000 25.1 / 13.8 / 7.2 against
    // 36.1 / 25.0 / 9.4, 2000 29.3 / 18.6 / 8.6 against 38.5 / 27.4 / 11.8, 2500 33.1 / 22.0 / 10.4 against
    // 41.2 / 30.0 / 11.5, 3000 34.4 / 23.5 / 11.7 against 41.7 / 30.5 / 11.8, 4096 39.3 / 28.4 / 15.3 against
    // 42.7 / 31.4 / 13.0; IMIX as these, one length of 1420 bytes crosses at 2700 with three streams.  (One
    // stream alone in view it would end at 5000.)
    const uint64_t most = 5ull * a.spread_max / 8;
    if (a.lens) return a.n <= most;
    return a.n <= std::min<uint64_t>(most, (4ull * a.len + a.spread_max) * 4ull / 10);
}

// Room per packet: what the batch's packets take up on average in an arena that just holds them,
// as far as the host can tell.  From the lengths themselves where it has them (16 bytes more, for
// a tag and for the gaps between slots); of a batch in GPU memory it knows the stride, or else
// only the arena, which may hold far more than the batch: room is then too large, and a wave gets
// fewer packets than would fit.
constexpr uint32_t SPLIT_ROOM_MAX = 1500; // beyond it one rule holds
inline uint32_t aead_room(const bnk_batch &b)
{
    if (!b.lens || b.n == 0) return 0;
    uint64_t all = b.bytes;
    if (b.mem == BNK_MEM_HOST) {
        all = 16ull * b.n;
        for (uint32_t i = 0; i < b.n; i++) all += b.lens[i];
    } else if (!b.offsets) {
        all = std::min(all, (uint64_t)b.n * b.stride);
    }
    return (uint32_t)std::min<uint64_t>(all / b.n, SPLIT_ROOM_MAX);
}

constexpr uint32_t SPLIT_MAX_PACKETS = 32; // per wave
constexpr uint32_t SPLIT_ALWAYS_ONE = 5;
constexpr uint32_t SPLIT_ONE_BLOCK_WAVES = 1024; // a wave per SIMD

// Packets per wave of the launch that splits packets over lanes, 0 where a launch of
// a lane per packet is the better one.
//
// How many: n / 2048 of them fill the chip with waves once and say how many pieces a run
// must hold; what decides the cost is then how many of a wave's 64 lanes have a run, so the
// wave takes as many more as still fit at that length (16384 packets x 1420: 10 instead of 8,
// 38 us a pair of launches instead of 46 with three streams at work, 58 on one stream either
// way).  Where the lengths vary the room per packet (aead_room) stands for
// their mean, with a margin for how much of it a wave may get: beyond 64 lanes all of a wave's
// runs get longer (24000 packets of 1 to 1420 bytes, 15 per wave instead of 12: 39 us instead
// of 47 on three streams, 70 instead of 63 on one).
//
// Where it ends: on one stream it is ahead up to where lanes fill the chip (65536 x 1420: 121
// us a pair against 145), but it does half as much work again, and with several streams at
// work the launches of a lane per packet overlap: 16384 x 1420 38 us against 50, x 600 25
// against 27, 32768 x 1420 66 against 55.  Where lengths vary the other choice has the
// grouping ahead of it as well: 40000 packets of 1 to 1420 bytes 61 us against 83, 57344 84
// against 87, 65536 97 against 89.  Short packets end it earlier, since a lane each is then
// done in no time (pairs with three streams at work, slots of a multiple of 128 bytes): 32000
// of 1 to 44 bytes 16 us against 18, 40000 19.0 against 18.5, 48000 22 against 19; 1 to 200
// bytes 40000 27 against 28, 48000 33 against 27; 1 to 400 bytes 48000 40 against 44, 57000 47
// against 46.  (Back to back without gaps they hold out longer, 1 to 200 bytes 29 against 35 at
// 57000, but the host sees the room alone.)
//
// A host batch has the chip to itself and its grouping in the call's way, so short packets do not
// end it there: calls on pinned rings, a lane per packet against split, 38000 of 1 to 100 bytes
// sealed 258 us against 234, through the tunnel 366 out and 403 in against 320 and 317, 50000 340
// against 301 and 461 and 521 against 419 and 415; 40000 of 1 to 200 bytes 345 against 334; only
// 54000 of 1 to 60 bytes are sealed in 275 against 281, with 408 and 417 against 398 and 395
// through the tunnel.
//
// Up to 10240 packets whose lengths the host does not know, five per wave: whatever mix of
// up to 1471 bytes they are, a piece is then all that a run ever holds, and the launch lasts
// as long as that (3400 packets of 1 to 1420 bytes 46 -> 32 us a pair against as many as fit on
// average, 10000 51 -> 40).
//
// A wave with a lane for every block of its packets (the kernel deals them out so whenever the
// lanes allow) is done sooner still, so where that takes no more than a wave per SIMD it gets no
// more packets than surely fit: two of any lengths up to 1984, five where twice the mean room
// does, as many as the common length allows.  Pairs, us alone / with three streams at work:
// tunnel passes of 200 IMIX packets 47.7 / 21.6 -> 42.7 / 19.3, of 900 58.6 / 21.7 -> 54.5 / 21.0, of
// 2000 of 500 bytes 61 / 22.4 against 65 / 24.2; 3500 packets of 600 bytes 30.8 / 12.0 -> 27.1 / 10.7,
// 8000 of 300 29.1 / 11.4 -> 26.2 / 10.6.  With more than one such wave per SIMD it only helps a launch
// that is alone: 4000 packets of 1 to 1420 bytes two to a wave 34.5 / 23.7 against 32.1 / 13.1 five to
// a wave, 8000 of 600 five to a wave 32.1 / 19.4 against 33.1 / 13.8.  (Not for one or two blocks
// of data: 4000 of 60 bytes 22.2 / 8.5 against 15.8 / 7.8 a lane per packet, 20000 of 124 28.4 / 12.1
// against 27.3 / 10.6.)
inline uint32_t aead_split_packets(const AeadArgs &a)
{
    // (spread_max 0 asks for a lane per packet; order[] is only built for that launch)
    if (a.spread_max == 0 || a.order || aead_runs_spread(a)) return 0;
    const uint32_t per = (a.n + 2047u) / 2048u;
    const uint32_t room = a.lens ? std::min(a.room, SPLIT_ROOM_MAX) : a.len;
    if (per > (!a.lens ? 12u : room < 256u && !a.host_batch ? 18u : 27u)) return 0;
    const uint32_t blocks = (room + 63u) / 64u, pieces = blocks / 2u + 1u;
    auto fits = [&](uint32_t k, uint32_t q) {
        if (!a.lens) return k * ((pieces + q - 1u) / q) <= 64u;
        const double mean = (double)room / (128.0 * q) + 1.0;
        return k * mean + 0.3 * mean * sqrt((double)k) <= 64.0;
    };
    uint32_t q = 1, k = per;
    // a lane per block wherever that leaves no more than a wave per SIMD
    const uint32_t one_block = a.lens ? (5u * ((room + 31u) / 32u + 1u) <= 64u ? SPLIT_ALWAYS_ONE : 2u)
                                      : std::min(64u / (blocks + 1u), SPLIT_MAX_PACKETS);
    const bool ahead_of_lanes = a.lens || 150u + 920u < 275u * (blocks + 1u);
    if (ahead_of_lanes && one_block >= 2u && a.n <= one_block * SPLIT_ONE_BLOCK_WAVES) return one_block;
    if (a.lens && per <= SPLIT_ALWAYS_ONE) return std::max(per, SPLIT_ALWAYS_ONE);
    while (q < pieces && !fits(k, q)) q++;
    while (k < SPLIT_MAX_PACKETS && fits(k + 1u, q)) k++;
    return a.lens || 150u + 920u * q < 275u * (blocks + 1u) ? k : 0u;
}

// True when the launch would run faster with order[] (a lane per packet, lengths vary).
inline bool aead_wants_order(const AeadArgs &a)
{
    return a.lens && a.n > 64 && !aead_runs_spread(a) && aead_split_packets(a) == 0;
}

// How a batch's lengths are grouped (launch_length_sort).  A block takes GROUP_CHUNK packets at a time,
// one round of them in batches of up to LEN_FUSED_SCAN_MAX_BLOCKS blocks (2^20 packets, a block per
// compute unit).  Beyond, a block takes LEN_MANY_ROUNDS: fewer blocks add to the same few words of
// hist[] and cursor[], and up to 2^22 packets the scatter launch still scans for itself, without a
// launch for the scan (2^22: 10.5 us to count and 19.8 to place; with one round and the scan launch
// 16.0, 4.7 and 20.7, with two rounds 11.8, 4.8 and 15.5, with eight and no scan launch 15.0 and 26.6).  Where
// the blocks are more than that, a launch of its own scans: every block would fetch the same few lines
// (2^22 packets, one round: 3.6 us more than the scan launch; 2^20: 1.6 less).
constexpr uint32_t GROUP_THREADS = 1024;
constexpr uint32_t GROUP_PER_THREAD = 4; // consecutive packets
constexpr uint32_t GROUP_CHUNK = GROUP_THREADS * GROUP_PER_THREAD;
constexpr uint32_t LEN_FUSED_SCAN_MAX_BLOCKS = 256;
constexpr uint32_t LEN_MANY_ROUNDS = 4;
struct LenSortPlan {
    uint32_t rounds, blocks;
    bool fused; // the scatter launch scans
};
// (for any n: the packets of a full grid are at most 2^32, so a thread's first one never wraps)
inline LenSortPlan len_sort_plan(uint32_t n)
{
    const uint32_t chunks = n / GROUP_CHUNK + (n % GROUP_CHUNK != 0u);
    const uint32_t rounds = chunks <= LEN_FUSED_SCAN_MAX_BLOCKS ? 1u : LEN_MANY_ROUNDS;
    const uint32_t blocks = (chunks + rounds - 1u) / rounds;
    return {rounds, blocks, blocks <= LEN_FUSED_SCAN_MAX_BLOCKS};
}

} // namespace bnk
