// Tunnel calls of small batches in one launch each: a wave per packet (aead_kernels.hip) that does,
// beside the framing, what the launches around it do for larger batches.
#pragma once

#include "filter_dev.hpp"
#include "kernels.hpp"
#include "wg_dev.hpp"

namespace bnk {

// At most this many packets: a thread per packet of the workgroup that ends the launch.
constexpr uint32_t WG_SMALL_MAX = 256;
// And up to this many: encapsulated in one launch all the same, decapsulated in two (WG_WAVES_PEERS peers
// at most), the second of which is one workgroup that takes the batch through the windows and says what
// has become of it.  That workgroup's time goes with the packets, and so does a wave's look through the
// peers: device-resident passes of IMIX packets with three streams at work, us against those of five
// launches, 700 packets 11.4 against 16.4, 1500 12.2, 16.6, 2000 13.8, 16.6, 2500 17.4, 16.6.
constexpr uint32_t WG_WAVES_MAX = 2048;
constexpr uint32_t WG_WAVES_PEERS = 255;
// Packets in a ring are a wave each all the same up to here (aead_runs_spread), and what the launches of
// their own would fetch over the link again, headers and results, takes 14 us in each: calls out and back,
// 1024 packets of 1400 bytes 154 -> 146.5 us, 2500 of the internet mix 156 -> 142, 4096 of 1 to 600 bytes
// 220 -> 196, 300 of 1400 73 -> 72.5.
constexpr uint32_t WG_RING_WAVES_MAX = 4096;
constexpr uint32_t WG_SMALL_RECORD = 8; // words per packet, see TunnelSmall::records
// Workgroups count themselves in groups of this many, each in a line of its own, and the groups in the first
// line: an addition to the same word whose answer is wanted takes 23 ns of everybody's time.
constexpr uint32_t WG_ARRIVE_GROUP = 64, WG_ARRIVE_LINE = 32; // (words of a line)
constexpr uint32_t WG_ARRIVE_WORDS = (1u + WG_RING_WAVES_MAX / WG_ARRIVE_GROUP) * WG_ARRIVE_LINE;
constexpr size_t WG_SMALL_PEERS = (WG_ARRIVE_WORDS + WG_RING_WAVES_MAX * WG_SMALL_RECORD) * 4u; // (a ring's, in 16 bytes more)
constexpr size_t WG_SMALL_BYTES = WG_SMALL_PEERS + WG_RING_WAVES_MAX * 4u + 16u;

struct TunnelSmall {
    uint32_t *arrived;  // [WG_ARRIVE_WORDS] workgroups that have done their packets, 0 between launches
    uint32_t *records;  // [n][WG_SMALL_RECORD] what a packet's wave leaves for the last workgroup
    uint64_t *send_ctr; // encapsulate: the peers' next counters
    uint64_t *windows;  // decapsulate: the anti-replay windows, or nullptr where they are off
    bool filter;        // NoteOutbound / CheckInbound in the same launch
};

// a: as for a wave-per-packet launch that does the framing, without counters; f: see TunnelSmall::filter.
// Batches of up to WG_RING_WAVES_MAX packets (opened: of no more peers than WG_WAVES_PEERS above WG_SMALL_MAX).
hipError_t launch_tunnel_seal_small(const AeadArgs &a, const TunnelSmall &t, const FilterArgs &f, uint32_t max_blocks,
                                    uint64_t claimed_upper, hipStream_t s);
hipError_t launch_tunnel_open_small(const AeadArgs &a, const TunnelSmall &t, const FilterArgs &f, hipStream_t s);
// The second launch of those (wg_replay.hip).
hipError_t launch_tunnel_open_rest(const AeadArgs &a, const TunnelSmall &t, const FilterArgs &f, hipStream_t s);

} // namespace bnk
