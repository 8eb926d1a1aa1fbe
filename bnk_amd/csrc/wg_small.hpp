// Tunnel calls of small batches in one launch each: a wave per packet (aead_kernels.hip) that does,
// beside the framing, what the launches around it do for larger batches.
#pragma once

#include "filter_dev.hpp"
#include "kernels.hpp"
#include "wg_dev.hpp"

namespace bnk {

// At most this many packets: a thread per packet of the workgroup that ends the launch.
constexpr uint32_t WG_SMALL_MAX = 256;
constexpr uint32_t WG_SMALL_RECORD = 8; // words per packet, see TunnelSmall::records
constexpr size_t WG_SMALL_BYTES = 64u + WG_SMALL_MAX * WG_SMALL_RECORD * 4u;

struct TunnelSmall {
    uint32_t *arrived;  // workgroups that have done their packets, 0 between launches
    uint32_t *records;  // [n][WG_SMALL_RECORD] what a packet's wave leaves for the last workgroup
    uint64_t *send_ctr; // encapsulate: the peers' next counters
    uint64_t *windows;  // decapsulate: the anti-replay windows, or nullptr where they are off
    bool filter;        // NoteOutbound / CheckInbound in the same launch
};

// a: as for a wave-per-packet launch that does the framing, without counters; f: see TunnelSmall::filter.
hipError_t launch_tunnel_seal_small(const AeadArgs &a, const TunnelSmall &t, const FilterArgs &f, uint32_t max_blocks,
                                    uint64_t claimed_upper, hipStream_t s);
hipError_t launch_tunnel_open_small(const AeadArgs &a, const TunnelSmall &t, const FilterArgs &f, hipStream_t s);

} // namespace bnk
