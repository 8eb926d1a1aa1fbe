// The host's upper bound on the slots claimed in the flow table.  Plain host code
// (tests/cpp/route_test.cpp runs it without a GPU).
#pragma once
#include <stdint.h>

#include <algorithm>

namespace bnk {

// Every batch may claim a slot per packet, and most claim next to none: the bound outgrows their
// number by a batch per call.  What brings it down again without waiting for the stream: every
// note batch has a number, its launch leaves (the number before << 32 | slots claimed so far) in a
// record in pinned memory as it starts, and at[] knows how much the batches after that number may
// have added.  A record from before the table last grew still holds: the new table starts with no
// more than the old one had.
struct FlowBound {
    uint64_t upper = 0;    // slots ever claimed in the current table, or more
    uint32_t seq = 0;      // the newest batch
    uint64_t reserved = 0; // packets of all batches
    uint64_t at[64] = {0}; // that sum as of batch (number & 63)

    void take(uint32_t n)
    {
        upper += n;
        reserved += n;
        at[++seq & 63u] = reserved;
    }
    // Whether the record is the newest batch's.  Numbers wrap; one 64 or more behind says nothing.
    bool lower(uint64_t record)
    {
        const uint32_t of = (uint32_t)(record >> 32);
        if (seq - of < 64u) upper = std::min(upper, (record & 0xFFFFFFFFu) + reserved - at[of & 63u]);
        return of == seq;
    }
};

} // namespace bnk
