// CPU check of the host-side rules around a launch (bnk_amd/csrc): which packets lie in the
// arena.  Prints PASS/FAIL lines; exit status is the number of failures.
#include <stdio.h>

#include <initializer_list>

#include "../../bnk_amd/csrc/kernels.hpp"

using namespace bnk;

static int failures = 0;
static void expect(bool ok, const char *what)
{
    if (!ok) {
        printf("FAIL %s\n", what);
        failures++;
    }
}

// Offset words of a device-resident batch may hold anything: [off, off + skip + len) against the
// arena, in integers that cannot wrap.
static void arena_bounds()
{
    const uint64_t top = ~0ull;
    for (uint64_t limit : std::initializer_list<uint64_t>{1ull, 15ull, 16ull, 17ull, 48ull, 4096ull, 1ull << 33, 1ull << 63, top})
        for (uint32_t skip : {0u, 16u})
            for (uint64_t len : std::initializer_list<uint64_t>{0ull, 1ull, 16ull, 1436ull, 0x7FFFFFFFull, 0xFFFFFFFFull + 16ull})
                for (uint64_t off : std::initializer_list<uint64_t>{0, 1, 16, limit - 32, limit - 17, limit - 16, limit - 1, limit,
                                                                    limit + 1, top / 2, top - 31, top - 16, top - 15, top - 1, top}) {
                    const unsigned __int128 end = (unsigned __int128)off + skip + len;
                    expect(beyond_arena(off, skip, len, limit) == (end > limit), "bytes behind an offset word against the arena");
                }
    expect(!beyond_arena(top, 16u, 100u, 0), "limit 0 checks nothing");
}

int main()
{
    arena_bounds();
    if (!failures) printf("PASS launch rules\n");
    return failures;
}
