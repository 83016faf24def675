// The cut of a host copy into pieces (host_copy.h), on the CPU.
#include "host_copy.h"

#include <cstdio>
#include <initializer_list>

using namespace perks;

#define CHECK(c) \
    if (!(c)) { std::printf("%s at %zu bytes\n", #c, bytes); return 1; }

int main()
{
    const size_t MiB = (size_t)1 << 20;
    for (size_t base : {8 * MiB, 12 * MiB, 16 * MiB, 24 * MiB + 7, 32 * MiB, 35 * MiB, 36 * MiB, 37 * MiB, 64 * MiB, 1024 * MiB}) {
        for (size_t bytes = base - 5; bytes <= base + 5; ++bytes) {
            const size_t cap = staging_capacity(bytes), own = staging_piece(cap, bytes);
            const size_t pieces = (bytes + own - 1) / own;
            CHECK(own <= cap && cap <= 12 * MiB + 8192);
            // a process's first copies: no more transfers than buffers
            if (bytes <= 36 * MiB) CHECK(pieces <= kStagingBuffers);
            if (bytes > 36 * MiB) CHECK(own == 4 * MiB);
            // through a set that another copy made
            for (size_t made : {8 * MiB, 30 * MiB, 36 * MiB, 512 * MiB}) {
                const size_t c = staging_capacity(made), p = staging_piece(c, bytes);
                CHECK(p > 0 && p <= c);
            }
        }
    }
    std::puts("ok");
    return 0;
}
