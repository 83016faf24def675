// Thread model of the grid barrier's per-XCD form (grid_sync.h): built and run
// by tests/test_grid_sync_xcd_model.py; exits non-zero on the first violation.
//
// G threads stand for G workgroups on given XCDs and run R barriers with the
// device code's steps on std::atomic words.  First barrier: read the counters'
// start values, count in, meet (here: one counter for all), the last arrival
// empties the counts and publishes them.  Later ones: arrive at the XCD's
// counter; its last arrival arrives at the root, waits there for the other
// XCDs and releases its own.  No thread may leave barrier r before every
// thread has arrived at it.  Launches follow one another on the same words
// with other grids, from counters close to wrapping around.
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

#include "grid_sync.h"

using perks::gs_last;
using perks::gs_reached;
using perks::kSyncXcds;

struct Words {
    std::atomic<unsigned int> count[kSyncXcds], gen[kSyncXcds], census[kSyncXcds], members[kSyncXcds], active[kSyncXcds];
    std::atomic<unsigned int> root, flat, flat_gen;
};

static void workgroup(Words& w, unsigned int G, int xcd, int rounds, std::vector<std::atomic<int>>& arrived,
                      std::atomic<int>& bad)
{
    unsigned int epoch = 0, count0 = 0, gen0 = 0, root0 = 0, members = 0, active = 0;
    for (int r = 0; r < rounds; ++r) {
        arrived[r].fetch_add(1);
        if (r == 0) {
            count0 = w.count[xcd].load();
            gen0 = w.gen[xcd].load();
            root0 = w.root.load();
            w.census[xcd].fetch_add(1);
            const unsigned int g0 = w.flat_gen.load();
            if (w.flat.fetch_add(1) == G - 1) {
                w.flat.exchange(0);
                unsigned int m[kSyncXcds], act = 0;
                for (int x = 0; x < kSyncXcds; ++x) act += (m[x] = w.census[x].exchange(0)) != 0 ? 1u : 0u;
                for (int x = 0; x < kSyncXcds; ++x)
                    if (m[x]) w.members[x] = m[x], w.active[x] = act;
                w.flat_gen.fetch_add(1);
            } else {
                while (w.flat_gen.load() == g0) std::this_thread::yield();
            }
            members = w.members[xcd].load();
            active = w.active[xcd].load();
        } else {
            ++epoch;
            if (gs_last(w.count[xcd].fetch_add(1), count0, epoch, members)) {
                w.root.fetch_add(1);
                while (!gs_reached(w.root.load(), root0, epoch * active)) std::this_thread::yield();
                w.gen[xcd].fetch_add(1);
            } else {
                while (!gs_reached(w.gen[xcd].load(), gen0, epoch)) std::this_thread::yield();
            }
        }
        if (arrived[r].load() != (int)G) bad.fetch_add(1);  // left before everyone arrived
    }
}

static int launch(Words& w, const std::vector<int>& xcd, int rounds, const char* name)
{
    std::vector<std::atomic<int>> arrived(rounds);
    for (auto& a : arrived) a = 0;
    std::atomic<int> bad{0};
    std::vector<std::thread> t;
    for (int x : xcd) t.emplace_back([&, x] { workgroup(w, (unsigned)xcd.size(), x, rounds, arrived, bad); });
    for (auto& x : t) x.join();
    for (int x = 0; x < kSyncXcds; ++x)
        if (w.census[x].load() != 0) return std::printf("%s: a count is left over\n", name), 1;
    if (bad.load()) return std::printf("%s: %d early releases\n", name, bad.load()), 1;
    return 0;
}

int main()
{
    static Words w{};
    const unsigned int start[] = {0u, 0xfffffff0u, 0x7ffffff8u};
    for (unsigned int s : start) {
        for (int x = 0; x < kSyncXcds; ++x) {
            w.count[x] = s;
            w.gen[x] = s + 3u;
            w.census[x] = 0;
        }
        w.root = s + 5u;
        w.flat = 0;
        w.flat_gen = s;
        for (int G : {2, 7, 8, 64, 96}) {
            std::vector<int> robin, one, uneven;
            for (int i = 0; i < G; ++i) {
                robin.push_back(i % 8);
                one.push_back(5);
                uneven.push_back(i == 0 ? 15 : (i % 3 == 0 ? 2 : 0));
            }
            if (launch(w, robin, 40, "round-robin") || launch(w, robin, 1, "one barrier") ||
                launch(w, one, 20, "one XCD") || launch(w, uneven, 20, "uneven"))
                return 1;
        }
    }
    std::printf("ok\n");
    return 0;
}
