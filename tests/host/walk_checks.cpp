// walk_checks.cpp -- the walk kernel's layout (procell_walk.hpp) on the CPU.
// usage: walk_checks <check>; exit status 0 when it held.
#include <stdio.h>
#include <string.h>

#include "procell_walk.hpp"

using namespace procell;

static int g_failures = 0;

#define CHECK(c)                                                                    \
    do {                                                                            \
        if (!(c)) {                                                                 \
            fprintf(stderr, "CHECK failed at %s:%d: %s\n", __FILE__, __LINE__, #c); \
            ++g_failures;                                                           \
        }                                                                           \
    } while (0)

// Segments cover the cells in order, each with the rows of its first and last
// cell and no more units than the kernel counts, also where a set of billions
// of shallow cells gets a single segment's share of the cost.
static void check_segments()
{
    const uint64_t most = 0xFFFFFFFFull;
    for (uint64_t cells : {1ull, 1000ull, 1ull << 30, (1ull << 31) + 5, 3000000000ull, (unsigned long long)most})
        for (uint32_t n_prolif : {1u, 64u, 65u, 256u})
            for (uint64_t n_seg : {1ull, 3ull, 1024ull}) {
                Setup s;
                s.v = {8.0, 4.0, 2.0};
                s.start = {0, cells / 3, cells - cells / 7, cells};
                s.n_cells = cells;
                std::vector<Segment> segs;
                const uint64_t chunks = (n_prolif + 63) / 64;
                split_set(s, {5.0, 2.0, 1.0}, n_seg, 4, 100, kMaxSegmentUnits / chunks, segs);
                uint64_t at = 0;
                for (const Segment &p : segs) {
                    CHECK(p.set == 4 && p.c0 == at && p.c1 > p.c0);
                    // the 32-bit cursor also takes a claim of each wavefront past the end
                    CHECK((uint64_t)(p.c1 - p.c0) * chunks + 4 * 64 <= 0xFFFFFFFFull);
                    CHECK(s.start[p.r0 - 100] <= p.c0 && p.c0 < s.start[p.r0 - 99]);
                    CHECK(s.start[p.r1 - 100] < p.c1 && p.c1 <= s.start[p.r1 - 99]);
                    at = p.c1;
                }
                CHECK(at == cells);
            }
}

// Every part of a workgroup's LDS starts at a multiple of 16 bytes and holds
// what it is for, for any number of types; entries and timers, read and
// written in 16-byte words, stay on them for every lane.
static void check_lds()
{
    for (int mode : {kForward, kAdjoint, kJacobian})
        for (uint32_t t = 1; t <= 256; ++t) {
            const WalkLds l = walk_lds(t, mode);
            const uint32_t sums = mode == kAdjoint ? std::max(kGradSums, 3 * t) : 0;
            for (uint32_t at : {l.theta, l.prolif, l.cursor, l.entries, l.held, l.window, walk_entry_bytes(mode != kForward)})
                CHECK(at % 16 == 0);
            CHECK(l.theta >= kWalkTables * 16 && l.sums >= l.theta + 3 * t * 8 && l.sums % 8 == 0);
            CHECK(l.prolif >= l.sums + sums * 8 && l.cursor >= l.prolif + 4 * t && l.entries >= l.cursor + 16);
            CHECK(l.held >= l.entries + kWalkThreads * walk_entry_bytes(mode != kForward));
            CHECK(l.window >= l.held + kWalkThreads * 16 && l.fixed >= l.window + 8 && l.fixed <= 40960);
        }
}

int main(int argc, char **argv)
{
    const struct {
        const char *name;
        void (*f)();
    } checks[] = {{"segments", check_segments}, {"lds", check_lds}};
    for (const auto &c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.f();
            printf("%s: %d failed\n", c.name, g_failures);
            return g_failures ? 1 : 0;
        }
    fprintf(stderr, "usage: walk_checks <check>\n");
    return 2;
}
