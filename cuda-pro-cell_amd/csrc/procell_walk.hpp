// procell_walk.hpp -- how the relaxed estimator's walk kernel
// (procell_relaxed.hip) is laid out over a plan's initial cells.  No HIP: also
// built and checked on its own by the host compiler.
#pragma once

#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "procell_setup.hpp"

#ifdef __HIP__
#define PROCELL_WALK_HD __host__ __device__
#else
#define PROCELL_WALK_HD
#endif

namespace procell {

// What a pass of the walk computes.
enum WalkMode : int {
    kForward = 0,   // h
    kAdjoint = 1,   // gradient of <g, h>
    kJacobian = 2,  // h and its derivatives in each type's mean and sd
};

// A workgroup: one wavefront per SIMD, a quarter of a CU's LDS.  128 registers
// and four wavefronts per SIMD; five (the forward pass: six) gained nothing,
// the walks in flight then being more and the end of a launch longer.
constexpr uint32_t kWalkThreads = 256;
constexpr uint32_t kWalkTables = 384;  // entries of the log and sin/cos tables
constexpr uint32_t kGradSums = 384;    // gradient sums of a workgroup, all copies

// Bytes of a buffered root walk: without and with tangents.
PROCELL_WALK_HD constexpr uint32_t walk_entry_bytes(bool tan) { return tan ? 48u : 32u; }

// LDS of a workgroup, in bytes from its start: log and sin/cos tables | theta
// [3][T] | (adjoint) gradient sums, up to 16 copies of [3][T] | proliferating
// types u32 [T] | cursor of the root steps, walks cut, expansions u32 [4] |
// entries, per wavefront [64] (once the roots are done: the walks' expansions
// by origin lane, u32 [64], and each lane's origin, u32 [64]) | redraws'
// timers, per lane | window.  Entries and timers are read and written in
// 16-byte words, so every part starts at a multiple of 16 (3 T doubles are
// not one where T is odd); 16 bytes more at the end (`fixed`) for the gap
// behind the window's last copy.
struct WalkLds {
    uint32_t theta, sums, prolif, cursor, entries, held, window, fixed;
};

PROCELL_WALK_HD constexpr WalkLds walk_lds(uint32_t n_types, int mode)
{
    const uint32_t n = 3 * n_types, sums = mode == kAdjoint ? (n > kGradSums ? n : kGradSums) : 0u;
    WalkLds l{};
    l.theta = kWalkTables * 16;
    l.sums = l.theta + n * 8;
    l.prolif = (l.sums + sums * 8 + 15) / 16 * 16;
    l.cursor = l.prolif + (n_types * 4 + 15) / 16 * 16;
    l.entries = l.cursor + 16;
    l.held = l.entries + kWalkThreads * walk_entry_bytes(mode != kForward);
    l.window = l.held + kWalkThreads * 16;
    l.fixed = l.window + 16;
    return l;
}

// One workgroup's initial cells.
struct Segment {
    uint32_t set;
    uint32_t c0, c1;  // first and end initial cell (set-local)
    uint32_t r0, r1;  // first and last row (global)
};

// Most units of a segment (its cells, times the 64-type chunks of each): the
// kernel counts and claims them in 32 bits, four wavefronts of which may each
// claim 64 past the end.
constexpr uint64_t kMaxSegmentUnits = 1ull << 31;

// Splits the initial cells of one set into `n_seg` segments of equal cost
// (fewer where a cell costs more than that), none of more than `max_cells`.
inline void split_set(const Setup &s, const std::vector<double> &cell_cost, uint64_t n_seg, uint32_t set, uint32_t row_base,
                      uint64_t max_cells, std::vector<Segment> &out)
{
    const uint32_t n_rows = (uint32_t)s.v.size();
    double total = 0.0;
    for (uint32_t i = 0; i < n_rows; ++i)
        total += cell_cost[i] * (double)(s.start[i + 1] - s.start[i]);
    auto row_of = [&](uint64_t cell) {
        return row_base + (uint32_t)(std::upper_bound(s.start.begin(), s.start.end() - 1, cell) - s.start.begin() - 1);
    };
    uint32_t row = 0;
    double acc = 0.0;  // cost of the rows before `row`
    uint64_t c0 = 0;
    for (uint64_t v = 1; v <= n_seg; ++v) {
        uint64_t c1 = s.n_cells;
        if (v < n_seg) {
            const double want = total * ((double)v / (double)n_seg);
            for (; row < n_rows; ++row) {
                const double rc = cell_cost[row] * (double)(s.start[row + 1] - s.start[row]);
                if (acc + rc > want)
                    break;
                acc += rc;
            }
            if (row < n_rows) {
                c1 = s.start[row] + (uint64_t)std::max(0.0, ceil((want - acc) / cell_cost[row]));
                c1 = std::max(c0, std::min<uint64_t>(c1, s.start[row + 1]));
            }
        }
        while (c0 < c1) {
            const uint64_t end = std::min(c1, c0 + max_cells);
            out.push_back(Segment{set, (uint32_t)c0, (uint32_t)end, row_of(c0), row_of(end - 1)});
            c0 = end;
        }
    }
}

}  // namespace procell
