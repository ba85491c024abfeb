// procell_api.hip -- host side of libprocell: validation, problem set-up,
// device buffers, launches and the merge of tallies into the output
// histogram.  Replaces the host halves of create_cells_population
// (src/simulation/cells_population.cu:18-54) and proliferate
// (src/simulation/proliferation.cu:26-215), and the bin-set construction of
// load_fluorescences (src/io/parser.cu:68-154).
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <new>
#include <vector>

#include "procell_internal.hpp"

namespace procell {

}  // namespace procell

using namespace procell;

// ---------------------------------------------------------------------------
// Plan: device buffers for one problem (or a batch of parameter sets), reused
// across runs.
// ---------------------------------------------------------------------------
constexpr uint32_t kSeedSlots = 4;  // pinned host staging slots for batch seeds
// Segments per resident workgroup unless tuned: each segment ends with its
// wavefronts draining their last trees, and more of them balance the CUs
// better, so the more work there is per resident workgroup, the more segments
// (see segments_per_workgroup).  A batch of many small sets balances better
// with finer segments.
constexpr uint32_t kSegmentsPerWorkgroup = 2;  // 64-bit kernel
constexpr uint32_t kBatchSegmentsPerWorkgroup = 8;
// most lane-stack levels a batch keeps in LDS (a 256-lane workgroup: 2 KB per level)
constexpr uint32_t kLdsStackLevels = 11;

struct procell_plan {
    int device = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    bool timing = false;
    std::vector<int32_t> track_ratio;  // per set
    std::vector<Setup> setups;         // per set
    std::vector<size_t> tally_base, tally_len;  // per set, in tally entries
    LaunchShape shape{};
    int per_cu = 0;  // resident workgroups per CU that the layout is for
    RunArgs args{};
    void *d_block = nullptr;  // one allocation holding every table
    bool own_block = true;    // false: d_block is the static scratch array
    size_t tally_total = 0;
    size_t zero_words = 0;    // counters and tally, cleared per run
    uint64_t *d_seeds = nullptr;       // [n_sets] seeds of the current batch run (in d_block)
    uint64_t *h_seeds = nullptr;       // pinned [kSeedSlots][n_sets]
    hipEvent_t seed_ev[kSeedSlots] = {};
    hipGraph_t graph = nullptr;        // batch runs: clearing and simulation kernels
    hipGraphExec_t graph_exec = nullptr;
    std::vector<hipEvent_t> kev;   // PROCELL_FLAG_TIMING: start/stop of each run's kernels (ring)
    uint64_t runs = 0;             // runs since the last kernel-time read
    size_t last_slot = 0;          // event slot of the last timed run
    bool timed = false;            // a run has recorded its events
    uint64_t batch_runs = 0;
    bool ran = false;
    // results: bins of the tally entries, made at a set's first result, and
    // pinned memory for downloads, made at the plan's second (a plan used once
    // would pay for it more than it gains); `stage` holds the sets
    // [stage_set, stage_end) of run `stage_run`
    std::mutex result_mu;
    std::vector<std::vector<int32_t>> bin_of;
    uint64_t results = 0, run_id = 0, stage_run = 0;
    uint32_t stage_set = 0, stage_end = 0;
    uint64_t next_run = 0;             // a download of set next_set of this run brings next_n sets
    uint32_t next_set = 0, next_n = 1;
    void *stage = nullptr;
    size_t stage_bytes = 0;
    // copies of the inputs (the autotuner re-creates the layout from them)
    std::vector<procell_params> params;
    std::vector<std::vector<procell_row>> rows;
    std::vector<std::vector<procell_type>> types;
};

constexpr uint32_t kTimedRuns = 256;

// Device memory of procell_simulate_noalloc, one copy per GPU (see
// scratch_address below for how host code reaches it).
constexpr size_t kScratchBytes = PROCELL_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

thread_local hipError_t g_last_hip = hipSuccess;

#define HIP_TRY(expr)                        \
    do {                                     \
        hipError_t e_ = (expr);              \
        if (e_ != hipSuccess) {              \
            g_last_hip = e_;                 \
            return PROCELL_E_HIP;            \
        }                                    \
    } while (0)

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

int check_device(int device, int *n_cu, size_t *lds_per_cu = nullptr, size_t *lds_per_block = nullptr)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0 || device < 0 || device >= count)
        return PROCELL_E_NO_DEVICE;
    HIP_TRY(hipSetDevice(device));
    hipDeviceProp_t prop;
    HIP_TRY(hipGetDeviceProperties(&prop, device));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return PROCELL_E_NO_DEVICE;
    *n_cu = prop.multiProcessorCount;
    if (lds_per_cu)
        *lds_per_cu = prop.maxSharedMemoryPerMultiProcessor ? prop.maxSharedMemoryPerMultiProcessor : 65536;
    if (lds_per_block)
        *lds_per_block = prop.sharedMemPerBlock ? prop.sharedMemPerBlock : 65536;
    return PROCELL_OK;
}

void destroy_plan(procell_plan *pl)
{
    if (!pl)
        return;
    (void)hipSetDevice(pl->device);
    if (pl->graph_exec)
        (void)hipGraphExecDestroy(pl->graph_exec);
    if (pl->graph)
        (void)hipGraphDestroy(pl->graph);
    for (hipEvent_t &e : pl->kev)
        if (e)
            (void)hipEventDestroy(e);
    for (hipEvent_t &e : pl->seed_ev)
        if (e)
            (void)hipEventDestroy(e);
    if (pl->h_seeds)
        (void)hipHostFree(pl->h_seeds);
    if (pl->stage)
        (void)hipHostFree(pl->stage);
    if (pl->d_block && pl->own_block)
        (void)hipFree(pl->d_block);
    if (pl->own_stream && pl->stream)
        (void)hipStreamDestroy(pl->stream);
    delete pl;
}

// Whether the filtered kernel's error bounds cover these sets: times, means
// and standard deviations of magnitudes that single precision holds with
// their products and the differences of their 64-bit values (t_max 0 or
// infinite, or beyond these ranges, goes to the 64-bit kernel).  Whether it
// is the faster kernel is filter_pays' matter.
bool filter_covers(const std::vector<Setup> &sets)
{
    for (const Setup &s : sets) {
        if (!(s.t_max >= 1e-9 && s.t_max <= 1e12))
            return false;
        for (size_t j = 0; j < s.type_mean.size(); ++j)
            if (fabs(s.type_mean[j]) > 1e12 || fabs(s.type_sd[j]) > 1e12)
                return false;
    }
    return true;
}

// Segments per resident workgroup of a single set, from the expected
// lane-steps per resident workgroup.  Filtered kernel, 3 workgroups of 512 per
// CU, the five-type histogram at 1e6 cells (4.6e3 lane-steps), 3e6 (1.4e4),
// 1e7 (4.6e4) and 1e8 (4.6e5), microseconds per run with 1 / 2 / 3 / 4
// segments: 36 / 38 / 45 / 51, 66 / 59 / 66 / 74, 172 / 139 / 141 / 147,
// 1484 / 1185 / 1094 / 1096.
uint32_t segments_per_workgroup(double lane_steps, bool filter)
{
    if (!filter)
        return kSegmentsPerWorkgroup;
    return lane_steps < 8e3 ? 1 : lane_steps < 1.5e5 ? 2 : 3;
}

// A plan over n_sets parameter sets (1: a plain run).  Rows, cells, type
// entries, tally entries and segments of the sets are concatenated in set
// order; the device code finds a set's values through its SetInfo.
// With `arena` (device memory of `arena_bytes`, already on ps[0].device) the
// plan's device block is carved from it instead of allocated, no stream or
// event is created (the plan runs on ps[0].stream, NULL: the default stream)
// and timing is off.  Without `may_filter` the plan keeps the 64-bit kernel.
int create_plan(const procell_params *ps, uint32_t n_sets, procell_plan **out, void *arena = nullptr,
                size_t arena_bytes = 0, bool may_filter = true)
{
    if (!ps || !out || n_sets == 0)
        return PROCELL_E_INVALID;
    *out = nullptr;
    const procell_tuning &tu = ps[0].tuning;
    if (tu.block_size && (tu.block_size % 64 || tu.block_size > 256))
        return PROCELL_E_INVALID;
    for (uint32_t i = 1; i < n_sets; ++i)
        if (ps[i].device != ps[0].device)
            return PROCELL_E_INVALID;
    procell_plan *pl = new (std::nothrow) procell_plan();
    if (!pl)
        return PROCELL_E_OUT_OF_MEMORY;
    pl->setups.resize(n_sets);
    pl->track_ratio.resize(n_sets);
    for (uint32_t i = 0; i < n_sets; ++i) {
        const int rc = build_setup(&ps[i], pl->setups[i], true);
        if (rc != PROCELL_OK) {
            delete pl;
            return rc;
        }
        pl->track_ratio[i] = ps[i].track_ratio;
    }
    pl->params.assign(ps, ps + n_sets);
    pl->rows.resize(n_sets);
    pl->types.resize(n_sets);
    for (uint32_t i = 0; i < n_sets; ++i) {
        pl->rows[i].assign(ps[i].rows, ps[i].rows + ps[i].n_rows);
        pl->types[i].assign(ps[i].types, ps[i].types + ps[i].n_types);
        pl->params[i].rows = pl->rows[i].data();
        pl->params[i].types = pl->types[i].data();
    }
    int n_cu = 0;
    size_t lds_per_cu = 0, lds_per_block = 0;
    {
        const int rc = check_device(ps[0].device, &n_cu, &lds_per_cu, &lds_per_block);
        if (rc != PROCELL_OK) {
            delete pl;
            return rc;
        }
    }
    pl->device = ps[0].device;
    pl->timing = !arena && (tu.flags & PROCELL_FLAG_TIMING) != 0;
    if (arena && n_sets != 1) {
        delete pl;
        return PROCELL_E_INVALID;
    }
    auto fail = [&](int code) {
        destroy_plan(pl);
        return code;
    };

    // ---- concatenation of the sets ----
    std::vector<SetInfo> info(n_sets);
    uint64_t n_cells = 0, n_rows64 = 0, n_types_tot = 0;
    uint32_t T = 1, kdim = 1;
    pl->tally_base.resize(n_sets);
    pl->tally_len.resize(n_sets);
    for (uint32_t i = 0; i < n_sets; ++i) {
        const Setup &s = pl->setups[i];
        const uint32_t Ti = s.n_types ? s.n_types : 1;
        const uint32_t ki = (uint32_t)s.kmax + 1;
        SetInfo &si = info[i];
        memset(&si, 0, sizeof si);
        si.t_max = s.t_max;
        si.cell_base = n_cells;
        si.tally_base = pl->tally_total;
        si.kdim = ki;
        si.n_types = Ti;
        si.type_base = (uint32_t)n_types_tot;
        si.row_base = (uint32_t)n_rows64;
        pl->tally_base[i] = pl->tally_total;
        pl->tally_len[i] = (size_t)s.v.size() * ki * Ti;
        pl->tally_total += pl->tally_len[i];
        n_cells += s.n_cells;
        n_rows64 += s.v.size();
        n_types_tot += Ti;
        T = std::max(T, Ti);
        kdim = std::max(kdim, ki);
    }
    if (n_cells > kMaxCells || n_rows64 > kMaxRows)
        return fail(PROCELL_E_TOO_MANY_CELLS);
    const uint32_t n_rows = (uint32_t)n_rows64;

    // ---- launch shape: block size, resident workgroups, LDS split ----
    LaunchShape &ls = pl->shape;
    RunArgs &a = pl->args;
    a.stack_levels = kdim > 3 ? kdim - 1 : 2;  // levels 1 .. kmax, at least 2 (idle lanes store at level 2)
    // A batch whose deepest set needs more than kLdsStackLevels stack levels
    // keeps the lanes' stacks in device memory: in LDS they would be sized for
    // that set and leave no room for the tally window at more than two
    // workgroups per CU (512-set batch of 128-1024 bins, up to 17 generations:
    // 2.65 ms per run at 2 workgroups per CU, 5.9 ms at 3 or 4 without a window).
    const bool gstack = n_sets > 1 && a.stack_levels > kLdsStackLevels;
    const uint32_t lds_levels = gstack ? 0u : a.stack_levels;
    const bool filter = may_filter && filter_covers(pl->setups) && filter_pays(pl->setups);
    // row tables (8 bytes per row) go to LDS when they are small and do not
    // cost a resident workgroup (the root steps read them when a wavefront's
    // rows advance, so from device memory they cost little).  The filtered
    // kernel's LDS is short of window rows, not of bandwidth: 8 KB of row
    // tables left its three workgroups of 512 per CU no window on the
    // 1024-bin histogram (0.80 ms per run of 1e7 cells; without them 0.143).
    uint32_t lds_rows = (size_t)(2 * n_rows + 1) * 4 <= (filter ? 2048u : 16384u) ? n_rows : 0u;
    int bs = tu.block_size ? (int)tu.block_size : filter ? (int)kFilterThreads : 256;
    int occ = 0;
    for (;;) {
        const size_t base = sim_lds_bytes(0, kdim, T, lds_levels, (uint32_t)bs, lds_rows, filter);
        int occ_v = 0;
        if (sim_occupancy(bs, base, lds_rows != 0, kdim, gstack, filter, &occ_v) != hipSuccess)
            return fail(PROCELL_E_HIP);
        if (occ_v >= 1) {
            occ = occ_v;
            break;
        }
        if (bs == 64)
            return fail(PROCELL_E_DEPTH);
        bs -= 64;  // deep trees: a smaller workgroup keeps the stack within LDS
    }
    // by default at most 16 resident wavefronts per CU for the 64-bit kernel (4
    // per SIMD, its register budget) and 24 for the filtered one (6 per SIMD):
    // with fewer vector instructions per step its wavefronts wait more on each
    // other's latencies.  1e8-cell histogram: 16 wavefronts per CU in four
    // workgroups of 256 1.236 ms per run, 20 1.248, 24 1.092, and 24 in three
    // workgroups of 512 1.099 (fewer set-ups and window flushes on smaller
    // runs); workgroups of 384 put 8 wavefronts on two of a CU's SIMDs and 4 on
    // the others (1e7 cells: 0.187 against 0.143 ms).
    const int want = tu.blocks_per_cu ? (int)tu.blocks_per_cu : std::max(1, (filter ? 24 : 16) * 64 / bs);
    if (lds_rows && occ < want) {
        int occ_g = 0;
        if (sim_occupancy(bs, sim_lds_bytes(0, kdim, T, lds_levels, (uint32_t)bs, 0, filter), false, kdim, gstack, filter, &occ_g) !=
            hipSuccess)
            return fail(PROCELL_E_HIP);
        if (occ_g > occ) {
            lds_rows = 0;
            occ = occ_g;
        }
    }
    a.rows_in_lds = lds_rows ? 1u : 0u;
    occ = std::min<int>(occ, want);
    ls.block_size = bs;

    // the sets in the order their cells are simulated: the filtered kernel's
    // rows by decreasing cost, so that the runs end with short trees
    std::vector<Setup> ordered(filter ? n_sets : 0);
    std::vector<std::vector<uint32_t>> file_row(filter ? n_sets : 0);
    for (uint32_t i = 0; i < n_sets && filter; ++i)
        ordered[i] = order_rows(pl->setups[i], file_row[i]);
    const std::vector<Setup> &lay = filter ? ordered : pl->setups;
    std::vector<double> cost(n_sets);  // expected work of each set
    double all_cost = 0.0;
    for (uint32_t i = 0; i < n_sets; ++i) {
        cost[i] = set_cost(lay[i]);
        all_cost += cost[i];
    }

    // u32 window counters must not overflow: bound the leaves any window can
    // see.  leaves[]: those of the rows before each row, one sum per set (a row
    // counts for 1e10 at most, which is over the limit by itself and keeps the
    // differences of the sums exact enough)
    std::vector<double> leaves;
    for (uint32_t i = 0; i < n_sets; ++i) {
        const Setup &s = lay[i];
        double sum = 0.0;
        for (size_t r = 0; r < s.v.size(); ++r) {
            leaves.push_back(sum);
            sum += std::min(1e10, (double)(s.start[r + 1] - s.start[r]) * ldexp(1.0, (int)(s.row_info[r] & 0xFFu)));
        }
        leaves.push_back(sum);
    }
    // Segment sizes: a single set's decrease geometrically in launch order
    // (rounds of `resident` segments, each round's segments a factor q
    // smaller, the last ones 1/8 or less of the first), so the last workgroups
    // dispatched are short and the CUs finish together; a batch's sets are
    // split evenly and all segments are launched largest first.
    // Within a round, segment k goes to CU slot (k mod resident) / n_cu: the
    // dispatcher fills every CU's first slot, then its second, and the
    // instruction arbiter favours the older workgroups of a CU (measured with
    // three per CU: 1175, 1570 and 2050 cycles per division step for the
    // oldest, middle and youngest), so a slot's segments are sized by its
    // issue rate, 1.32 per slot of age (1e7-cell histogram workload: 0.2617
    // -> 0.2587 ms and 0.2644 -> 0.2603 ms on two boxes).  The filtered
    // kernel's wavefronts compete less for the vector unit: 1.1 per slot, and
    // its last segments are 1/20 of the first (1.0, 1.1, 1.2 and 1.32 per slot
    // at 1e7 cells: 0.146, 0.142, 0.145 and 0.184 ms).
    struct Seg {
        double cost;
        uint32_t set;
        uint64_t b0, b1;  // cells, relative to the set
        uint32_t row;
    };
    // The segments and the window for `occ` resident workgroups per CU.
    struct Layout {
        int occ = 0;
        std::vector<uint64_t> begin, end;  // cells, over all sets
        std::vector<uint32_t> row, set;
        uint32_t win_rows = 0;
        size_t lds_bytes = 0;
        double load = 0.0;                 // expected lane-steps per resident workgroup
        double outside = 0.0;              // share of the expected work in rows beyond its segment's window
    };
    auto lay_out = [&](int occ, Layout &L) -> int {
        L = Layout{};
        L.occ = occ;
        // ---- segments: one per workgroup, each within one set ----
        // `per_wg` segments per resident workgroup in total, of about equal
        // expected work: workgroups beyond the resident ones start as others
        // finish, so the dispatcher balances the segments over the CUs.  In a
        // batch each set gets segments in proportion to its expected work (at
        // least one).
        const uint32_t resident = (uint32_t)((int64_t)n_cu * occ);
        const uint32_t per_wg = tu.segments   ? std::min<uint32_t>(tu.segments, 64)
                                : n_sets == 1 ? segments_per_workgroup(cost[0] / resident, filter)
                                              : kBatchSegmentsPerWorkgroup;
        std::vector<uint32_t> g_set(n_sets, 1);
        if (n_sets == 1) {
            g_set[0] = (uint32_t)std::min<uint64_t>((uint64_t)resident * per_wg,
                                                    std::max<uint64_t>(1, (lay[0].n_cells + 63) / 64));
        } else {
            const double target = (double)per_wg * (double)resident;
            for (uint32_t i = 0; i < n_sets; ++i)
                g_set[i] = all_cost > 0.0 ? (uint32_t)std::max(1.0, std::floor(cost[i] / all_cost * target + 0.5)) : 1u;
        }
        std::vector<Seg> segs;
        for (uint32_t i = 0; i < n_sets; ++i) {
            const Setup &s = lay[i];
            const uint32_t gi = g_set[i];
            std::vector<double> wseg(gi, 1.0);
            if (n_sets == 1 && per_wg > 1 && gi == resident * per_wg) {
                const double q = pow(filter ? 0.05 : 0.125, 1.0 / (double)(per_wg - 1));
                for (uint32_t k = 0; k < gi; ++k) {
                    const uint32_t slot = (k % resident) / (uint32_t)n_cu;  // 0: oldest on its CU
                    wseg[k] = pow(q, (double)(k / resident)) * pow(filter ? 1.1 : 1.32, (double)(occ - 1 - (int)slot));
                }
            }
            std::vector<double> cum(gi);
            double acc = 0.0, tot = 0.0;
            for (double x : wseg)
                tot += x;
            for (uint32_t k = 0; k < gi; ++k) {
                acc += wseg[k];
                cum[k] = k + 1 == gi ? 1.0 : acc / tot;
            }
            std::vector<uint64_t> b;
            std::vector<uint32_t> r;
            split_segments(s, cum, b, r);
            for (uint32_t k = 0; k < gi; ++k)
                segs.push_back(Seg{cost[i] * wseg[k] / tot, i, b[k], b[k + 1], r[k]});
        }
        std::stable_sort(segs.begin(), segs.end(), [](const Seg &x, const Seg &y) { return x.cost > y.cost; });
        for (const Seg &sg : segs) {
            const SetInfo &si = info[sg.set];
            L.begin.push_back(si.cell_base + sg.b0);
            L.end.push_back(si.cell_base + sg.b1);
            L.row.push_back(si.row_base + sg.row);
            L.set.push_back(sg.set);
        }
        const uint32_t g = (uint32_t)L.row.size();
        L.load = all_cost / resident;
        // no more window rows than a segment spans
        const size_t base = sim_lds_bytes(0, kdim, T, lds_levels, (uint32_t)bs, lds_rows, filter);
        const size_t budget = std::min(lds_per_cu / (size_t)occ, lds_per_block);
        const size_t row_bytes = (size_t)kdim * T * 4;
        L.win_rows = budget > base + 16 ? (uint32_t)((budget - base - 16) / row_bytes) : 0;
        uint32_t span = 1;
        std::vector<uint32_t> last(g, 0);  // rows, relative to the set
        for (uint32_t k = 0; k < g; ++k) {
            const Setup &s = lay[L.set[k]];
            const SetInfo &si = info[L.set[k]];
            if (!s.n_cells)
                continue;
            const uint64_t first = L.begin[k] - si.cell_base;
            const uint64_t end = L.end[k] - si.cell_base;
            const uint64_t lc = end > first ? end - 1 : first;
            const uint64_t lcc = lc < s.n_cells ? lc : s.n_cells - 1;
            last[k] = (uint32_t)(std::upper_bound(s.start.begin(), s.start.end() - 1, lcc) - s.start.begin()) - 1;
            span = std::max(span, last[k] - (L.row[k] - si.row_base) + 1);
        }
        L.win_rows = std::min(L.win_rows, span);
        for (uint32_t k = 0; k < g && L.win_rows; ++k) {
            const uint32_t nr = (uint32_t)lay[L.set[k]].v.size();
            const uint32_t r0 = L.row[k] - info[L.set[k]].row_base;
            const double *before = &leaves[info[L.set[k]].row_base + L.set[k]];
            if (before[std::min<uint32_t>(nr, r0 + L.win_rows)] - before[std::min(nr, r0)] >= 4.0e9)
                L.win_rows = 0;
        }
        // the window must not cost a resident workgroup (LDS allocation granularity)
        for (;;) {
            L.lds_bytes = sim_lds_bytes(L.win_rows, kdim, T, lds_levels, (uint32_t)bs, lds_rows, filter);
            int occ_w = 0;
            if (sim_occupancy(bs, L.lds_bytes, lds_rows != 0, kdim, gstack, filter, &occ_w) != hipSuccess)
                return PROCELL_E_HIP;
            // keep a margin for the per-workgroup LDS allocation granularity
            const bool fits = (size_t)occ * align_up(L.lds_bytes, 2048) <= lds_per_cu;
            if ((occ_w >= occ && fits) || L.win_rows == 0)
                break;
            L.win_rows -= std::max(1u, L.win_rows / 8);
        }
        for (uint32_t k = 0; k < g && L.win_rows < span && all_cost > 0.0; ++k) {
            const Setup &s = lay[L.set[k]];
            const SetInfo &si = info[L.set[k]];
            for (uint32_t r = L.row[k] - si.row_base + L.win_rows; r <= last[k] && r < (uint32_t)s.v.size(); ++r) {
                const uint64_t b = std::max(s.start[r], L.begin[k] - si.cell_base), e = std::min(s.start[r + 1], L.end[k] - si.cell_base);
                L.outside += e > b ? s.cap_cost[s.row_info[r] & 0xFFu] * (double)(e - b) / all_cost : 0.0;
            }
        }
        return PROCELL_OK;
    };
    // Tallies of rows beyond the window are device atomics, which cost up to
    // several times the run's other work, the more of it there is.  A workgroup
    // less per CU leaves the others more LDS; it costs some 12 % of a run, two
    // some 30 %, and a wider window takes longer to clear and flush.  5 types,
    // 14 generations, microseconds per run with 3 / 2 / 1 workgroups per CU
    // (64-bit kernel): 6000 rows and 1e7 cells 1188 / 187 / 197 (306), 1e5 rows
    // 816 / 401 / 303 (756), with 1e6 cells 120 / 71 / 89 (120); 2 types: 25,000
    // rows and 1e7 cells 734 / 290 / 299 (500), with 1e5 29 / 32 / 39 (39); 2
    // types, 11 generations, 1e5 rows and 1e7 cells (3 % outside) 264 / 277 /
    // 279 (689).  Runs below 2000 lane-steps per workgroup are mostly their
    // start and end.
    Layout L;
    if (const int rc = lay_out(occ, L); rc != PROCELL_OK)
        return fail(rc);
    if (filter && !tu.blocks_per_cu && L.outside > 0.02 && L.load >= 2000.0) {
        auto price = [&](const Layout &l) {
            const double d = occ - l.occ;
            return (1.0 + 1.2 * log10(l.load / 600.0) * l.outside) * (1.0 + 0.12 * d + 0.03 * d * (d - 1.0)) +
                   (l.occ > 1 ? 0.3 : 0.7) * (double)l.win_rows * kdim * T / l.load;
        };
        for (int o = occ - 1; o >= 1; --o) {
            Layout less;
            if (const int rc = lay_out(o, less); rc != PROCELL_OK)
                return fail(rc);
            if (price(less) < price(L))
                L = std::move(less);
        }
    }
    const uint32_t g = (uint32_t)L.row.size();
    const uint32_t win_rows = L.win_rows;
    ls.lds_bytes = L.lds_bytes;
    const std::vector<uint64_t> &seg_begin = L.begin, &seg_end = L.end;
    const std::vector<uint32_t> &seg_row = L.row, &seg_set = L.set;
    ls.blocks = (int)g;
    pl->per_cu = L.occ;
    a.win_rows = win_rows;
    a.idle_limit = tu.idle_lanes ? std::min<uint32_t>(tu.idle_lanes, 63) : 12;

    // ---- one device allocation: counters | tally | tables ----
    size_t off = 0;
    const size_t o_cnt = off; off += (size_t)n_sets * kCounterCopies * kNumCounters * 8;
    const size_t o_tally = off; off += pl->tally_total * 8;
    pl->zero_words = off / 8;
    off = align_up(off, 256);
    const size_t o_rs = off; off = align_up(off + (size_t)(n_rows + 1) * 4, 256);
    const size_t o_ri = off; off = align_up(off + (size_t)(n_rows + 1) * 4, 256);
    const size_t o_rc = off; off = align_up(off + (filter ? (size_t)n_rows * 4 : 0), 256);
    const size_t o_cum = off; off = align_up(off + (size_t)n_types_tot * 8, 256);
    const size_t o_mean = off; off = align_up(off + (size_t)n_types_tot * 8, 256);
    const size_t o_sd = off; off = align_up(off + (size_t)n_types_tot * 8, 256);
    const size_t o_tf = off; off = align_up(off + (size_t)n_types_tot * 4, 256);
    const size_t o_sb = off; off = align_up(off + (size_t)g * 8, 256);
    const size_t o_se = off; off = align_up(off + (size_t)g * 8, 256);
    const size_t o_sr = off; off = align_up(off + (size_t)g * 4, 256);
    const size_t o_ss = off; off = align_up(off + (size_t)g * 4, 256);
    const size_t o_info = off; off = align_up(off + (size_t)n_sets * sizeof(SetInfo), 256);
    const size_t o_seed = off; off = align_up(off + (size_t)n_sets * 8, 256);
    const size_t o_gs = off; off = align_up(off + (gstack ? (size_t)g * sim_stack_bytes(a.stack_levels, (uint32_t)bs, filter) : 0), 256);
    if (arena) {
        if (off > arena_bytes) {
            // the filtered kernel's tables take 4 bytes per row more: what only
            // fits without them runs on the 64-bit kernel
            destroy_plan(pl);
            return filter ? create_plan(ps, n_sets, out, arena, arena_bytes, false) : PROCELL_E_SCRATCH;
        }
        pl->stream = (hipStream_t)ps[0].stream;
        pl->d_block = arena;
        pl->own_block = false;
    } else {
        if (ps[0].stream) {
            pl->stream = (hipStream_t)ps[0].stream;
        } else {
            if (hipStreamCreateWithFlags(&pl->stream, hipStreamNonBlocking) != hipSuccess)
                return fail(PROCELL_E_HIP);
            pl->own_stream = true;
        }
        if (hipMalloc(&pl->d_block, off) != hipSuccess)
            return fail(PROCELL_E_OUT_OF_MEMORY);
    }
    char *dbase = (char *)pl->d_block;
    a.n_sets = n_sets;
    a.n_cells = n_cells;
    a.n_rows = n_rows;
    a.n_types = T;
    a.kdim = kdim;
    a.counters = (unsigned long long *)(dbase + o_cnt);
    a.tally = (unsigned long long *)(dbase + o_tally);
    a.filter = filter ? 1u : 0u;
    a.gstack = gstack ? dbase + o_gs : nullptr;

    a.row_start = (const uint32_t *)(dbase + o_rs);
    a.row_info = (const uint32_t *)(dbase + o_ri);
    a.row_cell = (const uint32_t *)(dbase + o_rc);
    a.type_cum = (const double *)(dbase + o_cum);
    a.type_mean = (const double *)(dbase + o_mean);
    a.type_sd = (const double *)(dbase + o_sd);
    a.type_file = (const uint32_t *)(dbase + o_tf);
    a.seg_begin = (const uint64_t *)(dbase + o_sb);
    a.seg_end = (const uint64_t *)(dbase + o_se);
    a.seg_row = (const uint32_t *)(dbase + o_sr);
    a.seg_set = (const uint32_t *)(dbase + o_ss);
    a.sets = (const SetInfo *)(dbase + o_info);
    a.set_seed = (const uint64_t *)(dbase + o_seed);
    pl->d_seeds = (uint64_t *)(dbase + o_seed);
    // concatenated host tables (cells < 2^32)
    std::vector<uint32_t> start32, info32, cell32;
    std::vector<double> cum, mean, sd;
    std::vector<uint32_t> tfile;
    start32.reserve(n_rows + 1);
    for (uint32_t i = 0; i < n_sets; ++i) {
        const Setup &s = lay[i];
        for (size_t r = 0; r < s.v.size(); ++r) {
            start32.push_back((uint32_t)(info[i].cell_base + s.start[r]));
            if (!filter) {
                info32.push_back(s.row_info[r]);
                continue;
            }
            const uint32_t fr = file_row[i][r];
            info32.push_back(row_word(s.row_info[r] & 0xFFu, (s.row_info[r] >> 8) & 1u, fr));
            cell32.push_back((uint32_t)(pl->setups[i].start[fr] - s.start[r]));
        }
        const uint32_t Ti = info[i].n_types;
        for (uint32_t j = 0; j < Ti; ++j) {
            cum.push_back(j < s.type_cum.size() ? s.type_cum[j] : 1.0);
            mean.push_back(j < s.type_mean.size() ? s.type_mean[j] : -1.0);
            sd.push_back(j < s.type_sd.size() ? s.type_sd[j] : -1.0);
            tfile.push_back(j < s.type_file.size() ? s.type_file[j] : 0u);
        }
    }
    start32.push_back((uint32_t)n_cells);
    info32.push_back(0u);
    // one copy for all tables (as separate copies of a few hundred bytes to a
    // few KB each, twelve of them took 52 us; one takes 14)
    std::vector<char> image(o_seed - o_rs, 0);
    auto put = [&](size_t o, const void *src, size_t bytes) {
        if (bytes)
            memcpy(&image[o - o_rs], src, bytes);
    };
    put(o_rs, start32.data(), start32.size() * 4);
    put(o_ri, info32.data(), info32.size() * 4);
    put(o_rc, cell32.data(), cell32.size() * 4);
    put(o_cum, cum.data(), cum.size() * 8);
    put(o_mean, mean.data(), mean.size() * 8);
    put(o_sd, sd.data(), sd.size() * 8);
    put(o_tf, tfile.data(), tfile.size() * 4);
    put(o_sb, seg_begin.data(), seg_begin.size() * 8);
    put(o_se, seg_end.data(), seg_end.size() * 8);
    put(o_sr, seg_row.data(), seg_row.size() * 4);
    put(o_ss, seg_set.data(), seg_set.size() * 4);
    put(o_info, info.data(), info.size() * sizeof(SetInfo));
    if (hipMemcpyAsync(dbase + o_rs, image.data(), image.size(), hipMemcpyHostToDevice, pl->stream) != hipSuccess)
        return fail(PROCELL_E_HIP);
    if (hipStreamSynchronize(pl->stream) != hipSuccess)
        return fail(PROCELL_E_HIP);
    if (pl->timing) {
        pl->kev.assign(2 * kTimedRuns, nullptr);
        for (hipEvent_t &e : pl->kev)
            if (hipEventCreate(&e) != hipSuccess)
                return fail(PROCELL_E_HIP);
    }
    if (n_sets > 1) {
        if (hipHostMalloc((void **)&pl->h_seeds, (size_t)kSeedSlots * n_sets * 8) != hipSuccess)
            return fail(PROCELL_E_OUT_OF_MEMORY);
        for (hipEvent_t &e : pl->seed_ev)
            if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess)
                return fail(PROCELL_E_HIP);
    }
    *out = pl;
    return PROCELL_OK;
}

// The run's kernels: clearing, then the simulation.
hipError_t launch_run(procell_plan *pl)
{
    hipError_t e = launch_zero(pl->args.counters, pl->zero_words, pl->stream);
    if (e == hipSuccess)
        e = launch_sim(pl->args, pl->shape, pl->stream);
    return e;
}

// Batch runs replay one graph of the two kernels; it is captured on the
// first run (the kernels read the seeds from device memory, so the graph
// does not change between runs) and again after the launch knobs change.
int capture_graph(procell_plan *pl)
{
    if (pl->graph_exec)
        return PROCELL_OK;
    HIP_TRY(hipStreamBeginCapture(pl->stream, hipStreamCaptureModeThreadLocal));
    const hipError_t e = launch_run(pl);
    hipGraph_t graph = nullptr;
    const hipError_t e2 = hipStreamEndCapture(pl->stream, &graph);
    if (e != hipSuccess || e2 != hipSuccess) {
        if (graph)
            (void)hipGraphDestroy(graph);
        g_last_hip = e != hipSuccess ? e : e2;
        return PROCELL_E_HIP;
    }
    pl->graph = graph;
    HIP_TRY(hipGraphInstantiate(&pl->graph_exec, pl->graph, nullptr, nullptr, 0));
    return PROCELL_OK;
}

void drop_graph(procell_plan *pl)
{
    if (pl->graph_exec)
        (void)hipGraphExecDestroy(pl->graph_exec);
    if (pl->graph)
        (void)hipGraphDestroy(pl->graph);
    pl->graph_exec = nullptr;
    pl->graph = nullptr;
}

// One run: every set gets seeds[i] (or `seed` when seeds is null).
int run_plan(procell_plan *pl, const uint64_t *seeds, uint64_t seed, bool use_graph = true)
{
    HIP_TRY(hipSetDevice(pl->device));
    const uint32_t n_sets = pl->args.n_sets;
    {
        // from here on the device's tallies may be this run's, also if a later
        // step fails: sets staged from an earlier run are not served any more
        std::lock_guard<std::mutex> lk(pl->result_mu);
        ++pl->run_id;
    }
    // timing events bracket the whole run: an event recorded between two
    // kernels of the run would add a gap of several microseconds there
    const size_t slot = (size_t)(pl->runs % kTimedRuns);
    if (n_sets == 1) {
        pl->args.seed = seeds ? seeds[0] : seed;
        if (pl->timing)
            HIP_TRY(hipEventRecord(pl->kev[2 * slot], pl->stream));
        HIP_TRY(launch_run(pl));
    } else {
        // stage the seeds in a pinned slot whose previous copy has run, and
        // copy them to the device ahead of the kernels
        const uint32_t k = (uint32_t)(pl->batch_runs % kSeedSlots);
        HIP_TRY(hipEventSynchronize(pl->seed_ev[k]));
        uint64_t *h = pl->h_seeds + (size_t)k * n_sets;
        for (uint32_t i = 0; i < n_sets; ++i)
            h[i] = seeds ? seeds[i] : seed;
        HIP_TRY(hipMemcpyAsync(pl->d_seeds, h, (size_t)n_sets * 8, hipMemcpyHostToDevice, pl->stream));
        HIP_TRY(hipEventRecord(pl->seed_ev[k], pl->stream));
        ++pl->batch_runs;
        if (use_graph) {
            const int rc = capture_graph(pl);
            if (rc != PROCELL_OK)
                return rc;
        }
        if (pl->timing)
            HIP_TRY(hipEventRecord(pl->kev[2 * slot], pl->stream));
        if (use_graph)
            HIP_TRY(hipGraphLaunch(pl->graph_exec, pl->stream));
        else
            HIP_TRY(launch_run(pl));
    }
    if (pl->timing)
        HIP_TRY(hipEventRecord(pl->kev[2 * slot + 1], pl->stream));
    if (pl->timing) {
        pl->last_slot = slot;
        pl->timed = true;
    }
    ++pl->runs;
    pl->ran = true;
    return PROCELL_OK;
}

// Downloads one set's counter copies and tally.  A batch's sets are usually
// read one after the other, so a set that follows the last download brings
// twice as many along, up to kStageBytes; they serve later calls until the
// next run.  (512 sets one by one: two copies and a wait, about 35 us, each.)
constexpr size_t kStageBytes = 8u << 20;

int download_set(procell_plan *pl, uint32_t set, std::vector<unsigned long long> &counters, std::vector<int64_t> &tally)
{
    constexpr size_t kCntBytes = (size_t)kCounterCopies * kNumCounters * 8;
    const uint32_t n_sets = pl->args.n_sets;
    counters.resize(kCntBytes / 8);
    tally.resize(pl->tally_len[set]);
    auto fetch = [&](char *cnt, char *tal, uint32_t a, uint32_t b) -> int {
        const size_t tal_bytes = (pl->tally_base[b - 1] + pl->tally_len[b - 1] - pl->tally_base[a]) * 8;
        const char *d_cnt = (const char *)pl->args.counters + a * kCntBytes;
        const char *d_tal = (const char *)(pl->args.tally + pl->tally_base[a]);
        if (n_sets == 1 && tal == cnt + kCntBytes) {  // (a single set's counters and tally lie together)
            HIP_TRY(hipMemcpyAsync(cnt, d_cnt, kCntBytes + tal_bytes, hipMemcpyDeviceToHost, pl->stream));
        } else {
            HIP_TRY(hipMemcpyAsync(cnt, d_cnt, (b - a) * kCntBytes, hipMemcpyDeviceToHost, pl->stream));
            if (tal_bytes)
                HIP_TRY(hipMemcpyAsync(tal, d_tal, tal_bytes, hipMemcpyDeviceToHost, pl->stream));
        }
        HIP_TRY(hipStreamSynchronize(pl->stream));
        return PROCELL_OK;
    };
    std::lock_guard<std::mutex> lk(pl->result_mu);
    if (n_sets == 1 || pl->stage_run != pl->run_id || set < pl->stage_set || set >= pl->stage_end) {  // (runs count from 1)
        auto bytes_of = [&](uint32_t n) {
            return n * kCntBytes + (pl->tally_base[set + n - 1] + pl->tally_len[set + n - 1] - pl->tally_base[set]) * 8;
        };
        uint32_t want = pl->next_run == pl->run_id && set == pl->next_set ? std::min(pl->next_n, n_sets - set) : 1;
        while (want > 1 && bytes_of(want) > kStageBytes)
            want /= 2;
        const size_t need = bytes_of(want);
        pl->next_run = pl->run_id;
        pl->next_set = set + want;
        pl->next_n = 2 * want;
        pl->stage_run = 0;
        if (pl->own_block && pl->results++ > 0 && need <= kStageBytes && need > pl->stage_bytes) {
            if (pl->stage)
                (void)hipHostFree(pl->stage);
            pl->stage_bytes = n_sets > 1 ? kStageBytes : need;
            if (hipHostMalloc(&pl->stage, pl->stage_bytes) != hipSuccess) {
                (void)hipGetLastError();
                pl->stage = nullptr;
                pl->stage_bytes = 0;
            }
        }
        if (need > pl->stage_bytes) {  // no pinned memory: this set, straight to the caller's buffers
            pl->next_set = set + 1;
            return fetch((char *)counters.data(), (char *)tally.data(), set, set + 1);
        }
        const int rc = fetch((char *)pl->stage, (char *)pl->stage + want * kCntBytes, set, set + want);
        if (rc != PROCELL_OK)
            return rc;
        pl->stage_run = pl->run_id;
        pl->stage_set = set;
        pl->stage_end = set + want;
    }
    const uint32_t n = pl->stage_end - pl->stage_set, i = set - pl->stage_set;
    memcpy(counters.data(), (const char *)pl->stage + i * kCntBytes, kCntBytes);
    if (!tally.empty())
        memcpy(tally.data(), (const char *)pl->stage + n * kCntBytes + (pl->tally_base[set] - pl->tally_base[pl->stage_set]) * 8,
               tally.size() * 8);
    return PROCELL_OK;
}

int plan_result(procell_plan *pl, uint32_t set, procell_result *r)
{
    if (!r || !pl->ran || set >= pl->args.n_sets)
        return PROCELL_E_INVALID;
    const Setup &s = pl->setups[set];
    const size_t tally_len = pl->tally_len[set];
    if (r->capacity && !(r->value && r->count))
        return PROCELL_E_INVALID;
    HIP_TRY(hipSetDevice(pl->device));
    std::vector<unsigned long long> cnt_all, cnt(kNumCounters, 0);
    std::vector<int64_t> tally;
    const int rc = download_set(pl, set, cnt_all, tally);
    if (rc != PROCELL_OK)
        return rc;
    for (size_t i = 0; i < cnt_all.size(); ++i)
        cnt[i % kNumCounters] += cnt_all[i];
    procell_stats &st = r->stats;
    fill_stats(cnt.data(), tally.data(), tally_len, st);
    st.workgroups = (uint32_t)pl->shape.blocks;
    st.block_size = (uint32_t)pl->shape.block_size;
    st.lds_bytes = (uint32_t)pl->shape.lds_bytes;
    st.window_rows = pl->args.win_rows;
    if (pl->timing && pl->timed) {
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, pl->kev[2 * pl->last_slot], pl->kev[2 * pl->last_slot + 1]));
        st.ms_tree = ms;
        st.ms_run = ms;
    }
    if (r->raw_tally) {
        if (r->raw_tally_len < tally_len)
            return PROCELL_E_CAPACITY;
        memcpy(r->raw_tally, tally.data(), tally_len * 8);
    }
    const std::vector<int32_t> *bin_of = nullptr;
    {
        std::lock_guard<std::mutex> lk(pl->result_mu);
        if (pl->bin_of.empty())
            pl->bin_of.resize(pl->args.n_sets);
        if (pl->bin_of[set].empty())
            pl->bin_of[set] = index_bins(s);
        bin_of = &pl->bin_of[set];
    }
    return merge_tally(s, *bin_of, tally.data(), r);
}

// Streams of procell_simulate calls: making and destroying one took 58 us of a
// small call's 146.  Up to kKeptStreams idle ones per device wait for the next
// call; a call takes one for itself and gives it back once its work has ended,
// so concurrent calls never share one.  The host program's hipDeviceReset
// deletes them with everything else on the device, and their handles may then
// belong to streams of its own.  So a small device allocation is kept beside
// them: while the runtime knows it by the same allocation id (unique in the
// process; 0.06 us to ask for), there was no reset, else the handles are
// forgotten and never used.
constexpr int kKeptDevices = 64, kKeptStreams = 4;
struct KeptStreams {
    std::mutex mu;
    hipStream_t stream[kKeptStreams];
    int n = 0;
    void *mark = nullptr;
    uint64_t mark_id = 0;
};
KeptStreams g_kept[kKeptDevices];

// The id of a device allocation, 0 if there is none at p.
uint64_t allocation_id(void *p)
{
    uint64_t id = 0;
    if (!p || hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return id;
}

// Whether k's streams still exist (under k.mu).
bool kept_valid(KeptStreams &k)
{
    if (k.mark && allocation_id(k.mark) == k.mark_id)
        return true;
    k.n = 0;
    k.mark = nullptr;
    return false;
}

hipStream_t borrow_stream(int device)
{
    if (device < 0 || device >= kKeptDevices)
        return nullptr;
    {
        KeptStreams &k = g_kept[device];
        std::lock_guard<std::mutex> lk(k.mu);
        if (kept_valid(k) && k.n > 0)
            return k.stream[--k.n];
    }
    int n_cu = 0;
    hipStream_t st = nullptr;
    if (check_device(device, &n_cu) != PROCELL_OK || hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess)
        return nullptr;  // (the plan reports what is wrong)
    return st;
}

void return_stream(int device, hipStream_t st)
{
    if (!st)
        return;
    if (hipSetDevice(device) == hipSuccess && hipStreamSynchronize(st) == hipSuccess) {
        KeptStreams &k = g_kept[device];
        std::lock_guard<std::mutex> lk(k.mu);
        if (!kept_valid(k)) {
            void *mark = nullptr;
            if (hipMalloc(&mark, 8) == hipSuccess) {
                k.mark_id = allocation_id(mark);
                if (k.mark_id)
                    k.mark = mark;
                else  // a runtime without ids: nothing is kept
                    (void)hipFree(mark);
            }
        }
        if (k.mark && k.n < kKeptStreams) {
            k.stream[k.n++] = st;
            return;
        }
    }
    (void)hipStreamDestroy(st);
}

// In host code `scratch` names a host-side stand-in, not device memory: the
// device address of each GPU's copy comes from hipGetSymbolAddress, taken
// once per device with that device current, and only that address is handed
// to kernels and copies.
constexpr int kScratchDevices = 64;

std::mutex g_scratch_mu[kScratchDevices];  // held for a whole call on that device
std::mutex g_scratch_addr_mu;
void *g_scratch_ptr[kScratchDevices] = {};

// Device address of `device`'s scratch array; the device must be current.
int scratch_address(int device, void **ptr)
{
    std::lock_guard<std::mutex> lk(g_scratch_addr_mu);
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p)
            return PROCELL_E_HIP;
        g_scratch_ptr[device] = p;
    }
    *ptr = g_scratch_ptr[device];
    return PROCELL_OK;
}

}  // namespace

extern "C" {

int procell_abi_version(void) { return PROCELL_ABI_VERSION; }

const char *procell_strerror(int code)
{
    switch (code) {
    case PROCELL_OK: return "success";
    case PROCELL_E_INVALID: return "invalid argument";
    case PROCELL_E_PROPORTIONS: return "proportion distribution of cell types does not sum to 1";
    case PROCELL_E_ZERO_MEAN: return "a cell type has mean 0";
    case PROCELL_E_NONFINITE: return "non-finite value in the input";
    case PROCELL_E_PHI: return "phi must be > 0";
    case PROCELL_E_DEPTH: return "division tree deeper than 62 generations (phi too small)";
    case PROCELL_E_TOO_MANY_CELLS: return "input exceeds 2^32-1 cells, 2^24 rows or 256 types";
    case PROCELL_E_CAPACITY: return "result buffer too small";
    case PROCELL_E_HIP: return hipGetErrorString(g_last_hip);
    case PROCELL_E_NO_DEVICE: return "no usable gfx950 device";
    case PROCELL_E_IO: return "cannot write output file";
    case PROCELL_E_OUT_OF_MEMORY: return "out of memory";
    case PROCELL_E_SCRATCH: return "input needs more device memory than the 16 MiB static scratch of procell_simulate_noalloc";
    default: return "unknown error";
    }
}

int procell_plan_create(const procell_params *p, procell_plan **plan) { return create_plan(p, 1, plan); }

int procell_plan_run(procell_plan *plan, uint64_t seed)
{
    if (!plan)
        return PROCELL_E_INVALID;
    return run_plan(plan, nullptr, seed);
}

int procell_plan_result(procell_plan *plan, procell_result *r)
{
    if (!plan)
        return PROCELL_E_INVALID;
    return plan_result(plan, 0, r);
}

int procell_batch_create(const procell_params *sets, uint32_t n_sets, procell_plan **plan)
{
    return create_plan(sets, n_sets, plan);
}

int procell_batch_run(procell_plan *plan, const uint64_t *seeds)
{
    if (!plan || !seeds)
        return PROCELL_E_INVALID;
    return run_plan(plan, seeds, 0);
}

int procell_batch_result(procell_plan *plan, uint32_t set, procell_result *r)
{
    if (!plan)
        return PROCELL_E_INVALID;
    return plan_result(plan, set, r);
}

int procell_batch_autotune(procell_plan *plan, const uint64_t *seeds, uint32_t reps, procell_tuning *chosen)
{
    return procell_plan_autotune(plan, seeds, reps, chosen);
}

// Device time of warm-up + reps runs (eager launches) of a plan.
static int time_plan(procell_plan *pl, const uint64_t *seeds, uint32_t reps, hipEvent_t e0, hipEvent_t e1, float *ms)
{
    const bool timing = pl->timing;
    pl->timing = false;
    int rc = run_plan(pl, seeds, 0, false);  // warm-up
    if (rc == PROCELL_OK && hipEventRecord(e0, pl->stream) != hipSuccess)
        rc = PROCELL_E_HIP;
    for (uint32_t i = 0; rc == PROCELL_OK && i < reps; ++i)
        rc = run_plan(pl, seeds, 0, false);
    if (rc == PROCELL_OK &&
        (hipEventRecord(e1, pl->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
         hipEventElapsedTime(ms, e0, e1) != hipSuccess))
        rc = PROCELL_E_HIP;
    pl->timing = timing;
    return rc;
}

int procell_plan_autotune(procell_plan *plan, const uint64_t *seeds, uint32_t reps, procell_tuning *chosen)
{
    if (!plan || !seeds || !chosen || reps == 0)
        return PROCELL_E_INVALID;
    HIP_TRY(hipSetDevice(plan->device));
    // layouts: resident workgroups per CU (sets the LDS tally window's
    // width) x segments per resident workgroup; for each, the idle-lane
    // threshold, which needs no new layout.  More workgroups than a CU holds
    // are the layout of as many as it holds: timed once, and reported as that.
    static const uint32_t kBlocks[] = {2, 3, 4};
    static const uint32_t kSegments[] = {1, 2, 3, 4, 8};
    static const uint32_t kIdle[] = {6, 8, 12, 16};
    hipEvent_t e0 = nullptr, e1 = nullptr;
    HIP_TRY(hipEventCreate(&e0));
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return PROCELL_E_HIP;
    }
    const uint32_t n_sets = plan->args.n_sets;
    std::vector<procell_params> ps = plan->params;
    float best = -1.f;
    procell_plan *best_plan = nullptr;
    procell_tuning best_tu{};
    int rc = PROCELL_OK, per_cu = 0;
    for (uint32_t bpc : kBlocks) {
        const int timed = per_cu;  // workgroups per CU of the layouts before
        for (uint32_t seg : kSegments) {
            for (procell_params &p : ps) {
                p.tuning.blocks_per_cu = bpc;
                p.tuning.segments = seg;
                p.tuning.idle_lanes = 0;
                p.tuning.flags &= ~PROCELL_FLAG_TIMING;  // candidates need no timing ring
                p.stream = (void *)plan->stream;         // and run on the plan's stream
            }
            procell_plan *cand = nullptr;
            rc = create_plan(ps.data(), n_sets, &cand);
            if (rc != PROCELL_OK)
                break;
            cand->own_stream = false;
            per_cu = cand->per_cu;
            if (per_cu == timed) {
                destroy_plan(cand);
                break;
            }
            bool kept = false;
            for (uint32_t idle : kIdle) {
                cand->args.idle_limit = idle;
                float ms = 0.f;
                rc = time_plan(cand, seeds, reps, e0, e1, &ms);
                if (rc != PROCELL_OK)
                    break;
                if (best < 0.f || ms < best) {
                    best = ms;
                    best_tu = ps[0].tuning;
                    best_tu.blocks_per_cu = (uint32_t)per_cu;
                    best_tu.idle_lanes = idle;
                    if (best_plan && best_plan != cand)
                        destroy_plan(best_plan);
                    best_plan = cand;
                    kept = true;
                }
            }
            if (best_plan == cand)
                best_plan->args.idle_limit = best_tu.idle_lanes;
            if (!kept)
                destroy_plan(cand);
            if (rc != PROCELL_OK)
                break;
        }
        if (rc != PROCELL_OK)
            break;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != PROCELL_OK || !best_plan) {
        if (best_plan)
            destroy_plan(best_plan);
        return rc != PROCELL_OK ? rc : PROCELL_E_INVALID;
    }
    // the plan takes the fastest candidate's layout; its own stream, events
    // and timing ring stay
    drop_graph(plan);
    std::swap(plan->shape, best_plan->shape);
    std::swap(plan->per_cu, best_plan->per_cu);
    std::swap(plan->args, best_plan->args);
    std::swap(plan->d_block, best_plan->d_block);
    std::swap(plan->tally_total, best_plan->tally_total);
    std::swap(plan->zero_words, best_plan->zero_words);
    std::swap(plan->d_seeds, best_plan->d_seeds);
    std::swap(plan->tally_base, best_plan->tally_base);
    std::swap(plan->tally_len, best_plan->tally_len);
    std::swap(plan->setups, best_plan->setups);
    best_tu.flags = plan->params[0].tuning.flags;
    for (uint32_t i = 0; i < n_sets; ++i)
        plan->params[i].tuning = best_tu;
    destroy_plan(best_plan);
    plan->runs = 0;
    plan->ran = false;
    *chosen = best_tu;
    return PROCELL_OK;
}

int procell_plan_destroy(procell_plan *plan)
{
    destroy_plan(plan);
    return PROCELL_OK;
}

void *procell_plan_stream(procell_plan *plan) { return plan ? (void *)plan->stream : nullptr; }

int procell_plan_kernel_times(procell_plan *plan, double *ms, uint32_t max_runs, uint32_t *n_runs)
{
    if (!plan || !n_runs || (max_runs && !ms))
        return PROCELL_E_INVALID;
    if (!plan->timing)
        return PROCELL_E_INVALID;
    HIP_TRY(hipSetDevice(plan->device));
    HIP_TRY(hipStreamSynchronize(plan->stream));
    const uint64_t avail = plan->runs < kTimedRuns ? plan->runs : kTimedRuns;
    const uint32_t n = (uint32_t)(avail < max_runs ? avail : max_runs);
    for (uint32_t i = 0; i < n; ++i) {
        const size_t slot = (size_t)((plan->runs - n + i) % kTimedRuns);
        float t = 0.f;
        HIP_TRY(hipEventElapsedTime(&t, plan->kev[2 * slot], plan->kev[2 * slot + 1]));
        ms[i] = t;
    }
    *n_runs = n;
    plan->runs = 0;
    return PROCELL_OK;
}

int procell_simulate(const procell_params *p, procell_result *r)
{
    if (!p || !r)
        return PROCELL_E_INVALID;
    procell_params q = *p;
    q.stream = borrow_stream(p->device);  // NULL: the plan makes its own
    procell_plan *pl = nullptr;
    int rc = create_plan(&q, 1, &pl);
    if (rc == PROCELL_OK) {
        rc = run_plan(pl, nullptr, p->seed);
        if (rc == PROCELL_OK)
            rc = plan_result(pl, 0, r);
        destroy_plan(pl);
    }
    return_stream(p->device, (hipStream_t)q.stream);
    return rc;
}

int procell_simulate_noalloc(const procell_params *p, procell_result *r)
{
    if (!p || !r)
        return PROCELL_E_INVALID;
    int n_cu = 0;
    int rc = check_device(p->device, &n_cu);  // makes the device current
    if (rc != PROCELL_OK)
        return rc;
    if (p->device >= kScratchDevices)
        return PROCELL_E_INVALID;
    std::lock_guard<std::mutex> lk(g_scratch_mu[p->device]);
    void *ptr = nullptr;
    rc = scratch_address(p->device, &ptr);
    if (rc != PROCELL_OK)
        return rc;
    procell_params q = *p;
    q.tuning.flags &= ~PROCELL_FLAG_TIMING;
    procell_plan *pl = nullptr;
    rc = create_plan(&q, 1, &pl, ptr, kScratchBytes);
    if (rc != PROCELL_OK)
        return rc;
    rc = run_plan(pl, nullptr, p->seed);
    if (rc == PROCELL_OK)
        rc = plan_result(pl, 0, r);
    destroy_plan(pl);
    return rc;
}

int procell_debug_draws(int32_t device, uint64_t seed, const uint64_t *cell, const uint64_t *node,
                        const uint32_t *attempt, uint64_t n, uint32_t *words, double *z)
{
    if (n && (!cell || !node || !attempt || !words || !z))
        return PROCELL_E_INVALID;
    int n_cu = 0;
    int rc = check_device(device, &n_cu);
    if (rc != PROCELL_OK)
        return rc;
    if (n == 0)
        return PROCELL_OK;
    void *d = nullptr;
    const size_t bytes = n * (8 + 8 + 4 + 16 + 16);
    if (hipMalloc(&d, bytes) != hipSuccess)
        return PROCELL_E_OUT_OF_MEMORY;
    char *b = (char *)d;
    uint64_t *dc = (uint64_t *)b;
    uint64_t *dn = (uint64_t *)(b + n * 8);
    double *dz = (double *)(b + n * 16);
    uint32_t *dw = (uint32_t *)(b + n * 32);
    uint32_t *da = (uint32_t *)(b + n * 48);
    hipError_t e = hipMemcpy(dc, cell, n * 8, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dn, node, n * 8, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(da, attempt, n * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = launch_debug_draws(seed, dc, dn, da, n, dw, dz, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(words, dw, n * 16, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(z, dz, n * 16, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) {
        g_last_hip = e;
        return PROCELL_E_HIP;
    }
    return PROCELL_OK;
}

// For tests, not part of the C ABI: bounds[4] as launch_pair_bounds.
int procell_debug_pair_bounds(int32_t device, double *bounds)
{
    if (!bounds)
        return PROCELL_E_INVALID;
    int n_cu = 0;
    const int rc = check_device(device, &n_cu);
    if (rc != PROCELL_OK)
        return rc;
    void *d = nullptr;
    if (hipMalloc(&d, 4 * sizeof(double)) != hipSuccess)
        return PROCELL_E_OUT_OF_MEMORY;
    hipError_t e = launch_zero((unsigned long long *)d, 4, nullptr);
    if (e == hipSuccess) e = launch_pair_bounds((unsigned long long *)d, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(bounds, d, 4 * sizeof(double), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) {
        g_last_hip = e;
        return PROCELL_E_HIP;
    }
    return PROCELL_OK;
}

}  // extern "C"
