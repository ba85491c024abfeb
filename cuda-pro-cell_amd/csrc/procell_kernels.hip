// procell_kernels.hip -- gfx950 kernels of the plain proliferation method.
//
// The reference materialises every tree level as a dense array of 40-byte
// cells and recurses with device-side launches (src/simulation/
// proliferation.cu:289-402), creating the initial cells in a separate pass
// (cells_population.cu:74-117).  Here one persistent kernel does the whole
// run and no cell is ever stored in device memory: each wavefront draws its
// own initial cells (root steps, 64 at a time) into a small LDS buffer,
// hands the dividing ones to idle lanes, and every lane walks its cell's
// division tree depth first, keeping only the pending right daughters'
// completion times in its column of an LDS stack.  Work is balanced without
// device-scope coordination: the initial cells are split into several
// segments of about equal expected work per resident workgroup and the
// hardware dispatcher starts the workgroup of the next segment wherever one
// finishes; inside a workgroup, wavefronts claim root steps from an LDS
// cursor, and at the very end idle lanes take pending daughters of busy
// lanes of the same wavefront.  (Claims and work stealing through device
// memory were measured here: a device-scope probe of other workgroups'
// cursors took tens of microseconds under load.)
//
// Tallies (counts by nonzero row, generation, type) accumulate in a u32 LDS
// window over the first rows of the workgroup's segment and are added to the
// int64 device tally at the end; rows outside the window use 64-bit device
// atomics (aggregated per (row, type) for generation 0).
#include "procell_filter.hpp"
#include "procell_internal.hpp"
#include "procell_stream.hpp"

namespace procell {
namespace {

using dev::Words;

constexpr uint32_t kWave = 64;
constexpr uint32_t kNoWindow = 0xFFFFFFFFu;

__device__ __forceinline__ uint32_t lane_rank(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t x)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        x += __shfl_xor(x, off);
    return x;
}

// Index of the r-th set bit of m (r < popcount(m)).
__device__ __forceinline__ uint32_t nth_set_bit(uint64_t m, uint32_t r)
{
    uint32_t base = 0;
#pragma unroll
    for (uint32_t width = 32; width >= 1; width >>= 1) {
        const uint64_t low = m & ((width == 64 ? ~0ull : (1ull << width)) - 1ull);
        const uint32_t c = (uint32_t)__popcll(low);
        if (r >= c) {
            r -= c;
            m >>= width;
            base += width;
        } else {
            m = low;
        }
    }
    return base;
}

// Wave-uniform copies (lane 0's value).  The builtin works on int, so each
// half goes back through uint32_t: a widened int would be sign-extended.
__device__ __forceinline__ uint32_t uni(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

__device__ __forceinline__ uint64_t uni64(uint64_t x)
{
    return ((uint64_t)uni((uint32_t)(x >> 32)) << 32) | (uint64_t)uni((uint32_t)x);
}

__global__ void zero_kernel(unsigned long long *p, uint64_t n)
{
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

// Per-lane event counts.  Recorded and dropped cells are not counted on the
// device: the host takes recorded = the sum of the tally and dropped = cells
// + divisions - recorded - lost (every division adds one cell, and every
// cell ends recorded, dropped or lost).
// LDS copies of the stream's lookup tables (procell_math_tables.inc).
constexpr size_t kMathTableBytes = (128 + 256) * 16;

__device__ __forceinline__ void copy_tables(double (*m_log)[2], double (*m_sc)[2], uint32_t tid, uint32_t bdim)
{
    for (uint32_t i = tid; i < 128; i += bdim) {
        m_log[i][0] = dev::procell_log_table[i][0];
        m_log[i][1] = dev::procell_log_table[i][1];
    }
    for (uint32_t i = tid; i < 256; i += bdim) {
        m_sc[i][0] = dev::procell_sincos_table[i][0];
        m_sc[i][1] = dev::procell_sincos_table[i][1];
    }
}

struct Counts {
    uint32_t div, rej, lost, cells, pool;
};

// place of the refused candidates among the sums flush_counts makes in `red`
constexpr uint32_t kRedRejected = 3;

// Adds a workgroup's counts to counter copy blockIdx.x % kCounterCopies:
// wavefront sums, then one LDS atomic per wavefront and counter, then one
// device atomic per counter.  `red` is kNumCounters u32 of LDS, zeroed and
// followed by a barrier before the first call; every thread calls it.
__device__ __forceinline__ void flush_counts(const Counts &n, unsigned long long *counters, uint32_t lane,
                                             uint32_t *red)
{
    constexpr uint32_t kN = 5;
    const uint32_t v[kN] = {wave_sum(n.pool), wave_sum(n.div), wave_sum(n.lost), wave_sum(n.rej),
                            wave_sum(n.cells)};
    const uint32_t idx[kN] = {kPoolCount, kDivisions, kLost, kRejected, kCells};
    if (lane < kN) {
        uint32_t x = v[0];
#pragma unroll
        for (uint32_t i = 1; i < kN; ++i)
            x = lane == i ? v[i] : x;
        if (x)
            atomicAdd(&red[lane], x);
    }
    __syncthreads();
    if (threadIdx.x < kN) {
        const uint32_t x = red[threadIdx.x];
        uint32_t c = idx[0];
#pragma unroll
        for (uint32_t i = 1; i < kN; ++i)
            c = threadIdx.x == i ? idx[i] : c;
        if (x)
            atomicAdd(&counters[(blockIdx.x % kCounterCopies) * kNumCounters + c], (unsigned long long)x);
    }
}

// Highest / lowest set bit of a nonzero 32- or 64-bit mask.
__device__ __forceinline__ uint32_t top_bit(uint32_t m) { return 31u - (uint32_t)__builtin_clz(m); }
__device__ __forceinline__ uint32_t top_bit(uint64_t m) { return 63u - (uint32_t)__builtin_clzll(m); }
__device__ __forceinline__ uint32_t low_bit(uint32_t m) { return (uint32_t)__builtin_ctz(m); }
__device__ __forceinline__ uint32_t low_bit(uint64_t m) { return (uint32_t)__builtin_ctzll(m); }

// Lane state: the dividing cell a lane currently holds.  N holds a node's
// heap index and the pending-level mask: 32 bits when no tree is deeper than
// 31 generations, else 64.
template <typename N>
struct Lane {
    uint32_t cell;      // initial cell, relative to its set (cell ids < 2^32)
    N node, pend;
    uint32_t rowtf;     // row relative to the set's first row | file type << 24
    double s, mean, sd;
    double tl, tr;      // daughters' timers of the division in progress
    uint32_t k, kcap;
    uint32_t tb_lds;    // window index of (row, generation 0, type), or kNoWindow
    uint32_t redo;      // bit 0 / bit 1: left / right daughter's timer still to redraw
    uint32_t att;       // attempt number of that redraw
    bool active;
};

// ======================================================================
// sim_kernel: workgroup g runs segment g of the initial cells (contiguous,
// of about equal expected work; several per resident workgroup, so that the
// dispatcher balances them over the CUs); its wavefronts work independently:
//  * claims: a wavefront claims the segment's next root step (64 cells)
//    with one LDS atomic on the workgroup's cursor.
//  * root steps (cell.cu:25-143, cells_population.cu:97-117): when the
//    wavefront's buffer of dividing roots is empty and lanes are idle, the
//    64 lanes draw the next 64 initial cells of the segment, one each, whatever
//    the lanes hold: type, truncated first timer, phase.  Cells that never
//    divide are tallied at generation 0 (or lost); dividing ones become
//    48-byte entries of the wavefront's LDS buffer.
//  * hand-outs: idle lanes take buffered entries right before each division
//    step (the one place in the loop where lane state is handed over, so
//    that the compiler keeps the lane state in the same registers on every
//    path: with a second hand-out site in the refill branch the loop carried
//    about 40 register copies per refill, 3.5 % of the run); once the roots
//    are done and the buffer is empty, idle lanes take the shallowest pending
//    right daughter of a busy lane of the wavefront.
//  * refills (root steps, steals) run as a uniform branch of the one loop,
//    once more than idle_limit lanes are idle.
//  * division steps (proliferation.cu:317-381): each busy lane divides its
//    current cell per step: one Philox block and one Box-Muller pair give
//    both daughters' timers; daughters that will not divide are tallied or
//    dropped on the spot, so the lane's next cell is always a dividing one
//    (the left daughter, else the right, else the deepest pending right
//    daughter from the lane's column of the LDS stack).
// LDS: log and sin/cos tables | stream coefficients | type tables ((mean,
// sd): double2 [T]; cum: double [T]; file: u32 [T]) | row tables when they fit (first
// cell: u32 [n_rows + 1]; info: u32 [n_rows]) | counter sums u32 [8] | root
// step cursor u32 [4] | per wavefront: buffered entries QueueEntry [64] |
// window tally u32 [win_rows * kdim * T + 1 spare] | stack double
// [stack_levels * blockDim]
// ======================================================================
__host__ __device__ constexpr size_t sim_wave_lds_bytes()
{
    return (size_t)kWave * sizeof(QueueEntry);
}

constexpr size_t kSimSharedBytes = 48;  // counter sums u32 [8], root step cursor u32 [4]

template <bool RowsLds, typename N, bool GStack>
__global__ void __launch_bounds__(256, 4) sim_kernel(RunArgs a)
{
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t tid = threadIdx.x;
    const uint32_t bdim = blockDim.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = tid / kWave;
    const uint32_t n_waves = bdim / kWave;
    const uint32_t seg0 = blockIdx.x;
    // the workgroup's parameter set (every segment it drains belongs to it)
    const uint32_t set = a.n_sets > 1 ? a.seg_set[seg0] : 0u;
    const SetInfo S = a.sets[set];
    const uint64_t seed = a.n_sets > 1 ? a.set_seed[set] : a.seed;
    const double t_max = S.t_max;
    const uint32_t T = S.n_types;
    const uint32_t kdim = S.kdim;
    const uint32_t win_len = a.win_rows * kdim * T;
    const uint32_t lds_rows = RowsLds ? a.n_rows : 0u;
    double(*m_log)[2] = (double(*)[2])lds;            // [128] log table
    double(*m_sc)[2] = (double(*)[2])(lds + 128 * 16);  // [256] sin/cos table
    dev::Coeffs *k_lds = (dev::Coeffs *)(lds + kMathTableBytes);
    double2 *t_msd = (double2 *)(lds + kMathTableBytes + (sizeof(dev::Coeffs) + 15) / 16 * 16);  // mean, sd
    double *t_cum = (double *)(t_msd + T);
    uint32_t *t_file = (uint32_t *)(t_cum + T);
    uint32_t *r_start = (uint32_t *)((unsigned char *)t_msd + ((size_t)T * 28 + 15) / 16 * 16);
    uint32_t *r_info = r_start + lds_rows + 1;
    uint32_t *red = (uint32_t *)((unsigned char *)r_start + (RowsLds ? ((size_t)(2 * lds_rows + 1) * 4 + 15) / 16 * 16 : 0));
    uint32_t *cursor = red + kNumCounters;  // root steps of the segment claimed so far
    QueueEntry *ent = (QueueEntry *)((unsigned char *)red + kSimSharedBytes + (size_t)wave * sim_wave_lds_bytes());
    unsigned int *win = (unsigned int *)((unsigned char *)red + kSimSharedBytes + (size_t)n_waves * sim_wave_lds_bytes());
    // the lanes' stacks: in LDS after the window, or (GStack: plans whose
    // deep trees would leave no LDS for the window) the workgroup's block of
    // device memory, same layout
    double *stack = GStack ? (double *)a.gstack + (size_t)seg0 * a.stack_levels * bdim
                           : (double *)((unsigned char *)win + ((size_t)win_len * 4 + 4 + 15) / 16 * 16);
    // the lane's stack column: level l (1-based) at stk_pop + l * stride,
    // i.e. at stk_push + (l - 1) * stride (bytes)
    const uint32_t stride = bdim * (uint32_t)sizeof(double);
    unsigned char *const stk_push = (unsigned char *)(stack + tid);
    unsigned char *const stk_pop = stk_push - stride;

    const uint64_t seg_begin = uni64(a.seg_begin[seg0]);
    const uint64_t seg_cells = uni64(a.seg_end[seg0]) - seg_begin;
    const uint32_t row_lo = uni(a.seg_row[seg0]);  // first row of the segment and of the tally window
    if (tid == 0)
        *k_lds = dev::coeffs();
    copy_tables(m_log, m_sc, tid, bdim);
    for (uint32_t i = tid; i < T; i += bdim) {
        t_cum[i] = a.type_cum[S.type_base + i];
        t_msd[i] = make_double2(a.type_mean[S.type_base + i], a.type_sd[S.type_base + i]);
        t_file[i] = a.type_file[S.type_base + i];
    }
    for (uint32_t i = tid; i <= lds_rows && RowsLds; i += bdim)
        r_start[i] = a.row_start[i];
    for (uint32_t i = tid; i < lds_rows; i += bdim)
        r_info[i] = a.row_info[i];
    for (uint32_t i = tid; i <= win_len; i += bdim)
        win[i] = 0u;  // win[win_len] absorbs the adds of lanes outside the window
    if (tid < kNumCounters + 1)
        red[tid] = 0u;  // counter sums and the root step cursor
    __syncthreads();

    // the stream's FP64 coefficients, held in vector registers for the whole
    // kernel (loaded from LDS, so they are not re-materialised as scalar literals)
    const dev::Coeffs K = *k_lds;
    const dev::Tables tb{m_log, m_sc};
    // the row tables' address space is known at compile time (no flat loads)
    const uint32_t *rs = RowsLds ? r_start : a.row_start;
    const uint32_t *ri = RowsLds ? r_info : a.row_info;

    uint32_t rpos = 0, rn = 0;      // buffered dividing roots: entries [rpos, rn) of ent
    uint32_t roots_done = 0;
    // the first eight cumulative proportions of the type search, in scalar
    // registers (-inf for types not searched: the last one and those beyond T;
    // in vector registers they would take the 16 that keep the kernel within
    // the 128 of four wavefronts per SIMD)
    double cum8[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k)
        cum8[k] = __builtin_bit_cast(double, uni64(__builtin_bit_cast(uint64_t, k + 1 < T ? t_cum[k] : -__builtin_inf())));
    // Row boundaries of the wavefront's root steps, in registers: lane j holds
    // the first cell of row rb + 1 + j (~0 past the last row) and the info of
    // row rb + j.  A wavefront's root steps only move forward in its segment,
    // so rb only grows.
    uint32_t rb = row_lo, bnd = 0, rinfo = 0;
    auto load_rows = [&]() {
        const uint32_t r1 = rb + 1 + lane;
        bnd = r1 <= a.n_rows ? rs[r1] : 0xFFFFFFFFu;
        rinfo = rb + lane < a.n_rows ? ri[rb + lane] : 0u;
    };
    load_rows();

    Lane<N> L;
    L.cell = 0;
    L.rowtf = 0;
    L.node = L.pend = 0;
    L.s = L.mean = L.sd = L.tl = L.tr = 0.0;
    L.k = L.kcap = 0;
    L.redo = 0;
    L.att = 1;
    L.tb_lds = kNoWindow;
    L.active = false;
    Counts n = {0, 0, 0, 0, 0};
    uint32_t w_div = 0;  // divisions of the wavefront's common-case steps (scalar)
    const uint32_t idle_limit = a.idle_limit;

    // idle lanes take buffered dividing roots, in lane order
    auto hand_out = [&](uint64_t idle, uint32_t n_idle) {
        const uint32_t rank = lane_rank(idle);
        const uint32_t avail = rn - rpos;
        if (!L.active && rank < avail) {
            const QueueEntry &e = ent[rpos + rank];
            L.cell = e.cell;
            L.s = e.s0;
            L.mean = e.mean;
            L.sd = e.sd;
            L.node = (N)1;
            L.k = 0u;
            L.pend = (N)0;
            L.redo = 0u;
            L.kcap = e.kcap;
            L.tb_lds = e.tb_lds;
            L.rowtf = e.rowtf;
            L.active = true;
        }
        rpos = uni(rpos + min(n_idle, avail));
    };

    for (;;) {
        const uint64_t idle = __ballot(!L.active);
        const uint32_t n_idle = uni((uint32_t)__popcll(idle));
        // ======== refill once more than idle_limit lanes are idle ========
        if (n_idle > idle_limit) {
            // ---- root step: the buffer is empty ----
            if (rpos >= rn && !roots_done) {
                // claim the segment's next root step
                uint32_t step = 0;
                if (lane == 0)
                    step = atomicAdd(cursor, 1u);
                const uint64_t c_off = (uint64_t)uni(__shfl(step, 0)) * kWave;
                if (c_off >= seg_cells)
                    roots_done = 1;
                if (!roots_done) {
                    const uint64_t c_cur = seg_begin + c_off;
                    const uint32_t n_valid = uni((uint32_t)min<uint64_t>(kWave, seg_cells - c_off));
                    const uint64_t c = c_cur + lane;
                    const bool valid = lane < n_valid;
                    // rows of the step's cells (cell ids < 2^32): move rb to the
                    // row of c_cur, then count the boundaries inside the step
                    const uint32_t c32 = (uint32_t)c_cur;
                    for (uint64_t le = __ballot(bnd <= c32); le; le = __ballot(bnd <= c32)) {
                        rb = uni(rb + (uint32_t)__popcll(le));
                        load_rows();
                    }
                    const uint32_t nb = uni((uint32_t)__popcll(__ballot((uint64_t)bnd < c_cur + n_valid)));
                    uint32_t rrel = 0;  // boundaries at or below this lane's cell
                    for (uint32_t j = 0; j < nb; ++j)
                        rrel += lane >= (uint32_t)__builtin_amdgcn_readlane((int)bnd, (int)j) - c32 ? 1u : 0u;
                    const uint32_t row = rb + rrel;
                    const uint32_t info = nb ? (uint32_t)__shfl(rinfo, (int)rrel)
                                             : (uint32_t)__builtin_amdgcn_readfirstlane((int)rinfo);
                    const uint32_t kc = info & 0xFFu;
                    const bool ge_phi = (info >> 8) & 1u;
                    // one block per initial cell: type uniform (word 0), phase
                    // (word 1) and the first timer's Box-Muller pair (words 2, 3)
                    const Words w = dev::draw_block(seed, c - S.cell_base, 0, 0);
                    const double ut = dev::uniform_co_hi(w.w0);
                    const double U = dev::uniform_oc_hi(w.w1);
                    // first type with ut < cumulative proportion (cell.cu:90-101):
                    // scanning from the highest index down, the last hit is the
                    // first; past the last proportion, the last type
                    uint32_t jt = T - 1;
                    if (T > 9) {
                        for (uint32_t k = T - 2; k >= 8; --k)
                            jt = ut < t_cum[k] ? k : jt;
                    }
    #pragma unroll
                    for (int k = 7; k >= 0; --k)
                        jt = ut < cum8[k] ? (uint32_t)k : jt;
                    const double2 msd = t_msd[jt];
                    const double m = msd.x;
                    const double sdv = msd.y;
                    const bool quiescent = m < 0.0;
                    // first timer (cell.cu:106-122): two candidates from the root
                    // block, then node 1's redraw stream
                    // (the second candidate only where the first is <= 0: its
                    // sine is computed there alone)
                    double z0, z1;
                    dev::normal_pair<true>(Words{w.w2, 0u, w.w3, 0u}, z0, z1, K, tb);
                    const double c0 = fma(z0, sdv, m);
                    const bool live = valid && !quiescent;
                    double tau0 = c0;
                    if (__builtin_expect(__ballot(live && !(c0 > 0.0)) != 0, 0)) {
                        if (live && !(c0 > 0.0)) {
                            ++n.rej;
                            const double c1 = fma(z1, sdv, m);
                            tau0 = c1;
                        }
                        if (live && !(tau0 > 0.0)) {
                            // rare: node 1's redraw stream from attempt 1
                            ++n.rej;
                            tau0 = m;
                            for (uint32_t att = 1; att < 65536u; ++att) {
                                const Words wr = dev::draw_block(seed, c - S.cell_base, 1, att);
                                double y0, y1;
                                dev::normal_pair(wr, y0, y1, K, tb);
                                const double d0 = fma(y0, sdv, m);
                                if (d0 > 0.0) { tau0 = d0; break; }
                                ++n.rej;
                                const double d1 = fma(y1, sdv, m);
                                if (d1 > 0.0) { tau0 = d1; break; }
                                ++n.rej;
                            }
                        }
                    }
                    const double t0 = tau0 * U;
                    const double s0 = t0 + tau0;
                    // quiescent or out of time: tallied if its value is in the
                    // output bin set; in time with f/2 <= phi: dropped; else it
                    // divides
                    const bool record = valid && (quiescent || s0 > t_max);
                    const bool rec_ok = record && ge_phi;
                    const bool divides = valid && !record && kc != 0;
                    n.cells += valid ? 1u : 0u;
                    n.lost += record && !ge_phi ? 1u : 0u;
                    n.pool += divides ? 1u : 0u;
                    // generation-0 tallies: the window, else one device atomic
                    // per distinct (row, type) of the step
                    const uint32_t tf = t_file[jt];
                    const uint32_t woff = row - row_lo;
                    const bool in_win = woff < a.win_rows;
                    if (rec_ok && in_win) {
                        atomicAdd(&win[woff * kdim * T + tf], 1u);
                    }
                    uint64_t pend = __ballot(rec_ok && !in_win);
                    while (pend) {
                        const uint32_t leader = (uint32_t)__builtin_ctzll(pend);
                        const uint32_t row_l = uni(__shfl(row, (int)leader));
                        const uint32_t tf_l = uni(__shfl(tf, (int)leader));
                        const uint64_t same = __ballot(rec_ok && !in_win && row == row_l && tf == tf_l);
                        if (lane == leader)
                            atomicAdd(&a.tally[S.tally_base + (uint64_t)(row_l - S.row_base) * kdim * T + tf_l],
                                      (unsigned long long)__popcll(same));
                        pend &= ~same;
                    }
                    // dividing cells: buffered for the hand-outs
                    const uint64_t dmask = __ballot(divides);
                    if (divides) {
                        QueueEntry &e = ent[lane_rank(dmask)];
                        e.s0 = s0;
                        e.mean = m;
                        e.sd = sdv;
                        e.cell = (uint32_t)(c - S.cell_base);
                        e.tb_lds = in_win ? woff * kdim * T + tf : kNoWindow;
                        e.rowtf = (row - S.row_base) | (tf << 24);
                        e.kcap = kc;
                    }
                    rpos = 0;
                    rn = uni((uint32_t)__popcll(dmask));
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // ---- steal pending daughters inside the wavefront ----
            if (rpos >= rn && roots_done) {
                const uint64_t donors = __ballot(L.active && L.pend != 0);
                const uint32_t nd = uni(min((uint32_t)__popcll(donors), n_idle));
                if (nd) {
                    const uint32_t my_lvl = L.pend ? low_bit(L.pend) : 0u;
                    const uint32_t r = lane_rank(idle);
                    const bool thief = !L.active && r < nd;
                    const uint32_t src = thief ? nth_set_bit(donors, r) : lane;
                    const uint32_t lvl = __shfl(my_lvl, (int)src);
                    const N d_node = __shfl(L.node, (int)src);
                    const uint32_t d_k = __shfl(L.k, (int)src);
                    const uint32_t d_cell = __shfl(L.cell, (int)src);
                    const uint32_t d_kcap = __shfl(L.kcap, (int)src);
                    const uint32_t d_tbl = __shfl(L.tb_lds, (int)src);
                    const uint32_t d_rtf = __shfl(L.rowtf, (int)src);
                    const double d_mean = __shfl(L.mean, (int)src);
                    const double d_sd = __shfl(L.sd, (int)src);
                    if (L.active && L.pend && lane_rank(donors) < nd)
                        L.pend &= ~((N)1 << my_lvl);
                    if (thief) {
                        L.s = stack[(size_t)(lvl - 1) * bdim + wave * kWave + src];
                        L.node = (d_node >> (d_k - lvl)) | (N)1;
                        L.k = lvl;
                        L.cell = d_cell;
                        L.kcap = d_kcap;
                        L.tb_lds = d_tbl;
                        L.rowtf = d_rtf;
                        L.mean = d_mean;
                        L.sd = d_sd;
                        L.pend = 0;
                        L.redo = 0;
                        L.active = true;
                    }
                }
            }

            if (rpos >= rn && __ballot(L.active) == 0) {
                if (roots_done)
                    break;
                continue;
            }
        }
        // ---- idle lanes take buffered roots ----
        if (rpos < rn) {
            const uint64_t idle2 = __ballot(!L.active);
            hand_out(idle2, uni((uint32_t)__popcll(idle2)));
        }

        // ======== division step ========
        // Straight-line code: every outcome is a select.  The step's flags
        // are lane masks, so their logic runs on the scalar unit beside the
        // vector work (the vector unit is the bound: 4.9 VALU instructions
        // per division against 1.1 scalar).  Idle lanes run the step too
        // with their results discarded.
        {
            // One Philox block + Box-Muller pair per lane and step: either the
            // pair block of a new division (timers of both daughters) or one
            // block of a daughter's truncated-normal redraw stream
            // (cell.cu:106-122); a lane with a redraw pending does not advance
            // its tree in that step.
            const uint32_t act = L.active ? 1u : 0u;
            // the level a pop at the end of this step reads: a lane pops
            // only when the step pushes nothing, so it is the deepest
            // pending level of the step's start; reading it here overlaps
            // the LDS round trip with the division step
            const uint32_t lvl = top_bit(L.pend | (N)2);  // 1 when nothing is pending (level bits start at 1)
            const double sp = *(const double *)(stk_pop + __umul24(lvl, stride));
            double tl, tr;
            bool cmp;  // division complete this step
            if (__builtin_expect(__ballot(L.redo != 0) == 0, 1)) {
                // no redraw pending in the wavefront (the common case): every
                // busy lane starts a new division with its pair block; every
                // lane's redo is 0 and its attempt number 1 (attempts restart
                // at 1 whenever a redraw ends)
                const Words w = dev::draw_block(seed, (uint64_t)L.cell, L.node, 0u);
                double z0, z1;
                dev::normal_pair(w, z0, z1, K, tb);
                tl = fma(z0, L.sd, L.mean);
                tr = fma(z1, L.sd, L.mean);
                const bool ok = tl > 0.0 && tr > 0.0;
                cmp = L.active && ok;
                w_div += (uint32_t)__popcll(__ballot(L.active));
                if (__builtin_expect(__ballot(L.active && !ok) != 0, 0)) {
                    // a timer <= 0: that daughter continues in its redraw stream
                    const uint32_t r0 = tl > 0.0 ? 0u : 1u;
                    const uint32_t r1 = tr > 0.0 ? 0u : 1u;
                    L.redo = act ? r0 | (r1 << 1) : 0u;
                    n.rej += act * (r0 + r1);
                }
            } else {
                const uint32_t fresh = L.redo == 0 ? 1u : 0u;
                const uint32_t rright = (L.redo & 1u) ? 0u : 1u;   // redraw the right daughter?
                const N bnode = fresh ? L.node : (L.node << 1) | (N)rright;
                const Words w = dev::draw_block(seed, (uint64_t)L.cell, bnode, fresh ? 0u : L.att);
                double z0, z1;
                dev::normal_pair(w, z0, z1, K, tb);
                const double c0 = fma(z0, L.sd, L.mean);
                const double c1 = fma(z1, L.sd, L.mean);
                const uint32_t r0 = c0 > 0.0 ? 0u : 1u;
                const uint32_t r1 = c1 > 0.0 ? 0u : 1u;
                // redraw: first candidate > 0 of this block; after 65535 blocks the mean
                const uint32_t got = (r0 & r1) ^ 1u;
                const uint32_t give_up = (got ^ 1u) & (L.att >= 65535u ? 1u : 0u);
                const double v = give_up ? L.mean : (r0 ? c1 : c0);
                const uint32_t done = got | give_up;
                const uint32_t rbit = rright ? 2u : 1u;
                tl = fresh ? c0 : ((done & (rright ^ 1u)) ? v : L.tl);
                tr = fresh ? c1 : ((done & rright) ? v : L.tr);
                const uint32_t redo = fresh ? (r0 | (r1 << 1)) : (done ? L.redo & ~rbit : L.redo);
                n.div += act & fresh;
                n.rej += act * (fresh ? r0 + r1 : r0 + (r0 & r1));
                L.att = fresh | done ? 1u : L.att + 1u;
                L.redo = act ? redo : 0u;
                cmp = L.active && redo == 0;
            }
            L.tl = tl;
            L.tr = tr;

            // daughters (proliferation.cu:317-381): out of time -> tallied,
            // f/2 <= phi -> dropped, else divides later.  The flags below are
            // lane masks (scalar registers), so their logic runs on the
            // scalar unit.
            const double sl = L.s + tl;
            const double sr = L.s + tr;
            const uint32_t k1 = L.k + 1;
            const bool rec_l = sl > t_max;
            const bool rec_r = sr > t_max;
            const bool can = k1 < L.kcap;
            const bool div_l = !rec_l && can;
            const bool div_r = !rec_r && can;
            const uint32_t nrec = cmp ? (uint32_t)rec_l + (uint32_t)rec_r : 0u;
            const bool in_win = L.tb_lds != kNoWindow;
            // lanes without a completed division add 0 to the spare slot win[win_len]
            atomicAdd(&win[(cmp && in_win) ? L.tb_lds + __umul24(k1, T) : win_len], nrec);
            if (__builtin_expect(__ballot(!in_win && nrec != 0) != 0, 0)) {
                if (!in_win && nrec != 0)
                    atomicAdd(&a.tally[S.tally_base + (uint64_t)(L.rowtf & 0xFFFFFFu) * kdim * T +
                                       (L.rowtf >> 24) + (uint64_t)k1 * T],
                              (unsigned long long)nrec);
            }
            // right daughter's completion time, at level k1; level k1 holds
            // no pending entry of an active lane, and idle lanes have none at
            // all (their L.k is at most 1 or a level they popped, below the
            // stack's depth), so the store is harmless when it is not pushed
            *(double *)(stk_push + __umul24(L.k, stride)) = sr;
            const bool go_l = cmp && div_l;
            const bool go_r = cmp && !div_l && div_r;
            const bool pop = cmp && !div_l && !div_r;
            // (k1 stays below the width of N for a lane that pushes; the
            // mask keeps the shift defined for the others)
            const N pend2 = L.pend | ((N)(go_l && div_r) << (k1 & (sizeof(N) * 8 - 1)));
            const bool has = pend2 != 0;
            // single-level selects only (nested ones turn into branches)
            const bool down = go_l || go_r;
            const N child = (L.node << 1) | (N)go_r;
            const uint32_t sh = pop ? ((L.k - lvl) & (sizeof(N) * 8 - 1)) : 0u;
            const N upn = (L.node >> sh) | (N)pop;  // pending right daughter
            const double s_child = go_l ? sl : sr;
            const double s_up = pop ? sp : L.s;
            const uint32_t k_up = pop ? lvl : L.k;
            const N clear = (N)pop << lvl;
            L.node = down ? child : upn;
            L.s = down ? s_child : s_up;
            L.k = down ? k1 : k_up;
            L.pend = pend2 & ~clear;
            L.active = L.active && !(pop && !has);
        }
    }

    n.div += lane == 0 ? w_div : 0u;
    flush_counts(n, a.counters + (size_t)set * kCounterCopies * kNumCounters, lane, red);
    const uint64_t gbase = S.tally_base + (uint64_t)(row_lo - S.row_base) * kdim * T;
    for (uint32_t i = tid; i < win_len; i += bdim) {
        const uint32_t c = win[i];
        if (c)
            atomicAdd(&a.tally[gbase + i], (unsigned long long)c);
    }
}

// ----------------------------------------------------------------------
// The filter.  A run's outputs are whole numbers, and the times enter them
// only through two tests: "timer > 0" and "completion time > t_max".  The
// filtered kernel evaluates both from single-precision times whose distance
// from the 64-bit times is bounded, accepts a test when the value is further
// from the threshold than the bound, and otherwise evaluates the cell's times
// again in 64 bits along its path from the root (exact_times: the same
// operations in the same order as the 64-bit kernel), so every test comes out
// as the 64-bit kernel's and the outputs are the same bit for bit.
//
// Why: the 64-bit Box-Muller pair is 87 of a division step's 180 vector
// instructions at 4 cycles each; the hardware's log2, sqrt, sin and cos take
// 8 cycles each and single-precision multiplies and adds 2 to 3.  Five-type
// histogram, 1024 bins: 0.219 -> 0.143 ms per run at 1e7 cells, 2.05 -> 1.10
// ms at 1e8 (2.58e8 divisions: 1.26e11 -> 2.35e11 per second; vector
// instructions per division 4.56 -> 2.70).
//
// The bound.  For a block whose first word w0 lies in [2^16, 2^32 - 2^16)
// (pair_sure; the others, 1 in 2^15, are evaluated in 64 bits)
// normal_pair_f32 is within 5.42e-6 of the 64-bit pair.  Measured on gfx950
// over all 2^32 values of each word (pair_bounds_kernel repeats it): the
// radius is off by at most 5.42e-6 (next to u1 = 1, where it is below 0.01)
// and 3.64e-6 for u1 <= 1/2, sine and cosine by 2.7e-7 (times a radius of at
// most 4.71).  kPairErr allows 7e-6.  A timer fma(z, sd, mean) adds the
// rounding of sd, mean and itself: at most 2^-23 (|mean| + 8.6 |sd|);
// a completion time adds 2^-24 t_max per addition (times are kept relative to
// t_max, so a value near the threshold is small, and no partial sum of a path
// exceeds t_max) and 3.5 of those for t_max and the root's phase.  After k
// levels below the root that is (k + 2) e + (k + 3.5) 2^-24 t_max with e =
// 6.7e-6 |sd| + 1.2e-7 |mean|; filter_type_err and filter_cell_err round it up, with the
// row's cap for k.
// ----------------------------------------------------------------------
constexpr uint32_t kPairLow = 1u << 16;

__device__ __forceinline__ bool pair_sure(uint32_t w0) { return w0 - kPairLow < 0u - 2u * kPairLow; }

__device__ __forceinline__ float radius_f32(uint32_t w0)
{
    const float u1 = (float)w0 * 0x1p-32f;
    return __builtin_amdgcn_sqrtf(__builtin_amdgcn_logf(u1) * -1.3862943611198906f);  // -2 ln 2
}

__device__ __forceinline__ void turn_f32(uint32_t w2, float &cs, float &sn)
{
    const float turn = (float)w2 * 0x1p-32f;
    cs = __builtin_amdgcn_cosf(turn);
    sn = __builtin_amdgcn_sinf(turn);
}

__device__ __forceinline__ void normal_pair_f32(uint32_t w0, uint32_t w2, float &z0, float &z1)
{
    const float rho = radius_f32(w0);
    float cs, sn;
    turn_f32(w2, cs, sn);
    z0 = rho * cs;
    z1 = rho * sn;
}

// Smaller of two magnitudes.
__device__ __forceinline__ float min_abs(float x, float y) { return fminf(fabsf(x), fabsf(y)); }

// Completion times in 64 bits, minus t_max and rounded to single precision
// (which keeps the sign of the 64-bit comparison: the difference of two
// doubles of magnitude above 1e-20 is 0 or above 1e-36): of the division of
// `node` (its daughters' l and r), or with node 0 of the root's first
// division (l).  The path from the root is walked again; rej counts the
// candidates refused for the returned times.  Needed
// about once in a thousand steps.
struct ExactTimes {
    float l, r;
    uint32_t rej;
};

__device__ __forceinline__ ExactTimes exact_times(uint64_t seed, uint32_t cell, uint64_t node, double mean, double sd,
                                                  double t_max)
{
    const dev::Tables tb = dev::global_tables();
    constexpr dev::Coeffs K = dev::coeffs();
    const uint32_t levels = node ? 64u - (uint32_t)__builtin_clzll(node) : 0u;  // divisions on the path, this one included
    double s = 0.0, last_l = 0.0;
    uint32_t rej = 0;
    // step 0: the root's first timer from block (cell, 0, 0); step i >= 1: the
    // pair of the path's i-th node, of which the path takes one timer and the
    // last node both
    for (uint32_t step = 0; step <= levels; ++step) {
        const uint64_t at = step ? node >> (levels - step) : 0ull;
        Words w = dev::draw_block(seed, cell, at, 0u);
        const double U = dev::uniform_oc_hi(w.w1);
        if (step == 0)
            w = Words{w.w2, 0u, w.w3, 0u};
        double z0, z1;
        dev::normal_pair(w, z0, z1, K, tb);
        rej = 0;
        const bool both = step == levels && step != 0;
        for (uint32_t side = both ? 0u : step ? (uint32_t)(node >> (levels - step - 1)) & 1u : 0u; side < 2; ++side) {
            double tau = fma(side ? z1 : z0, sd, mean);
            if (!(tau > 0.0)) {
                // truncated normal (cell.cu:106-122): the root's second
                // candidate, then the node's redraw stream, the mean after
                // 65535 blocks
                ++rej;
                uint32_t att = 1;
                double y0 = z0, y1 = z1;
                bool pair = step == 0;  // y1 still to be tried
                for (;;) {
                    if (pair) {
                        tau = fma(y1, sd, mean);
                        if (tau > 0.0)
                            break;
                        ++rej;
                    }
                    if (att > 65535u) {
                        tau = mean;
                        break;
                    }
                    dev::normal_pair(dev::draw_block(seed, cell, step ? at << 1 | side : 1ull, att), y0, y1, K, tb);
                    ++att;
                    tau = fma(y0, sd, mean);
                    if (tau > 0.0)
                        break;
                    ++rej;
                    pair = true;
                }
            }
            if (both && side == 0) {
                last_l = s + tau;
                continue;
            }
            s = step ? s + tau : tau * U + tau;
            break;
        }
    }
    return levels ? ExactTimes{(float)(last_l - t_max), (float)(s - t_max), rej}
                  : ExactTimes{(float)(s - t_max), 0.0f, rej};
}

// ======================================================================
// sim_filter_kernel: the same run as sim_kernel (segments, claims, root
// steps, hand-outs and division steps as there), with the two tests on times
// filtered as described above; it runs every plan whose times the bound
// covers (the host's filter_covers) and which it does not slow down
// (filter_pays).  What bounds it is the vector unit's issue rate (1.04
// instructions per CU and clock at 1e8 cells; most take 4 cycles of a SIMD,
// additions, logic, moves and single-precision arithmetic on vector registers
// 2 to 3) and, with fewer instructions per step than sim_kernel, the latency
// of a wavefront's own instruction stream: 6 wavefronts per SIMD instead of 4
// gave 1.24 -> 1.09 ms, which holds it to 80 registers (the 64-bit evaluation
// spills a few, in its own branch only).  The tree logic is arranged for few
// instructions and few values carried round the loop:
//  * a set's rows come in order of decreasing cost (the host's order_rows), so
//    the last trees of a segment, and of the run, are its shallowest: 0.143 ->
//    0.136 ms at 1e7 cells.
//  * a lane's pending right daughters are a mask relative to its level (bit i:
//    level k - i), with one more bit for level 0 that no daughter uses.  Going
//    down shifts the mask up by one; "the left daughter does not divide" takes
//    the lowest set bit, whichever of the right daughter (bit 0) or an older
//    level it is, and the same shift takes node and level there.  Taking the
//    level-0 bit leaves the mask empty: the lane is idle exactly when its mask
//    is 0.
//  * idle lanes, and lanes with a redraw pending, are masked off (the exec
//    mask, scalar work) instead of having every result selected.
//  * the state of a redraw (1 in 10 steps has one) waits in LDS: in registers
//    it cost some 20 copies per step at the loop's branches.
//  * event counts are scalar; a step looks at tallies outside the window only
//    where the workgroup's rows exceed it.
// LDS: type tables ({mean, sd, error bound, file index}: 16 bytes [T]; last
// drawn word + 1: u32 [T]) | row tables when they fit | counter sums u32 [8] |
// root step cursor u32 [4] | buffered entries, per wavefront [64] | redraws,
// per lane | window tally u32 [win_rows * kdim * T] | stacks float, per wavefront
// [stack_levels][64]
// ======================================================================
struct alignas(16) FilterType {
    float mean, sd;
    float err;      // error bound of a completion time per level
    uint32_t file;  // file index
};

// per wavefront: buffered entries, lanes' redraws
__host__ __device__ constexpr uint32_t filter_wave_bytes()
{
    return kWave * (uint32_t)(sizeof(FilterEntry) + 16);
}

__host__ __device__ constexpr size_t filter_type_bytes(uint32_t n_types)
{
    return (size_t)n_types * sizeof(FilterType) + ((size_t)n_types * 4 + 15) / 16 * 16;
}

// A lane of sim_filter_kernel.
template <typename N>
struct FilterLane {
    N node, pend;       // heap index; pending levels relative to k, 0: the lane is idle
    float s;            // completion time of the node's division minus t_max
    float mean, sd;
    float err;          // bound of |s - its 64-bit value| at any level of the tree
    uint32_t cell;      // initial cell, relative to its set
    uint32_t tb;        // LDS address of the window entry (row, generation 0, type), or kNoWindow
    uint32_t rowt;      // row in the set's file order | sorted type << 24
    uint32_t k, kcap;
};

// A division with a redraw pending, kept in LDS (rarely used: in registers it
// would be copied at every branch of the loop).
struct alignas(16) FilterRedo {
    float tl, tr;       // timers so far
    uint32_t redo;      // bit 0 / bit 1: left / right timer still to redraw; attempt number << 2
    uint32_t rej;       // refused candidates
};

typedef __attribute__((address_space(3))) unsigned int LdsWord;

// LDS address of an entry of the dynamic block, and an add to such an entry.
__device__ __forceinline__ uint32_t lds_address(void *p) { return (uint32_t)(uintptr_t)(LdsWord *)p; }
__device__ __forceinline__ void lds_add(uint32_t at, uint32_t v)
{
    __hip_atomic_fetch_add((LdsWord *)(uintptr_t)at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <bool RowsLds, typename N, bool GStack>
__global__ void __launch_bounds__(kFilterThreads, 6) sim_filter_kernel(RunArgs a)
{
    extern __shared__ __align__(16) unsigned char lds[];
    const uint32_t tid = threadIdx.x;
    const uint32_t bdim = blockDim.x;
    const uint32_t lane = tid & (kWave - 1);
    const uint32_t wave = uni(tid / kWave);
    const uint32_t n_waves = bdim / kWave;
    const uint32_t seg0 = blockIdx.x;
    const uint32_t set = a.n_sets > 1 ? a.seg_set[seg0] : 0u;
    const SetInfo S = a.sets[set];
    const uint64_t seed = a.n_sets > 1 ? a.set_seed[set] : a.seed;
    const double t_max = S.t_max;
    const float t_max32 = (float)t_max;
    const uint32_t T = S.n_types;
    const uint32_t kdim = S.kdim;
    const uint32_t T4 = T * 4;
    const uint32_t row_bytes = kdim * T4;
    const uint32_t win_len = a.win_rows * kdim * T;
    const uint32_t lds_rows = RowsLds ? a.n_rows : 0u;
    FilterType *types = (FilterType *)lds;
    uint32_t *lims = (uint32_t *)(types + T);
    uint32_t *r_start = (uint32_t *)(lds + filter_type_bytes(T));
    uint32_t *r_info = r_start + lds_rows + 1;
    uint32_t *red = (uint32_t *)((unsigned char *)r_start + (RowsLds ? ((size_t)(2 * lds_rows + 1) * 4 + 15) / 16 * 16 : 0));
    uint32_t *cursor = red + kNumCounters;  // root steps of the segment claimed so far
    FilterEntry *ent = (FilterEntry *)((unsigned char *)red + kSimSharedBytes) + wave * kWave;
    FilterRedo *redo = (FilterRedo *)((unsigned char *)red + kSimSharedBytes + n_waves * kWave * sizeof(FilterEntry)) + tid;
    const uint32_t win_off = (uint32_t)((unsigned char *)red - lds) + kSimSharedBytes + n_waves * filter_wave_bytes();
    const uint32_t win_base = lds_address(lds + win_off);
    unsigned int *win = (unsigned int *)(lds + win_off);
    constexpr uint32_t kStride = kWave * (uint32_t)sizeof(float);  // bytes between levels
    const uint32_t levels = a.stack_levels;
    // level l (1-based) at stack + l * kWave; "level 0" is what lies before,
    // never stored to
    float *stack = (GStack ? (float *)a.gstack + (size_t)seg0 * levels * bdim
                           : (float *)(lds + win_off + ((size_t)win_len * 4 + 15) / 16 * 16)) +
                   (size_t)wave * levels * kWave - kWave;
    unsigned char *const stk = (unsigned char *)(stack + lane);

    const uint64_t seg_begin = uni64(a.seg_begin[seg0]);
    const uint64_t seg_end = uni64(a.seg_end[seg0]);
    const uint64_t seg_cells = seg_end - seg_begin;
    const uint32_t row_lo = uni(a.seg_row[seg0]);  // first row of the segment and of the tally window
    const uint32_t cell0 = (uint32_t)(seg_begin - S.cell_base);
    for (uint32_t i = tid; i < T; i += bdim) {
        const double cum = a.type_cum[S.type_base + i], m = a.type_mean[S.type_base + i], sd = a.type_sd[S.type_base + i];
        // the sign of a quiescent type's mean from the 64-bit value: one above
        // -2^-150 rounds to -0 in single precision
        types[i] = FilterType{m < 0.0 ? -1.0f : (float)m, (float)sd, (float)filter_type_err(m, sd, t_max), a.type_file[S.type_base + i]};
        // w 2^-32 < cum for a whole number w: w < ceil(cum 2^32); a limit of
        // 2^32 or more is stored as 2^32 - 1, and a drawn 2^32 - 1 looked at
        // again (the sums are > 0: the largest proportion comes first and the
        // last sum is 1)
        lims[i] = (uint32_t)fmin(ceil(cum * 0x1p32), 0x1p32 - 1.0);
    }
    for (uint32_t i = tid; i <= lds_rows && RowsLds; i += bdim)
        r_start[i] = a.row_start[i];
    for (uint32_t i = tid; i < lds_rows; i += bdim)
        r_info[i] = a.row_info[i];
    for (uint32_t i = tid; i < win_len; i += bdim)
        win[i] = 0u;
    if (tid < kNumCounters + 1)
        red[tid] = 0u;  // counter sums and the root step cursor
    __syncthreads();

    // the row tables' address space is known at compile time (no flat loads)
    const uint32_t *rs = RowsLds ? r_start : a.row_start;
    const uint32_t *ri = RowsLds ? r_info : a.row_info;
    // every row of the segment has its window
    const bool all_in = uni(row_lo + a.win_rows >= a.n_rows || (uint64_t)rs[row_lo + a.win_rows] >= seg_end ? 1u : 0u) != 0;

    uint32_t rpos = 0, rn = 0;      // buffered dividing roots: entries [rpos, rn) of ent
    uint32_t roots_done = 0;
    // limits of the type search (0: never met, for the last type and beyond)
    uint32_t lim8[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k)
        lim8[k] = uni(k + 1 < T ? lims[k] : 0u);
    // Row boundaries of the wavefront's root steps (as in sim_kernel)
    uint32_t rb = row_lo, bnd = 0, rinfo = 0, rcell = 0;
    auto load_rows = [&]() {
        const uint32_t r1 = rb + 1 + lane;
        bnd = r1 <= a.n_rows ? rs[r1] : 0xFFFFFFFFu;
        rinfo = rb + lane < a.n_rows ? ri[rb + lane] : 0u;
        rcell = rb + lane < a.n_rows ? a.row_cell[rb + lane] : 0u;
    };
    load_rows();

    FilterLane<N> L{};
    uint64_t redoing = 0;                                     // lanes with a redraw pending
    uint32_t w_div = 0, w_lost = 0, w_cells = 0, w_pool = 0;  // event counts, scalar
    unsigned int *n_rej = &red[kRedRejected];                 // refused candidates: rare, counted in LDS
    const uint32_t idle_limit = a.idle_limit;

    for (;;) {
        const uint64_t idle = __ballot(L.pend == 0);
        const uint32_t n_idle = uni((uint32_t)__popcll(idle));
        // ======== refill once more than idle_limit lanes are idle ========
        if (n_idle > idle_limit) {
            // ---- root step: the buffer is empty ----
            if (rpos >= rn && !roots_done) {
                uint32_t step = 0;
                if (lane == 0)
                    step = atomicAdd(cursor, 1u);
                const uint64_t c_off = (uint64_t)uni(step) * kWave;
                if (c_off >= seg_cells)
                    roots_done = 1;
                if (!roots_done) {
                    const uint64_t c_cur = seg_begin + c_off;
                    const uint32_t n_valid = uni((uint32_t)min<uint64_t>(kWave, seg_cells - c_off));
                    const bool valid = lane < n_valid;
                    // rows of the step's cells (cell ids < 2^32): move rb to the
                    // row of c_cur, then count the boundaries inside the step
                    const uint32_t c32 = (uint32_t)c_cur;
                    for (uint64_t le = __ballot(bnd <= c32); le; le = __ballot(bnd <= c32)) {
                        rb = uni(rb + (uint32_t)__popcll(le));
                        load_rows();
                    }
                    const uint32_t nb = uni((uint32_t)__popcll(__ballot((uint64_t)bnd < c_cur + n_valid)));
                    uint32_t rrel = 0;  // boundaries at or below this lane's cell
                    uint32_t info = uni(rinfo), dcell = uni(rcell);
                    if (nb) {
                        for (uint32_t j = 0; j < nb; ++j)
                            rrel += lane >= (uint32_t)__builtin_amdgcn_readlane((int)bnd, (int)j) - c32 ? 1u : 0u;
                        info = (uint32_t)__shfl(rinfo, (int)rrel);
                        dcell = (uint32_t)__shfl(rcell, (int)rrel);
                    }
                    const uint32_t row = rb + rrel, file_row = info >> 7;
                    const uint32_t kc = info & 63u;
                    const bool ge_phi = (info >> 6) & 1u;
                    const uint32_t cell = cell0 + (uint32_t)c_off + lane + dcell;
                    // one block per initial cell: type uniform (word 0), phase
                    // (word 1) and the first timer's Box-Muller pair (words 2, 3)
                    const Words w = dev::draw_block(seed, cell, 0, 0);
                    // first type with w 2^-32 < cumulative proportion
                    // (cell.cu:90-101): scanning from the highest index down, the
                    // last hit is the first; past the last proportion, the last type
                    uint32_t jt = T - 1;
                    if (T > 9) {
                        for (uint32_t k = T - 2; k >= 8; --k)
                            jt = w.w0 < lims[k] ? k : jt;
                    }
                    if (T > 5) {
#pragma unroll
                        for (int k = 7; k >= 4; --k)
                            jt = w.w0 < lim8[k] ? (uint32_t)k : jt;
                    }
#pragma unroll
                    for (int k = 3; k >= 0; --k)
                        jt = w.w0 < lim8[k] ? (uint32_t)k : jt;
                    if (__builtin_expect(__ballot(w.w0 == 0xFFFFFFFFu) != 0, 0)) {
                        if (w.w0 == 0xFFFFFFFFu)
                            for (jt = 0; jt + 1 < T && !(dev::uniform_co_hi(w.w0) < a.type_cum[S.type_base + jt]); ++jt) {
                            }
                    }
                    const FilterType ty = types[jt];
                    const float err = filter_cell_err(kc, ty.err);
                    const bool quiescent = ty.mean < 0.0f;
                    const bool live = valid && !quiescent;
                    // first timer (cell.cu:106-122): two candidates from the root
                    // block, then node 1's redraw stream (in 64 bits)
                    float z0, z1;
                    normal_pair_f32(w.w2, w.w3, z0, z1);
                    const float u1 = fmaf((float)w.w1, 0x1p-32f, 1.0f);
                    const float tau0 = fmaf(z0, ty.sd, ty.mean);
                    float s0 = fmaf(tau0, u1, -t_max32);
                    const bool sure = (int)(min_abs(tau0, s0) > err) & (int)(tau0 > 0.0f) & (int)pair_sure(w.w2);
                    if (__builtin_expect(__ballot(live && !sure) != 0, 0)) {
                        if (live && !sure) {
                            // the second candidate where the first is surely refused
                            const float tau1 = fmaf(z1, ty.sd, ty.mean);
                            s0 = fmaf(tau1, u1, -t_max32);
                            uint32_t rej = 1;
                            if (!(pair_sure(w.w2) && tau0 < -err && tau1 > err && fabsf(s0) > err)) {
                                const ExactTimes e = exact_times(seed, cell, 0, a.type_mean[S.type_base + jt],
                                                                 a.type_sd[S.type_base + jt], t_max);
                                s0 = e.l;
                                rej = e.rej;
                            }
                            atomicAdd(n_rej, rej);
                        }
                    }
                    // quiescent or out of time: tallied if its value is in the
                    // output bin set; in time with f/2 <= phi: dropped; else it
                    // divides
                    const bool record = valid && (quiescent || s0 > 0.0f);
                    const bool rec_ok = record && ge_phi;
                    const bool divides = valid && !record && kc != 0;
                    const uint64_t dmask = __ballot(divides);
                    w_cells += n_valid;
                    w_lost += (uint32_t)__popcll(__ballot(record && !ge_phi));
                    w_pool += (uint32_t)__popcll(dmask);
                    // generation-0 tallies: the window, else one device atomic
                    // per distinct (row, type) of the step
                    const uint32_t woff = row - row_lo;
                    const bool in_win = all_in || woff < a.win_rows;
                    const uint32_t tb = win_base + __umul24(woff, row_bytes) + ty.file * 4;
                    if (rec_ok && in_win)
                        lds_add(tb, 1u);
                    if (!all_in) {
                        uint64_t pend = __ballot(rec_ok && !in_win);
                        while (pend) {
                            const uint32_t leader = (uint32_t)__builtin_ctzll(pend);
                            const uint32_t row_l = uni(__shfl(file_row, (int)leader));
                            const uint32_t tf_l = uni(__shfl(ty.file, (int)leader));
                            const uint64_t same = __ballot(rec_ok && !in_win && file_row == row_l && ty.file == tf_l);
                            if (lane == leader)
                                atomicAdd(&a.tally[S.tally_base + (uint64_t)row_l * kdim * T + tf_l],
                                          (unsigned long long)__popcll(same));
                            pend &= ~same;
                        }
                    }
                    // dividing cells: buffered for the hand-outs
                    if (divides)
                        ent[lane_rank(dmask)] = FilterEntry{s0, ty.mean, ty.sd, err, cell, in_win ? tb : kNoWindow,
                                                            file_row | (jt << 24), kc};
                    rpos = 0;
                    rn = uni((uint32_t)__popcll(dmask));
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // ---- steal pending daughters inside the wavefront ----
            if (rpos >= rn && roots_done) {
                // a lane's shallowest pending daughter: the highest bit below
                // its level-0 bit k
                const N mine = L.pend & (((N)1 << L.k) - (N)1);
                const uint64_t donors = __ballot(mine != 0);
                const uint32_t nd = uni(min((uint32_t)__popcll(donors), n_idle));
                if (nd) {
                    const uint32_t my_up = mine ? top_bit(mine) : 0u;
                    const uint32_t r = lane_rank(idle);
                    const bool thief = L.pend == 0 && r < nd;
                    const uint32_t src = thief ? nth_set_bit(donors, r) : lane;
                    const uint32_t up = __shfl(my_up, (int)src);
                    const N d_node = __shfl(L.node, (int)src);
                    const uint32_t d_k = __shfl(L.k, (int)src);
                    const uint32_t d_cell = __shfl(L.cell, (int)src);
                    const uint32_t d_kcap = __shfl(L.kcap, (int)src);
                    const uint32_t d_tb = __shfl(L.tb, (int)src);
                    const uint32_t d_rowt = __shfl(L.rowt, (int)src);
                    const float d_mean = __shfl(L.mean, (int)src);
                    const float d_sd = __shfl(L.sd, (int)src);
                    const float d_err = __shfl(L.err, (int)src);
                    if (mine != 0 && lane_rank(donors) < nd)
                        L.pend &= ~((N)1 << my_up);
                    if (thief) {
                        L.k = d_k - up;
                        L.s = stack[L.k * kWave + src];
                        L.node = (d_node >> up) | (N)1;
                        L.pend = (N)1 << L.k;  // its level-0 bit alone
                        L.cell = d_cell;
                        L.kcap = d_kcap;
                        L.tb = d_tb;
                        L.rowt = d_rowt;
                        L.mean = d_mean;
                        L.sd = d_sd;
                        L.err = d_err;
                    }
                }
            }
        }
        // ---- idle lanes take buffered roots, in lane order ----
        if (rpos < rn) {
            const uint64_t idle2 = __ballot(L.pend == 0);
            const uint32_t rank = lane_rank(idle2) + rpos;
            if (L.pend == 0 && rank < rn) {
                const FilterEntry e = ent[rank];
                L.s = e.s0;
                L.mean = e.mean;
                L.sd = e.sd;
                L.err = e.err;
                L.cell = e.cell;
                L.tb = e.tb;
                L.rowt = e.rowt;
                L.kcap = e.kcap;
                L.node = (N)1;
                L.pend = (N)1;
                L.k = 0u;
            }
            rpos = uni(min(rpos + (uint32_t)__popcll(idle2), rn));
        }

        // ======== division step ========
        // One Philox block + Box-Muller pair per busy lane and step: either
        // the pair block of a new division (timers of both daughters) or one
        // block of a daughter's truncated-normal redraw stream
        // (cell.cu:106-122); a lane with a redraw pending does not advance its
        // tree in that step.
        const uint64_t busy = __ballot(L.pend != 0);
        if (busy == 0 && roots_done && rpos >= rn)
            break;
        w_div += uni((uint32_t)__popcll(busy & ~redoing));
        bool again = false;  // a redraw pending after this step
        if (L.pend != 0) {
            // the completion time a pop at the end of this step takes, read
            // here so that the LDS round trip overlaps the division (a lane
            // pops only when the step pushes nothing)
            const uint32_t fl = low_bit(L.pend);
            const float sp = *(const float *)(stk + __umul24(L.k - fl, kStride));
            float sl, sr;
            bool cmp = true;      // division complete this step
            bool unsure = false;  // a test of this step is within its error bound
            if (__builtin_expect(redoing == 0, 1)) {
                // no redraw pending in the wavefront (the common case)
                const Words w = dev::draw_block(seed, (uint64_t)L.cell, L.node, 0u);
                float z0, z1;
                normal_pair_f32(w.w0, w.w2, z0, z1);
                const float tl = fmaf(z0, L.sd, L.mean);
                const float tr = fmaf(z1, L.sd, L.mean);
                sl = L.s + tl;
                sr = L.s + tr;
                const bool fine = (int)(fminf(fminf(tl, tr), min_abs(sl, sr)) > L.err) & (int)pair_sure(w.w0);
                if (__builtin_expect(__ballot(!fine) != 0, 0)) {
                    if (!fine) {
                        // a timer surely < 0: that daughter continues in its
                        // redraw stream; else surely > 0 and surely in or out
                        // of time, or the division is evaluated in 64 bits
                        const uint32_t r0 = tl < 0.0f ? 1u : 0u;
                        const uint32_t r1 = tr < 0.0f ? 1u : 0u;
                        if (pair_sure(w.w0) && min_abs(tl, tr) > L.err && (r0 | r1) != 0u) {
                            *redo = FilterRedo{tl, tr, r0 | (r1 << 1) | 4u, r0 + r1};
                            cmp = false;
                        } else {
                            unsure = true;
                        }
                    }
                }
            } else {
                const bool fresh = ((redoing >> lane) & 1ull) == 0;
                FilterRedo q{0.0f, 0.0f, 4u, 0u};
                if (!fresh)
                    q = *redo;
                const uint32_t att = q.redo >> 2;
                const bool left = (q.redo & 1u) != 0;  // the left timer is drawn again first
                const N bnode = fresh ? L.node : (L.node << 1) | (N)(left ? 0u : 1u);
                const Words w = dev::draw_block(seed, (uint64_t)L.cell, bnode, fresh ? 0u : att);
                float z0, z1;
                normal_pair_f32(w.w0, w.w2, z0, z1);
                const float c0 = fmaf(z0, L.sd, L.mean);
                const float c1 = fmaf(z1, L.sd, L.mean);
                const uint32_t r0 = c0 > 0.0f ? 0u : 1u;
                const uint32_t r1 = c1 > 0.0f ? 0u : 1u;
                if (fresh) {
                    q = FilterRedo{c0, c1, r0 | (r1 << 1) | 4u, r0 + r1};
                } else {
                    // first candidate > 0 of this block; after 65535 blocks the mean
                    q.rej += r0 + (r0 & r1);
                    if ((r0 & r1) == 0u || att >= 65535u) {
                        const float v = r0 == 0u ? c0 : r1 == 0u ? c1 : L.mean;
                        (left ? q.tl : q.tr) = v;
                        q.redo = (q.redo & (left ? 2u : 0u)) | 4u;
                    } else {
                        q.redo += 4u;
                    }
                }
                sl = L.s + q.tl;
                sr = L.s + q.tr;
                cmp = (q.redo & 3u) == 0;
                unsure = !pair_sure(w.w0) || !(min_abs(c0, c1) > L.err) || (cmp && !(min_abs(sl, sr) > L.err));
                // refused candidates are counted when the division completes
                // (exact_times counts a division's anew)
                if (!unsure) {
                    if (cmp && q.rej)
                        atomicAdd(n_rej, q.rej);
                    if (!cmp)
                        *redo = q;
                }
            }
            if (__builtin_expect(__ballot(unsure) != 0, 0)) {
                if (unsure) {
                    const uint32_t jt = L.rowt >> 24;
                    const ExactTimes e = exact_times(seed, L.cell, L.node, a.type_mean[S.type_base + jt],
                                                     a.type_sd[S.type_base + jt], t_max);
                    sl = e.l;
                    sr = e.r;
                    if (e.rej)
                        atomicAdd(n_rej, e.rej);
                    cmp = true;
                }
            }
            again = !cmp;

            if (cmp) {
                // daughters (proliferation.cu:317-381): out of time ->
                // tallied, f/2 <= phi -> dropped, else divides later
                const uint32_t k1 = L.k + 1;
                const bool rec_l = sl > 0.0f;
                const bool rec_r = sr > 0.0f;
                const bool can = k1 < L.kcap;
                const bool div_l = (int)!rec_l & (int)can;
                const bool div_r = (int)!rec_r & (int)can;
                const uint32_t nrec = (uint32_t)rec_l + (uint32_t)rec_r;
                if (all_in) {
                    lds_add(L.tb + __umul24(k1, T4), nrec);
                } else if (L.tb != kNoWindow) {
                    lds_add(L.tb + __umul24(k1, T4), nrec);
                } else if (nrec) {
                    atomicAdd(&a.tally[S.tally_base + (uint64_t)(L.rowt & 0xFFFFFFu) * kdim * T + types[L.rowt >> 24].file +
                                       (uint64_t)k1 * T],
                              (unsigned long long)nrec);
                }
                // right daughter's completion time, at level k1 (which holds
                // no pending entry, so the store is harmless when it is not
                // pushed)
                *(float *)(stk + __umul24(k1, kStride)) = sr;
                // next: the left daughter, else the lowest pending level (the
                // right daughter's if it divides, else fl levels up)
                const N up = (N)(div_l ? 0u : 1u);
                const uint32_t sh = ((int)div_l | (int)div_r) ? 0u : fl + 1u;
                L.node = ((L.node << 1) >> sh) | up;
                L.pend = (((L.pend << 1) | (N)(div_r ? 1u : 0u)) >> sh) & ~up;
                L.k = k1 - sh;
                L.s = div_l ? sl : (div_r ? sr : sp);
            }
        }
        redoing = __ballot(again);
    }

    // places of the first 64 window rows, read ahead of the barrier
    const uint32_t n_win = min(a.win_rows, a.n_rows - row_lo);
    uint32_t place = lane < n_win ? ri[row_lo + lane] >> 7 : 0u;
    Counts n = {0, 0, 0, 0, 0};
    if (lane == 0) {
        n.div = w_div;
        n.lost = w_lost;
        n.cells = w_cells;
        n.pool = w_pool;
    }
    flush_counts(n, a.counters + (size_t)set * kCounterCopies * kNumCounters, lane, red);
    // one wavefront per window row, to the row's place in file order
    const uint32_t row_len = kdim * T;
    for (uint32_t r0 = 0; r0 < n_win; r0 += kWave) {
        if (r0)
            place = r0 + lane < n_win ? ri[row_lo + r0 + lane] >> 7 : 0u;
        for (uint32_t r = r0 + wave; r < min(r0 + kWave, n_win); r += n_waves) {
            unsigned long long *row =
                &a.tally[S.tally_base + (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)place, (int)(r - r0)) * row_len];
            for (uint32_t i = lane; i < row_len; i += kWave) {
                const uint32_t c = win[r * row_len + i];
                if (c)
                    atomicAdd(&row[i], (unsigned long long)c);
            }
        }
    }
}

__global__ void debug_draws_kernel(uint64_t seed, const uint64_t *cell, const uint64_t *node,
                                   const uint32_t *attempt, uint64_t n, uint32_t *words, double *z)
{
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const Words w = dev::draw_block(seed, cell[i], node[i], attempt[i]);
    words[4 * i + 0] = w.w0;
    words[4 * i + 1] = w.w1;
    words[4 * i + 2] = w.w2;
    words[4 * i + 3] = w.w3;
    double z0, z1;
    dev::normal_pair(w, z0, z1, dev::coeffs(), dev::global_tables());
    z[2 * i] = z0;
    z[2 * i + 1] = z1;
}

// The errors behind kPairErr, over all values of a block's words: word 0 with
// the least and the largest word 1 and word 2 with the least and the largest
// word 3 (the 64-bit radius and angle are monotone in them).  First pass
// (pairs 0): sine and cosine; second: the radius, and with the first pass's
// result a candidate: the radius' error, its sine's, and the rounding of their
// product.  out: the radius, the radius where the uniform is at most 1/2, sine
// and cosine, a candidate; as bits of doubles >= 0, which order like integers.
__global__ void pair_bounds_kernel(uint32_t pairs, unsigned long long *out)
{
    const dev::Tables tb = dev::global_tables();
    constexpr dev::Coeffs K = dev::coeffs();
    const double sc_err = __builtin_bit_cast(double, (uint64_t)out[2]);
    double worst[4] = {0.0, 0.0, 0.0, 0.0};
    const uint32_t stride = gridDim.x * blockDim.x, tid = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint64_t w = tid; w < 1ull << 32; w += stride)
        for (uint32_t lo : {0u, 0xFFFFFFFFu}) {
            if (!pairs) {
                float cs, sn;
                turn_f32((uint32_t)w, cs, sn);
                double c64, s64;
                dev::sincos_turns((uint32_t)w, lo, s64, c64, K, tb);
                worst[2] = fmax(worst[2], fmax(fabs(cs - c64), fabs(sn - s64)));
            } else if (pair_sure((uint32_t)w)) {
                const double rho = dev::sqrt_nonneg(-2.0 * dev::log_pos(dev::uniform_oc((uint32_t)w, lo), K, tb));
                const double e = fabs(radius_f32((uint32_t)w) - rho);
                worst[0] = fmax(worst[0], e);
                worst[1] = fmax(worst[1], w < 0x80000000u ? e : 0.0);
                worst[3] = fmax(worst[3], e * (1.0 + sc_err) + rho * sc_err + 0x1p-24 * (rho + e));
            }
        }
    for (int i = 0; i < 4; ++i)
        if (worst[i] > 0.0)
            atomicMax(&out[i], (unsigned long long)__builtin_bit_cast(uint64_t, worst[i]));
}

}  // namespace

hipError_t launch_pair_bounds(unsigned long long *out, hipStream_t st)
{
    hipLaunchKernelGGL(pair_bounds_kernel, dim3(4096), dim3(256), 0, st, 0u, out);
    hipLaunchKernelGGL(pair_bounds_kernel, dim3(4096), dim3(256), 0, st, 1u, out);
    return hipGetLastError();
}

size_t sim_lds_bytes(uint32_t win_rows, uint32_t kdim, uint32_t n_types, uint32_t stack_levels, uint32_t block_size,
                     uint32_t lds_rows, bool filter)
{
    const size_t types = filter ? filter_type_bytes(n_types)
                                : kMathTableBytes + (sizeof(dev::Coeffs) + 15) / 16 * 16 + ((size_t)n_types * 28 + 15) / 16 * 16;
    const size_t rows = lds_rows ? ((size_t)(2 * lds_rows + 1) * 4 + 15) / 16 * 16 : 0;
    const size_t waves = (size_t)(block_size / kWave) * (filter ? filter_wave_bytes() : sim_wave_lds_bytes());
    const size_t win = filter ? ((size_t)win_rows * kdim * n_types * 4 + 15) / 16 * 16
                              : ((size_t)win_rows * kdim * n_types * 4 + 4 + 15) / 16 * 16;
    const size_t stk = sim_stack_bytes(stack_levels, block_size, filter);
    return types + rows + kSimSharedBytes + waves + win + stk;
}

// One workgroup's lane stacks (stack_levels 0: none in LDS).
size_t sim_stack_bytes(uint32_t stack_levels, uint32_t block_size, bool filter)
{
    return (size_t)block_size * stack_levels * (filter ? sizeof(float) : sizeof(double));
}

hipError_t launch_zero(unsigned long long *p, uint64_t n, hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    uint64_t blocks = (n + 255) / 256;
    if (blocks > 4096)
        blocks = 4096;
    hipLaunchKernelGGL(zero_kernel, dim3((unsigned)blocks), dim3(256), 0, st, p, n);
    return hipGetLastError();
}

// The kernel of a launch: filtered tests or not, row tables in LDS, 32-bit
// heap indices and level masks (trees of at most 31 generations), lane stacks
// in device memory.
template <bool RowsLds, typename N, bool GStack>
auto sim_kernel_as(bool filter)
{
    return filter ? sim_filter_kernel<RowsLds, N, GStack> : sim_kernel<RowsLds, N, GStack>;
}

template <bool GStack>
auto sim_kernel_as(bool filter, bool rows_in_lds, bool narrow)
{
    if (rows_in_lds)
        return narrow ? sim_kernel_as<true, uint32_t, GStack>(filter) : sim_kernel_as<true, uint64_t, GStack>(filter);
    return narrow ? sim_kernel_as<false, uint32_t, GStack>(filter) : sim_kernel_as<false, uint64_t, GStack>(filter);
}

auto sim_kernel_of(bool rows_in_lds, uint32_t kdim, bool gstack, bool filter)
{
    return gstack ? sim_kernel_as<true>(filter, rows_in_lds, kdim <= 32) : sim_kernel_as<false>(filter, rows_in_lds, kdim <= 32);
}

hipError_t launch_sim(const RunArgs &a, const LaunchShape &ls, hipStream_t st)
{
    if (a.n_cells == 0)
        return hipSuccess;
    hipLaunchKernelGGL(sim_kernel_of(a.rows_in_lds != 0, a.kdim, a.gstack != nullptr, a.filter != 0), dim3(ls.blocks),
                       dim3(ls.block_size), ls.lds_bytes, st, a);
    return hipGetLastError();
}

hipError_t launch_debug_draws(uint64_t seed, const uint64_t *cell, const uint64_t *node,
                              const uint32_t *attempt, uint64_t n, uint32_t *words, double *z,
                              hipStream_t st)
{
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(debug_draws_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, seed,
                       cell, node, attempt, n, words, z);
    return hipGetLastError();
}

hipError_t sim_occupancy(int block_size, size_t lds_bytes, bool rows_in_lds, uint32_t kdim, bool gstack, bool filter,
                         int *blocks_per_cu)
{
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, sim_kernel_of(rows_in_lds, kdim, gstack, filter),
                                                        block_size, lds_bytes);
}

}  // namespace procell
