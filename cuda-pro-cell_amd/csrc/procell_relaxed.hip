// procell_relaxed.hip -- the relaxed (differentiable) estimator of the plain
// method's expected tally, and its gradient with respect to each type's
// (mean, sd, proportion).  No reference counterpart: the reference
// (src/simulation/proliferation.cu) only samples.
//
// Relaxation of the plain method (proliferation.cu:26-215, cell.cu:80-125):
//   * every initial cell takes every type j with weight p_j (no type draw);
//   * timers are the plain method's own, mean_j + sd_j z with z the first
//     candidate > 0 of the plain stream: the root's pair from block
//     (cell, 0, 0) words {2, -, 3, -}, then node 1's redraw stream; a node's
//     daughters' pair from block (cell, node, 0), a daughter whose candidate
//     is <= 0 continuing in its own node's redraw stream (with beta -> 0 and
//     one type the estimator is the plain tally of the same seed);
//     the root's phase U comes from word 1 of block (cell, 0, 0);
//   * the hard test "completes by t_max" becomes d = sigmoid((t_max - s)/beta)
//     for a node whose division would complete at s;
//   * a node of weight W records W (1 - d) at (row, generation k, type j) --
//     generation 0 only when the row's value is >= phi -- and its daughters
//     carry weight W d; fluorescence stays value / 2^k and the generation cap
//     is the plain method's;
//   * a node is expanded while k < cap and W d >= 1e-15.
// Along a path the completion time is s_k = tau_0 (1 + U) + tau_1 + ... +
// tau_k, so ds/dmean = (1 + U) + k, ds/dsd = z_0 (1 + U) + z_1 + ... + z_k,
// and dlog W/dtheta = -sum over ancestors of (1 - d)/beta ds/dtheta.  The
// backward pass recomputes every subtree from the Philox counters (nothing
// of the forward pass is stored) and accumulates
//   dL/dmean_j += p_j g W ((1 - d) dlogW/dmean + d (1 - d)/beta ds/dmean),
//   dL/dsd_j   += p_j g W ((1 - d) dlogW/dsd   + d (1 - d)/beta ds/dsd),
//   dL/dp_j    += g W (1 - d)
// for the cotangent g = dL/dh of each recorded entry.
//
// Kernel shape (walk_kernel): a workgroup of four wavefronts takes a segment
// of a set's initial cells, every proliferating type of each; its wavefronts
// claim root steps, which draw 64 roots at once into a buffer, and one walk
// per lane runs depth first.  A lane evaluates both daughters of a node as it
// expands it, so every step of every busy lane is one expansion (one Philox
// block, one Box-Muller pair, two sigmoids); expandable right daughters wait in
// a per-lane stack in device memory, the newest in registers.  Recorded
// weights go to an LDS window over the segment's rows (the cotangent's window
// in the backward pass) and reach the tally with FP64 atomics at the end.
//
// A plan covers one parameter set (procell_relaxed_*) or many (the batched
// calibration, procell_calib_*): sets' rows, cells and tally blocks are
// concatenated and every segment lies in one set.  A cell stride k
// (a power of two) restricts a pass to the initial cells of one residue
// class mod k.  A calibration step -- fill, forward pass, loss and cotangent,
// adjoint pass, Adam -- is captured once into a hipGraph and replayed.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <vector>

#include "procell_internal.hpp"
#include "procell_stream.hpp"
#include "procell_walk.hpp"

namespace procell {
namespace {

constexpr double kRelaxEps = 1e-15;        // smallest W d that is still expanded
// Expansions a single walk may take: a walk that needs more is cut short and
// counted, and the call reports PROCELL_E_DEPTH (parameters far outside the
// estimator's domain, e.g. sd a few times the mean with deep rows, where most
// timers lie near 0, would otherwise run for practically ever).
constexpr uint32_t kWalkBudget = 1u << 22;
// Calibration keeps sd <= 0.8 mean (log 0.8): the expected number of
// generation-k nodes, 2^k P(s_k <= t), grows with the timers' density near 0
// (for untruncated normal timers it would diverge beyond sd / mean = 0.85,
// where mean^2 / (2 sd^2) = ln 2), so the bound keeps the walks cheap.
constexpr double kLogMaxSdRatio = -0.22314355131420976;
constexpr uint32_t kWalkWaves = kWalkThreads / 64;
constexpr size_t kWalkLds = 40960;
// Idle lanes a wavefront tolerates before it draws roots (some 220
// instructions) or shares walks.  1e6 cells of 256 rows and 256 sets x 2e5
// cells: 231 us and 9.93 ms (8), 232 and 10.0 (12), 232 and 10.0 (16), 235
// and 10.3 (24).
constexpr uint32_t kWalkIdle = 12;
constexpr uint32_t kNoWindow = 0xFFFFFFFFu;
constexpr uint32_t kMaxCopies = 8;   // of a workgroup's window

// Expected expansions of a walk from which the last root steps of a segment
// are claimed in parts: a root step of short walks costs more than the
// wavefronts' uneven ends.
constexpr double kDeepWalk = 16.0;
// Least walks of a workgroup.
constexpr uint32_t kMinWalks = 256;
// Workgroups of a plan in resident workgroups.  One set: all resident at
// once, with equal shares of the estimated cost, so that none starts late
// (1e6 cells: 232 us; two 250).  Many sets: short segments cover few rows, so
// that the tallies stay in the LDS window.  256 sets x 2e5 cells and 64 sets:
// 11.1 and 2.31 ms (4), 10.0 and 2.32 (8), 9.66 and 2.55 (16); quarter of the
// cells 18.5 (8), 20.6 (16).
constexpr uint32_t kMultiSetFactor = 8;

// Device memory of a plan's lane stacks at most: a plan of more segments
// (every set has one; at 14 generations 50,000 fit) runs a pass as several
// launches, one after the other, over the same stacks.
constexpr size_t kStackBytes = 8ull << 30;

// Copies of a call's counters, one 128-byte line each; workgroup b adds to copy
// b mod 64.  One copy for all wavefronts: at 1e6 shallow walks their adds to
// one address came within 10 us and held up every CU's memory accesses for 30
// us (forward pass of the 1e6-cell calibration instance 107 -> 74 us).
constexpr uint32_t kCountCopies = 64, kCountWords = 16;

// One parameter set of a relaxed plan (a single-set plan has one).  Rows,
// initial cells, tally entries and type blocks of the sets are concatenated.
struct RelaxSet {
    uint64_t seed;
    double t_max;
    uint64_t cell_base;    // first initial cell (stream cell ids are relative to it)
    uint64_t h_base;       // first tally entry of the set's [rows][kdim][n_types]
    uint32_t row_base;     // first nonzero row
    uint32_t n_rows;
    uint32_t kdim;         // generations + 1
    uint32_t n_types;
    uint32_t theta_base;   // first entry of the set's [3][n_types] block of theta / gradient
    uint32_t prolif_base;  // first entry in the proliferating-type list
    uint32_t n_prolif;     // proliferating types (mean >= 0 when the plan was made)
    uint32_t quiet_base;
    uint32_t n_quiet;
    uint32_t deep;         // nonzero: walks of kDeepWalk expansions or more are expected
    uint32_t pad[2];
};

struct RelaxArgs {
    double beta;
    uint32_t n_sets;
    uint32_t n_rows;           // all sets
    uint32_t kdim_max;         // most generations + 1 of any set
    uint32_t even_ends;        // nonzero: every segment is resident at once
    uint32_t win_doubles[3];   // LDS window of a workgroup, per WalkMode
    uint32_t n_segments;
    uint32_t seg_first;        // first segment of a launch
    const RelaxSet *sets;
    const uint32_t *seg_set;   // [segments] set of each segment
    const uint32_t *seg_cell;  // [segments][2] first and end initial cell (set-local)
    const uint32_t *seg_row;   // [segments][2] first and last (global) row
    const uint32_t *seg_win;   // [3 modes][segments] first (global) row of the window
    const uint32_t *row_start; // [n_rows + 1] first initial cell of each row (all sets)
    const uint32_t *row_info;  // [n_rows] generation cap | (value >= phi) << 8
    const uint32_t *prolif;    // file index of each proliferating type, per set
    const uint32_t *quiet;     // file index of each quiescent type, per set
    const double *theta;       // per set [3][n_types]: mean, sd, proportion, file order
    double *stack;             // per workgroup of a launch and wavefront [kdim_max + 1 levels][64 lanes] frames
    double *h;                 // per set [rows][kdim][n_types] relaxed tally (forward)
    const double *g;           // cotangent, layout of h (backward)
    double *grad;              // per set [3][n_types] gradient (backward)
    unsigned long long *expansions;  // [kCountCopies][kCountWords] expansions of the call (roots drawn + nodes
                                     // expanded), walks cut; the sum over the copies counts
    unsigned long long *set_cuts;    // [n_sets] walks cut per set (NULL: not kept)
    // Cell stride: a pass walks only the initial cells c (set-local id) with
    // (c + phase) & stride_mask == 0; phase = (*step + phase) & stride_mask
    // when step is set (calibration: the step counter, the adjoint pass one
    // class ahead of the forward pass), else phase & stride_mask.
    const unsigned long long *step;
    uint32_t stride_mask;
    uint32_t phase;
    // Jacobian pass: [2][h_total] dh/dmean_j and dh/dsd_j of each entry's own
    // type j (h of type j depends on type j's parameters only)
    double *jac;
    uint64_t h_total;
};

// The FP64 constants of the walk, held in scalar registers: left to itself the
// compiler puts each 64-bit literal into a register again at every use, one
// or two scalar and often a vector instruction (0.45 to 0.56 scalar
// instructions per vector instruction, and half of the vector registers).
// An FP64 operation reads one scalar operand at no cost.  The log, sin/cos
// and exp polynomials share the factorials' reciprocals.
struct WalkConst {
    double r3, r5, r6, r7;              // 1/3, 1/5, 1/6, 1/7
    double f4, f5, f6, f7;              // 1/4!, 1/5!, 1/6!, 1/7!
    double f8, f9, f10, f12;
    double ln2_hi, ln2_lo, two_pi_hi, two_pi_lo;
    double log2e;
    double p53;                         // 2^-53
    // of these a polynomial's first step adds: an operation reads one scalar
    double f11, f4v, f5v, r6v;
};

__device__ __forceinline__ double in_sgpr(double x)
{
    asm("" : "+s"(x));
    return x;
}

__device__ __forceinline__ double in_vgpr(double x)
{
    asm("" : "+v"(x));
    return x;
}

__device__ __forceinline__ WalkConst walk_const()
{
    constexpr dev::Coeffs C = dev::coeffs();
    static_assert(C.lp[0] == -0.5 && C.lp[2] == -0.25 && C.lp[4] == C.s1 && C.c1 == -0.5, "shared coefficients");
    return WalkConst{in_sgpr(C.lp[1]), in_sgpr(C.lp[3]), in_sgpr(-C.lp[4]), in_sgpr(C.lp[5]),
                     in_sgpr(C.c2), in_sgpr(C.s2), in_sgpr(-C.c3), in_sgpr(-C.s3),
                     in_sgpr(2.48015873015873e-05), in_sgpr(2.7557319223985893e-06), in_sgpr(2.755731922398589e-07),
                     in_sgpr(2.08767569878681e-09),
                     in_sgpr(C.ln2_hi), in_sgpr(C.ln2_lo), in_sgpr(C.two_pi_hi), in_sgpr(C.two_pi_lo),
                     in_sgpr(1.4426950408889634), in_sgpr(0x1p-53),
                     in_vgpr(2.505210838544172e-08), in_vgpr(C.c2), in_vgpr(C.s2), in_vgpr(-C.lp[4])};
}

// The stream's coefficients from the shared ones.
__device__ __forceinline__ dev::Coeffs stream_coeffs(const WalkConst &c)
{
    return dev::Coeffs{{-0.5, c.r3, -0.25, c.r5, -c.r6v, c.r7}, c.ln2_hi, c.ln2_lo, c.two_pi_hi, c.two_pi_lo,
                       -c.r6, c.f5v, -c.f7, -0.5, c.f4v, -c.f6};
}

// dev::log_with_entry, bit for bit: the hardware splits x = m 2^e with m in
// [0.5, 1), and where m is halved against the table's (j < 64) the entry's
// 1/c comes doubled (see walk_log_table).
__device__ __forceinline__ double walk_log(double x, uint32_t j, double invc, double logc, const dev::Coeffs &K)
{
    const double r = fma(__builtin_amdgcn_frexp_mant(x), invc, -1.0);
    const double de = (double)(__builtin_amdgcn_frexp_exp(x) + (int)(j >> 6) - 1);
    const double r2 = r * r;
    double p = fma(K.lp[5], r, K.lp[4]);
    p = fma(p, r, K.lp[3]);
    p = fma(p, r, K.lp[2]);
    p = fma(p, r, K.lp[1]);
    p = fma(p, r, K.lp[0]);
    const double hi = fma(de, K.ln2_hi, logc);
    const double t = fma(r2, p, de * K.ln2_lo);
    return hi + (r + t);
}

// Entry j of the LDS copy of the log table.
__device__ __forceinline__ double2 walk_log_table(uint32_t j)
{
    const double invc = dev::procell_log_table[j][0];
    return make_double2(j < 64 ? 2.0 * invc : invc, dev::procell_log_table[j][1]);
}

// The stream's Box-Muller pair (dev::normal_pair) with the walk's constants:
// the same log and sin/cos; the square root by Goldschmidt's method from the
// hardware's estimate (Markstein, 1990) where the stream's, which a host must
// be able to repeat, starts from an integer estimate with three Newton steps.
__device__ __forceinline__ void walk_pair(const dev::Words &w, double &z0, double &z1, const WalkConst &c,
                                          const dev::Coeffs &K, const dev::Tables &tb)
{
    const double u = fma((double)w.w0, 0x1p-32, fma((double)(w.w1 >> 11), c.p53, c.p53));
    const uint32_t jl = dev::log_index(u);
    const double invc = tb.log[jl][0], logc = tb.log[jl][1];
    // the nearest 1/256 turn t and what is left of the turns: both exact
    const uint32_t t = w.w2 + 0x800000u;
    const uint32_t js = t >> 24;
    const double sa = tb.sincos[js][0], ca = tb.sincos[js][1];
    const double d = fma((double)(int32_t)(w.w2 - (t & 0xFF000000u)), 0x1p-32, (double)(w.w3 >> 11) * c.p53);
    const double a = fma(d, K.two_pi_hi, d * K.two_pi_lo);
    const double a2 = a * a;
    double ps = fma(a2, K.s3, K.s2);
    ps = fma(a2, ps, K.s1);
    const double st = fma(a * a2, ps, a);
    const double cm = a2 * fma(a2, fma(a2, K.c3, K.c2), K.c1);
    const double sn = sa + fma(sa, cm, ca * st), cs = ca + fma(ca, cm, -(sa * st));
    // (u = 1: log 0, for which the least normal number keeps rho finite and 0 in effect)
    const double x = fmax(-2.0 * walk_log(u, jl, invc, logc, K), 0x1p-1022);
    const double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * y;
    double g = x * y;
    g = fma(g, fma(-h, g, 0.5), g);
    const double rho = fma(fma(-g, g, x), h, g);
    z0 = rho * cs;
    z1 = rho * sn;
}

// exp(x) for -40 <= x <= 700 (below -40, 1 + exp(x) rounds to 1): x = k ln 2
// + r with |r| <= ln 2 / 2 (Cody-Waite reduction, ln 2 in two parts), exp(r)
// by its Taylor polynomial of degree 12 (truncation below 2e-16 relative),
// times 2^k.
__device__ __forceinline__ double exp_sig(double x, const WalkConst &c)
{
    const double k = __builtin_rint(x * c.log2e);
    double r = fma(-k, c.ln2_hi, x);
    r = fma(-k, c.ln2_lo, r);
    double p = fma(c.f12, r, c.f11);
    p = fma(p, r, c.f10);
    p = fma(p, r, c.f9);
    p = fma(p, r, c.f8);
    p = fma(p, r, c.f7);
    p = fma(p, r, c.f6);
    p = fma(p, r, c.f5);
    p = fma(p, r, c.f4);
    p = fma(p, r, c.r6);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return __builtin_ldexp(p, (int)k);
}

// 1 / x for x >= 1: the hardware estimate r (relative error e < 2^-24) and
// one cubic step r + r (e + e^2), which leaves e^3 and the last rounding.
__device__ __forceinline__ double recip_ge1(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// sigmoid(y / beta) with ib = 1 / beta.  The exponent is capped at 700 so
// that 1 + e stays finite (an infinite one would turn the Newton steps into
// inf x 0); there the sigmoid is below 1e-304 either way.
__device__ __forceinline__ double sigmoid_scaled(double y, double ib, const WalkConst &c)
{
    return recip_ge1(1.0 + exp_sig(fmin(fmax(-(y * ib), -40.0), 700.0), c));
}

// A root walk buffered in LDS between a root step and the hand-out to an idle
// lane: completion time and sigmoid of the root and (tangent passes) 1 + U of
// its phase and ds/dsd.
template <bool Tan>
struct WalkEntry;
template <>
struct alignas(16) WalkEntry<false> {
    double s, d;
    uint32_t cell;  // set-local id
    uint32_t tb;    // LDS address of the window entry (row, generation 0, type), or kNoWindow
    uint32_t rowt;  // row relative to the set's first row | type << 24
    uint32_t kcap;
};
template <>
struct alignas(16) WalkEntry<true> {
    double s, d;
    double u1, b;
    uint32_t cell, tb, rowt, kcap;
};

static_assert(sizeof(WalkEntry<false>) == walk_entry_bytes(false) && sizeof(WalkEntry<true>) == walk_entry_bytes(true),
              "LDS layout");

// Stacked right daughter: completion time and W d; tangent passes also ds/dsd
// and its daughters' dlogW/dmean, dlogW/dsd (padded to 16-byte words).
template <bool Tan>
struct WalkFrame;
template <>
struct alignas(16) WalkFrame<false> {
    double s, w;
};
template <>
struct alignas(16) WalkFrame<true> {
    double s, w, b, gm, gs, pad;
};
constexpr uint32_t kFrameBytes = sizeof(WalkFrame<true>);

typedef __attribute__((address_space(3))) double LdsDouble;
typedef __attribute__((address_space(3))) uint32_t LdsWord;
__device__ __forceinline__ void lds_add(uint32_t at, double v)
{
    __hip_atomic_fetch_add((LdsDouble *)(uintptr_t)at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ uint32_t uni(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ uint32_t lane_rank(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ uint32_t low_bit(uint32_t m) { return (uint32_t)__builtin_ctz(m); }
__device__ __forceinline__ uint32_t low_bit(uint64_t m) { return (uint32_t)__builtin_ctzll(m); }
__device__ __forceinline__ uint32_t top_bit(uint32_t m) { return 31u - (uint32_t)__builtin_clz(m); }
__device__ __forceinline__ uint32_t top_bit(uint64_t m) { return 63u - (uint32_t)__builtin_clzll(m); }
// Index of the r-th set bit of m (r < popcount(m)).
__device__ __forceinline__ uint32_t nth_set_bit(uint64_t m, uint32_t r)
{
    for (; r; --r)
        m &= m - 1;
    return (uint32_t)__builtin_ctzll(m);
}

__device__ __forceinline__ uint64_t again_value(uint64_t x)
{
    asm volatile("" : "+s"(x));
    return x;
}
typedef __attribute__((address_space(4))) RelaxArgs ConstArgs;
typedef __attribute__((address_space(4))) RelaxSet ConstSet;
template <typename P>
__device__ __forceinline__ P *again(P *p)
{
    asm volatile("" : "+s"(p));
    return p;
}

// ======================================================================
// walk_kernel: one workgroup walks the trees of one segment of a set's initial
// cells, every proliferating type of each.  As in sim_filter_kernel, its
// wavefronts claim root steps (64 walks: 64 / n_prolif cells, the lane's type
// fixed) from an LDS cursor, draw those roots on all lanes into an LDS buffer,
// hand them to idle lanes, and every busy lane expands one node per step:
// both daughters' timers, sigmoids and records; it goes on with the left
// daughter, else the right, else the lowest pending level of its mask.  At the
// end of the segment idle lanes take the shallowest pending daughter of busy
// lanes.
//
// What bounds it is the vector unit's issue rate (4 cycles per SIMD for nearly
// every FP64 and integer instruction): the forward pass takes some 275 of them
// per step, root steps and hand-outs included, with 64 of 64 lanes in work, and
// a CU 320 cycles per step; the Jacobian pass, 5 LDS and up to 6 memory
// accesses more, issues 0.81 per cycle.  One static range of walks per wavefront,
// roots drawn in the walks' own steps and no sharing at the end kept 40 to 45
// lanes busy at 0.71-0.73.  1e6 cells: 330 -> 219 us, adjoint 424 -> 245;
// Jacobian of 64 sets x 2e5 cells 3.63 -> 2.13 ms, calibration step of 256
// sets 14.0 -> 9.0 ms, with a quarter of the cells 7.4 -> 4.2 ms.
//  * constants, arguments: see WalkConst and args_again; the compiler's own choice
//    took 45 instructions per step more.
//  * the most recently pushed daughter stays in registers (the frame F): it is
//    the next one popped.  A push writes an F that is not in memory yet to its
//    level's frame in device memory; a pop lets the next step
//    begin with the read of the next F.  A second frame in LDS halved the
//    memory traffic and took as long (the LDS then has more to do).
//  * a node's frame holds what its own expansion needs, W d and its daughters'
//    tangents, rather than W, d and its own tangents: the sigmoid is not kept.
//  * p_j and, for the tangents, 1 / beta multiply the sums, not the records:
//    gm and gs are beta dlogW/dmean and beta dlogW/dsd.
//  * a timer <= 0 waits for the next steps, which draw from its redraw stream
//    on that lane beside the other lanes' expansions.
//  * the window is kept in up to 8 copies where it is small: the adds of 64
//    lanes meet in some 30 entries (Jacobian pass of 64 sets 2.58 -> 2.31 ms).
//  * the quiescent types' records are written here too and everything is
//    cleared in one launch: four launches per pass became two (forward
//    pass of one cell 23 -> 16 us).
//  * where all segments run at once, the hardware prefers the older of a
//    SIMD's wavefronts, so that the youngest ends alone, at a third of the
//    rate; a wavefront of a segment with more left to claim takes a higher
//    priority (242 -> 232 us).
// LDS: see walk_lds.
// ======================================================================
template <int Mode, typename N>
__global__ __launch_bounds__(kWalkThreads, 4) void walk_kernel(RelaxArgs args)
{
    constexpr bool Grad = Mode == kAdjoint, Jac = Mode == kJacobian, Tan = Mode != kForward;
    constexpr uint32_t kParts = Jac ? 3 : 1;  // values of a window entry
    using Entry = WalkEntry<Tan>;
    using Frame = WalkFrame<Tan>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uni(tid >> 6);
    const uint32_t seg = args.seg_first + blockIdx.x;
    const uint32_t set_id = args.seg_set[seg];
    // The arguments and the set's values are read again (scalar loads) where
    // they are rarely used: held through the loop they would take the scalar
    // registers of the walk's constants.
    const ConstArgs *ap = (const ConstArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    const ConstSet *sp = (const ConstSet *)(uintptr_t)(args.sets + set_id);
    auto args_again = [&]() -> const ConstArgs & { return *again(ap); };
    auto set_again = [&]() -> const ConstSet & { return *again(sp); };
    const ConstArgs &a = *ap;
    const ConstSet &S = *sp;
    const uint32_t T = S.n_types, T8 = T * 8, TW = T8 * kParts, KT = S.kdim * T;
    const uint32_t r_lo = a.seg_row[2 * seg], r_hi = a.seg_row[2 * seg + 1];
    const uint32_t w_lo = a.seg_win[Mode * a.n_segments + seg];  // first row of the window
    // selected cells of the segment: first, first + stride, ... (set-local)
    const uint32_t sshift = (uint32_t)__popc(a.stride_mask);
    const uint32_t phase = ((a.step ? (uint32_t)a.step[0] : 0u) + a.phase) & a.stride_mask;
    const uint32_t c_begin = a.seg_cell[2 * seg], c_end = a.seg_cell[2 * seg + 1];
    const uint32_t first = uni(c_begin + ((0u - (c_begin + phase)) & a.stride_mask));
    const uint32_t n_sel = uni(first >= c_begin && c_end > first ? ((c_end - 1u - first) >> sshift) + 1u : 0u);

    const WalkLds at_lds = walk_lds(T, Mode);
    double(*m_log)[2] = (double(*)[2])lds_raw;
    double(*m_sc)[2] = (double(*)[2])(lds_raw + 128 * 16);
    double *theta = (double *)(lds_raw + at_lds.theta);
    double *gsum = (double *)(lds_raw + at_lds.sums);
    uint32_t *prolif = (uint32_t *)(lds_raw + at_lds.prolif);
    uint32_t *cursor = (uint32_t *)(lds_raw + at_lds.cursor);
    Entry *ent = (Entry *)(lds_raw + at_lds.entries) + wave * 64;
    double *held = (double *)(lds_raw + at_lds.held) + tid * 2;  // a waiting lane's timers
    uint32_t *origin_exp = (uint32_t *)ent, *origin = origin_exp + 64;  // (steals)
    double *win = (double *)(lds_raw + at_lds.window);
    const uint32_t win_base = (uint32_t)(uintptr_t)(LdsDouble *)win;
    const uint32_t n_win = min(r_hi - w_lo + 1, a.win_doubles[Mode] / (KT * kParts));  // rows with a window
    const uint32_t win_n = n_win * KT;
    // copies of the window, a lane adding to one of them: 64 lanes meet in a few
    // entries, and adds to one address take turns
    const uint32_t win_stride = kParts * win_n + 1u;
    uint32_t copies = 1;
    if constexpr (!Grad)
        while (copies < kMaxCopies && 2 * copies * win_stride <= a.win_doubles[Mode])
            copies *= 2;
    const uint32_t lane_copy = (lane & (copies - 1u)) * win_stride * 8u;
    const bool all_in = w_lo == r_lo && n_win == r_hi - r_lo + 1;
    const uint64_t h0 = S.h_base + (uint64_t)(w_lo - S.row_base) * KT;  // tally index of the window
    for (uint32_t i = tid; i < 128; i += kWalkThreads) {
        const double2 e = walk_log_table(i);
        m_log[i][0] = e.x;
        m_log[i][1] = e.y;
    }
    for (uint32_t i = tid; i < 256; i += kWalkThreads) {
        m_sc[i][0] = dev::procell_sincos_table[i][0];
        m_sc[i][1] = dev::procell_sincos_table[i][1];
    }
    for (uint32_t i = tid; i < 3 * T; i += kWalkThreads) {
        theta[i] = a.theta[S.theta_base + i];
    }
    // copies of the gradient sums, as of the window
    uint32_t sums = 1;
    if constexpr (Grad) {
        while (sums < 16 && 2 * sums * 3 * T <= kGradSums)
            sums *= 2;
        for (uint32_t i = tid; i < sums * 3 * T; i += kWalkThreads)
            gsum[i] = 0.0;
    }
    const uint32_t lane_sums = (uint32_t)(uintptr_t)(LdsDouble *)gsum + (lane & (sums - 1u)) * 3 * T8;
    for (uint32_t i = tid; i < S.n_prolif; i += kWalkThreads)
        prolif[i] = a.prolif[S.prolif_base + i];
    for (uint32_t i = tid; i < (Grad ? win_n : copies * win_stride); i += kWalkThreads)
        win[i] = Grad ? a.g[h0 + i] : 0.0;
    if (tid < 4)
        cursor[tid] = 0u;
    __syncthreads();

    // Quiescent types: each initial cell of a row with value >= phi records p_j
    // at generation 0 (cell.cu:104-108 gives them timer -1, always out of
    // time).  A row's are this segment's if its first cell is.  One wavefront
    // takes them while the others draw roots.
    if (S.n_quiet && wave == kWalkWaves - 1) {
        const uint32_t row0 = r_lo + (a.row_start[r_lo] < (uint32_t)S.cell_base + c_begin ? 1u : 0u);
        for (uint32_t row = row0 + lane; row <= r_hi; row += 64) {
            if (((a.row_info[row] >> 8) & 1u) == 0)
                continue;
            // selected cells of the row: local ids c in [lo, hi) with c + phase
            // a multiple of the stride
            const uint64_t lo = a.row_start[row] - S.cell_base + phase, hi = a.row_start[row + 1] - S.cell_base + phase;
            const double cnt = (double)(((hi + a.stride_mask) >> sshift) - ((lo + a.stride_mask) >> sshift));
            const uint64_t e = S.h_base + (uint64_t)(row - S.row_base) * KT;
            for (uint32_t q = 0; q < S.n_quiet; ++q) {
                const uint32_t j = a.quiet[S.quiet_base + q];
                if constexpr (Grad)
                    lds_add(lane_sums + 2 * T8 + j * 8, cnt * a.g[e + j]);
                else
                    a.h[e + j] = cnt * theta[2 * T + j];
            }
        }
    }

    const WalkConst C = walk_const();
    const dev::Coeffs K = stream_coeffs(C);
    const dev::Tables tb{m_log, m_sc};
    const uint64_t seed = again_value(S.seed);
    const double t_max = in_sgpr(S.t_max), ib = 1.0 / a.beta;
    // root steps: cells of `n_prolif` types each, lanes in (cell, type) order,
    // or 64 types of one cell of several chunks
    const uint32_t n_prolif = max(1u, S.n_prolif);
    const uint32_t chunks = uni((n_prolif + 63) / 64);
    const uint32_t per_step = uni(chunks > 1 ? 1u : 64u / n_prolif);  // cells of a full step
    const uint32_t lane_cell = chunks > 1 ? 0u : lane / n_prolif, lane_type = chunks > 1 ? lane : lane % n_prolif;
    const uint32_t n_units = uni(S.n_prolif ? n_sel * chunks : 0u);
    // the last walks are claimed as they are needed, so that the wavefronts end together
    const uint32_t tail = uni(S.deep ? n_units - min(n_units, per_step * kWalkWaves) : n_units);

    uint32_t rpos = 0, rn = 0, roots_done = 0;
    uint32_t rb = r_lo, bnd = 0, rinfo = 0;  // row boundaries, as in sim_kernel
    auto load_rows = [&]() {
        const uint32_t r1 = rb + 1 + lane;
        bnd = r1 <= args_again().n_rows ? args_again().row_start[r1] : 0xFFFFFFFFu;
        rinfo = rb + lane < args_again().n_rows ? args_again().row_info[rb + lane] : 0u;
    };
    load_rows();
    // the lane's frames: level l at stk + l * kLevelBytes (level 0 is read, not
    // used).  By level, then lane: lanes at one level share their lines, and a
    // line holds no levels that are rarely touched.  By lane, then level (each
    // lane's levels in its own lines): Jacobian pass of 64 sets 2.26 -> 2.15
    // ms, calibration step 9.55 -> 9.0, adjoint of 1e6 cells 257 -> 249 us; a
    // frame's fields apart (16 bytes per lane): 2.44 ms.
    constexpr uint32_t kLevelBytes = 64 * sizeof(Frame);
    const size_t levels = (size_t)args_again().kdim_max + 1;
    unsigned char *const stk0 = (unsigned char *)args_again().stack + ((size_t)blockIdx.x * kWalkThreads + wave * 64) * levels * kFrameBytes;
    unsigned char *const stk = stk0 + (size_t)lane * sizeof(Frame);

    // lane state: the node to expand
    N node = 0, pend = 0;  // pend: pending levels relative to k and the level-0 bit; 0: idle
    uint32_t k = 0, kcap = 0, cell = 0, tbl = 0, rowt = 0;
    uint32_t redo = 0;   // redraw pending: timers still to draw (bits 0, 1) | attempt << 16
    uint32_t since = 0;  // step at which the walk started, and one more per step spent waiting for a redraw
    double mean = 0.0, sd = 0.0, s = 0.0, W = 0.0, u1 = 0.0, b = 0.0, gm = 0.0, gs = 0.0;
    double F_s = 0.0, F_w = 0.0, F_b = 0.0, F_gm = 0.0, F_gs = 0.0;
    double acc_m = 0.0, acc_s = 0.0, acc_p = 0.0;
    uint64_t dirty = 0;     // lanes whose F is not in memory
    uint64_t popped = 0;    // lanes that took their F in the last step: the next one is read
    uint64_t redoing = 0;   // lanes with a redraw pending
    uint64_t w_exp = 0;     // expansions
    uint32_t n_cut = 0, steps = 0;
    uint32_t check = kWalkBudget - 1u;  // first step at which a walk may be near its budget
    bool shared = false, counted = false;  // steals have begun; walks are counted in origin_exp

    // a frame to its level, F into `below` and back
    auto store_frame = [&](uint32_t level, double fs, double fw, double fb, double fgm, double fgs) {
        Frame *f = (Frame *)(stk + (size_t)level * kLevelBytes);
        f->s = fs;
        f->w = fw;
        if constexpr (Tan) {
            f->b = fb;
            f->gm = fgm;
            f->gs = fgs;
        }
    };
    // Reads of frames have arrived (vmcnt 0), on every path and before the
    // step's stores: where the compiler has to wait by itself, stores may
    // follow the reads, and it waits for those as well.
    auto frames_read = []() { __builtin_amdgcn_s_waitcnt(0x0F70); };
    // the adjoint's sums of a walk, or of the part of it that ran on this lane
    auto end_walk = [&]() {
        if constexpr (Grad) {
            const uint32_t at = lane_sums + (rowt >> 24) * 8;
            lds_add(at, acc_m);
            lds_add(at + T8, acc_s);
            lds_add(at + 2 * T8, acc_p);
            acc_m = acc_s = acc_p = 0.0;
        }
    };

    for (;;) {
        const uint64_t idle = __ballot(pend == 0);
        const uint32_t n_idle = uni((uint32_t)__popcll(idle));
        if (n_idle > kWalkIdle) {
            // ---- root step: the buffer is empty ----
            if (rpos >= rn && !roots_done) {
                uint32_t unit = 0, want = per_step;
                if (lane == 0) {
                    if (__hip_atomic_load((LdsWord *)cursor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= tail)
                        want = min(per_step, max((n_idle + n_prolif - 1) / n_prolif, (per_step + 3) / 4));
                    unit = atomicAdd(cursor, want);
                }
                unit = uni(unit);
                want = uni(want);
                if (unit >= n_units)
                    roots_done = 1;
                if (args_again().even_ends) {
                    const uint32_t left = n_units - min(unit, n_units);
                    if (left > n_units / 2)
                        __builtin_amdgcn_s_setprio(3);
                    else if (left > n_units / 4)
                        __builtin_amdgcn_s_setprio(2);
                    else if (left > n_units / 8)
                        __builtin_amdgcn_s_setprio(1);
                    else
                        __builtin_amdgcn_s_setprio(0);
                }
                if (!roots_done) {
                    const uint32_t i0 = chunks > 1 ? unit / chunks : unit;
                    const uint32_t type = chunks > 1 ? (unit % chunks) * 64 + lane_type : lane_type;
                    const bool valid = lane_cell < want && i0 + lane_cell < n_sel && type < n_prolif;
                    const uint32_t c = first + ((valid ? i0 + lane_cell : i0) << sshift);
                    const uint32_t gcell = (uint32_t)set_again().cell_base + c;  // (cells of all sets < 2^32)
                    const uint32_t g_first = uni((uint32_t)set_again().cell_base + first + (i0 << sshift));
                    const uint32_t g_last = uni((uint32_t)set_again().cell_base + first + ((min(i0 + want, n_sel) - 1u) << sshift));
                    for (uint64_t le = __ballot(bnd <= g_first); le; le = __ballot(bnd <= g_first)) {
                        rb = uni(rb + (uint32_t)__popcll(le));
                        load_rows();
                    }
                    const uint32_t nb = uni((uint32_t)__popcll(__ballot(bnd <= g_last)));
                    uint32_t row = rb, info = uni(rinfo);
                    if (nb == 64) {  // (a cell stride over short rows) beyond the boundaries at hand
                        uint32_t lo = rb, hi = r_hi;
                        while (lo < hi) {
                            const uint32_t mid = lo + (hi - lo + 1) / 2;
                            if (args_again().row_start[mid] <= gcell)
                                lo = mid;
                            else
                                hi = mid - 1;
                        }
                        row = lo;
                        info = args_again().row_info[row];
                    } else if (nb) {
                        for (uint32_t j = 0; j < nb; ++j)
                            row += gcell >= (uint32_t)__builtin_amdgcn_readlane((int)bnd, (int)j) ? 1u : 0u;
                        info = (uint32_t)__shfl(rinfo, (int)(row - rb));
                    }
                    const uint32_t cap = info & 255u;
                    const bool ge_phi = ((info >> 8) & 1u) != 0;
                    const uint32_t j = prolif[valid ? type : 0u];
                    const double m_j = theta[j], sd_j = theta[T + j];
                    const dev::Words w = dev::draw_block(set_again().seed, c, 0, 0u);
                    const double U1 = 1.0 + dev::uniform_oc(w.w1, 0u);
                    double z0, z1;
                    walk_pair(dev::Words{w.w2, 0u, w.w3, 0u}, z0, z1, C, K, tb);
                    // the plain method's timer (cell.cu:106-122): the second
                    // candidate, then node 1's redraw stream; after 65535
                    // blocks the timer is the mean (z = 0)
                    if (__builtin_expect(__ballot(valid && !(fma(z0, sd_j, m_j) > 0.0)) != 0, 0)) {
                        if (valid && !(fma(z0, sd_j, m_j) > 0.0)) {
                            z0 = z1;
                            if (!(fma(z0, sd_j, m_j) > 0.0)) {
                                z0 = 0.0;
                                for (uint32_t att = 1; att < 65536u; ++att) {
                                    double y0, y1;
                                    walk_pair(dev::draw_block(set_again().seed, c, 1, att), y0, y1, C, K, tb);
                                    if (fma(y0, sd_j, m_j) > 0.0) { z0 = y0; break; }
                                    if (fma(y1, sd_j, m_j) > 0.0) { z0 = y1; break; }
                                }
                            }
                        }
                    }
                    const double s0 = fma(z0, sd_j, m_j) * U1;
                    const double d0 = sigmoid_scaled(t_max - s0, ib, C);
                    const double e0 = 1.0 - d0, b0 = z0 * U1;
                    const uint32_t wrow = row - w_lo;
                    const uint32_t at = win_base + lane_copy + (__umul24(min(wrow, n_win), KT) + j) * (8 * kParts);
                    const bool in_win = wrow < n_win;
                    const uint64_t e = set_again().h_base + (uint64_t)(row - set_again().row_base) * KT + j;
                    if (valid && ge_phi) {
                        const double q = d0 * e0;
                        const double vm = q * U1, vs = q * b0;
                        if (Grad) {
                            const double gv = in_win ? *(LdsDouble *)(uintptr_t)at : args_again().g[e];
                            lds_add(lane_sums + j * 8, gv * vm);
                            lds_add(lane_sums + T8 + j * 8, gv * vs);
                            lds_add(lane_sums + 2 * T8 + j * 8, gv * e0);
                        } else if (in_win) {
                            lds_add(at, e0);
                            if (Jac) {
                                lds_add(at + 8, vm);
                                lds_add(at + 16, vs);
                            }
                        } else {
                            const double p = theta[2 * T + j];
                            unsafeAtomicAdd(args_again().h + e, p * e0);
                            if (Jac) {
                                const double p = theta[2 * T + j] * ib;
                                unsafeAtomicAdd(args_again().jac + e, p * vm);
                                unsafeAtomicAdd(args_again().jac + args_again().h_total + e, p * vs);
                            }
                        }
                    }
                    const uint64_t vmask = __ballot(valid);
                    w_exp += (uint64_t)__popcll(vmask);
                    const bool grows = valid && cap > 0 && d0 >= kRelaxEps;
                    const uint64_t gmask = __ballot(grows);
                    if (grows) {
                        Entry &q = ent[lane_rank(gmask)];
                        q.s = s0;
                        q.d = d0;
                        if constexpr (Tan) {
                            q.u1 = U1;
                            q.b = b0;
                        }
                        q.cell = c;
                        q.tb = in_win ? at : kNoWindow;
                        q.rowt = (row - set_again().row_base) | (j << 24);
                        q.kcap = cap;
                    }
                    rpos = 0;
                    rn = uni((uint32_t)__popcll(gmask));
                    __builtin_amdgcn_wave_barrier();
                }
            }
            // ---- steals: the walks left share the wavefront ----
            if (rpos >= rn && roots_done && !counted) {
                const N real = pend & (((N)1 << k) - (N)1);
                const uint64_t donors = __ballot(real != 0);
                const uint32_t nd = uni(min((uint32_t)__popcll(donors), n_idle));
                if (nd) {
                    if (!shared) {
                        shared = true;
                        check = min(check, steps + (kWalkBudget - 1u - min(steps, kWalkBudget - 1u)) / 64u);
                        origin_exp[lane] = 0u;
                        origin[lane] = lane;
                        __builtin_amdgcn_wave_barrier();
                    }
                    // the daughter taken is F where it is the only one and in
                    // the registers; any other lies in memory
                    const uint64_t in_reg = __ballot((real & (real - 1)) == 0) & ~popped;
                    const uint32_t my_up = real ? top_bit(real) : 0u;
                    const uint32_t r = lane_rank(idle);
                    const bool thief = pend == 0 && r < nd;
                    const uint32_t src = thief ? nth_set_bit(donors, r) : lane;
                    const uint32_t up = __shfl(my_up, (int)src);
                    const N d_node = __shfl(node, (int)src);
                    const uint32_t d_k = __shfl(k, (int)src), d_cell = __shfl(cell, (int)src);
                    const uint32_t d_kcap = __shfl(kcap, (int)src), d_tb = __shfl(tbl, (int)src);
                    const uint32_t d_rowt = __shfl(rowt, (int)src);
                    const double d_mean = __shfl(mean, (int)src), d_sd = __shfl(sd, (int)src);
                    const double d_u1 = Tan ? __shfl(u1, (int)src) : 0.0;
                    const uint32_t d_origin = origin[src];
                    const bool given = real != 0 && lane_rank(donors) < nd;
                    if (given)
                        pend &= ~((N)1 << my_up);
                    dirty &= ~(__ballot(given) & in_reg);
                    const double d_s = __shfl(F_s, (int)src), d_w = __shfl(F_w, (int)src);
                    const double d_b = Tan ? __shfl(F_b, (int)src) : 0.0, d_gm = Tan ? __shfl(F_gm, (int)src) : 0.0;
                    const double d_gs = Tan ? __shfl(F_gs, (int)src) : 0.0;
                    const bool from_memory = thief && ((in_reg >> src) & 1ull) == 0;
                    if (__ballot(from_memory))
                        frames_read();  // (and written: vmcnt counts both)
                    if (thief) {
                        k = d_k - up;
                        s = d_s;
                        W = d_w;
                        if constexpr (Tan) {
                            b = d_b;
                            gm = d_gm;
                            gs = d_gs;
                            u1 = d_u1;
                        }
                        if (from_memory) {
                            const Frame *f = (const Frame *)(stk0 + (size_t)k * kLevelBytes + src * sizeof(Frame));
                            s = f->s;
                            W = f->w;
                            if constexpr (Tan) {
                                b = f->b;
                                gm = f->gm;
                                gs = f->gs;
                            }
                        }
                        node = (d_node >> up) | (N)1;
                        pend = (N)1 << k;
                        cell = d_cell;
                        kcap = d_kcap;
                        tbl = d_tb;
                        rowt = d_rowt;
                        mean = d_mean;
                        sd = d_sd;
                        origin[lane] = d_origin;
                        since = steps;
                    }
                    frames_read();
                }
            }
        }
        // ---- idle lanes take buffered walks ----
        if (rpos < rn) {
            const uint64_t idle2 = __ballot(pend == 0);
            const uint32_t rank = lane_rank(idle2) + rpos;
            if (pend == 0 && rank < rn) {
                const Entry q = ent[rank];
                s = q.s;
                W = q.d;
                if constexpr (Tan) {
                    const double e = 1.0 - q.d;
                    u1 = q.u1;
                    b = q.b;
                    gm = -(e * u1);
                    gs = -(e * b);
                }
                cell = q.cell;
                tbl = q.tb;
                rowt = q.rowt;
                kcap = q.kcap;
                mean = theta[rowt >> 24];
                sd = theta[T + (rowt >> 24)];
                node = (N)1;
                pend = (N)1;
                k = 0;
                since = steps - 1u;  // (the root counts)
            }
            rpos = uni(min(rpos + (uint32_t)__popcll(idle2), rn));
        }
        const uint64_t busy = __ballot(pend != 0);
        if (busy == 0 && roots_done && rpos >= rn)
            break;
        ++steps;
        // A walk past its budget is cut short (counted; the call reports it).
        // A lane's walk has taken steps - since expansions after this step; no
        // walk can be near the budget before that many steps, or a 64th of
        // them once its parts run on several lanes.
        uint64_t over = 0;
        if (__builtin_expect(steps >= check, 0)) {
            if (!shared) {
                over = __ballot(pend != 0 && steps - since > kWalkBudget);
            } else {
                // exact: every walk's expansions summed by origin lane
                if (!counted) {
                    counted = true;
                    if (pend != 0)
                        atomicAdd(&origin_exp[origin[lane]], steps - 1u - since + (redo ? 1u : 0u));
                }
                bool past = false;
                if (pend != 0 && redo == 0) {
                    const uint32_t n = atomicAdd(&origin_exp[origin[lane]], 1u);
                    past = n >= kWalkBudget;
                    n_cut += n == kWalkBudget ? 1u : 0u;
                }
                over = __ballot(past);
            }
            if (over) {
                if (__builtin_amdgcn_inverse_ballot_w64(over)) {
                    n_cut += shared ? 0u : 1u;
                    end_walk();
                    pend = 0;
                    redo = 0;
                }
                redoing &= ~over;
                dirty &= ~over;
            }
        }

        // ======== one expansion per busy lane ========
        bool expanded = false, push = false, pop = false;
        if (pend != 0) {
            // the next F, for this step's end (level 0 when no level is
            // pending: read, not used)
            if (__builtin_amdgcn_inverse_ballot_w64(popped)) {
                const Frame *f = (const Frame *)(stk + (size_t)(k - low_bit(pend)) * kLevelBytes);
                F_s = f->s;
                F_w = f->w;
                if constexpr (Tan) {
                    F_b = f->b;
                    F_gm = f->gm;
                    F_gs = f->gs;
                }
            }
            N bnode = node;
            if (__builtin_expect(redoing != 0, 0))
                bnode = redo == 0 ? node : (node << 1) | (N)((redo & 1u) ? 0u : 1u);
            // (the round keys by scalar adds: held, they would not all fit)
            const dev::Words wd = dev::draw_block(again_value(seed), cell, bnode, redo >> 16);
            double z0, z1;
            walk_pair(wd, z0, z1, C, K, tb);
            // the plain method's timers (cell.cu:106-122): a candidate <= 0
            // gives way to the first candidate > 0 of the daughter's redraw
            // stream (the left daughter's first); after 65535 blocks the timer
            // is the mean (z = 0)
            double tauA = fma(z0, sd, mean), tauB = fma(z1, sd, mean);
            expanded = true;
            if (__builtin_expect(redoing != 0 || __ballot(!(tauA > 0.0) || !(tauB > 0.0)) != 0, 0)) {
                const bool okA = tauA > 0.0, okB = tauB > 0.0;
                // the timers of a lane that waits lie in LDS
                if (redo == 0) {
                    redo = (okA ? 0u : 1u) | (okB ? 0u : 2u);
                    if (redo) {
                        held[0] = z0;
                        held[1] = z1;
                        redo |= 0x10000u;
                        expanded = false;
                    }
                } else {
                    const uint32_t left = redo & 1u;
                    expanded = false;
                    if (okA || okB || (redo >> 16) >= 65535u) {
                        const double v = okA ? z0 : okB ? z1 : 0.0;
                        z0 = left ? v : held[0];
                        z1 = left ? held[1] : v;
                        redo = (redo & (left ? 2u : 0u)) | 0x10000u;
                        if ((redo & 3u) == 0u) {
                            redo = 0u;
                            expanded = true;
                            tauA = fma(z0, sd, mean);
                            tauB = fma(z1, sd, mean);
                        } else {
                            held[0] = z0;
                        }
                    } else {
                        redo += 0x10000u;
                    }
                }
                since += expanded ? 0u : 1u;
            }
            const uint32_t k1 = k + 1;
            const double sA = s + tauA, sB = s + tauB;
            const uint32_t at = tbl + __umul24(k1, TW);
            double gv = 0.0;
            if (Grad && (all_in || tbl != kNoWindow))
                gv = *(LdsDouble *)(uintptr_t)at;
            const double dA = sigmoid_scaled(t_max - sA, ib, C), dB = sigmoid_scaled(t_max - sB, ib, C);
            const double eA = 1.0 - dA, eB = 1.0 - dB, e2 = eA + eB;
            double a1 = 0.0, bA = 0.0, bB = 0.0, vm = 0.0, vs = 0.0;
            const double vh = W * e2;
            if constexpr (Tan) {
                // beta times the derivative of the recorded W (1 - d) in mean_j,
                // sd_j: W ((1 - d) beta dlogW/dtheta + d (1 - d) ds/dtheta)
                a1 = u1 + (double)k1;
                bA = b + z0;
                bB = b + z1;
                const double qA = dA * eA, qB = dB * eB;
                vm = W * fma(e2, gm, (qA + qB) * a1);
                vs = W * fma(e2, gs, fma(qA, bA, qB * bB));
            }
            frames_read();
            if (expanded) {
                if (all_in || tbl != kNoWindow) {
                    if constexpr (!Grad) {
                        lds_add(at, vh);
                        if constexpr (Jac) {
                            lds_add(at + 8, vm);
                            lds_add(at + 16, vs);
                        }
                    }
                } else {
                    const uint64_t e = set_again().h_base + (uint64_t)(rowt & 0xFFFFFFu) * KT + (rowt >> 24) + (uint64_t)k1 * T;
                    if constexpr (Grad) {
                        gv = args_again().g[e];
                    } else {
                        const double p = theta[2 * T + (rowt >> 24)];
                        unsafeAtomicAdd(args_again().h + e, p * vh);
                        if constexpr (Jac) {
                            const double p = theta[2 * T + (rowt >> 24)] * ib;
                            unsafeAtomicAdd(args_again().jac + e, p * vm);
                            unsafeAtomicAdd(args_again().jac + args_again().h_total + e, p * vs);
                        }
                    }
                }
                if constexpr (Grad) {
                    acc_m = fma(gv, vm, acc_m);
                    acc_s = fma(gv, vs, acc_s);
                    acc_p = fma(gv, vh, acc_p);
                }
                const double WA = W * dA, WB = W * dB;
                const bool can = k1 < kcap;
                const bool expA = can && WA >= kRelaxEps, expB = can && WB >= kRelaxEps;
                push = expA && expB;
                // next: the left daughter, else the lowest pending level (the
                // right daughter's if it is expanded, else F's)
                const uint32_t fl = low_bit(pend);
                const N right = (N)(expA ? 0u : 1u);
                const uint32_t sh = ((int)expA | (int)expB) ? 0u : fl + 1u;
                node = ((node << 1) >> sh) | right;
                pend = (((pend << 1) | (N)(expB ? 1u : 0u)) >> sh) & ~right;
                if (expA) {
                    asm volatile("");  // (a branch: the moves are masked, where selects take two each)
                    if (expB) {
                        if (__builtin_amdgcn_inverse_ballot_w64(dirty)) {
                            store_frame(k - fl, F_s, F_w, F_b, F_gm, F_gs);  // F to its level
                        }
                        F_s = sB;
                        F_w = WB;
                        if constexpr (Tan) {
                            F_b = bB;
                            F_gm = fma(-eB, a1, gm);
                            F_gs = fma(-eB, bB, gs);
                        }
                    }
                    s = sA;
                    W = WA;
                    if constexpr (Tan) {
                        gm = fma(-eA, a1, gm);
                        gs = fma(-eA, bA, gs);
                        b = bA;
                    }
                } else if (expB) {
                    asm volatile("");
                    s = sB;
                    W = WB;
                    if constexpr (Tan) {
                        gm = fma(-eB, a1, gm);
                        gs = fma(-eB, bB, gs);
                        b = bB;
                    }
                } else {
                    asm volatile("");
                    s = F_s;
                    W = F_w;
                    if constexpr (Tan) {
                        gm = F_gm;
                        gs = F_gs;
                        b = F_b;
                    }
                    pop = true;
                    if (pend == 0) {
                        end_walk();
                        if (shared && !counted)
                            atomicAdd(&origin_exp[origin[lane]], steps - since);
                    }
                }
                k = k1 - sh;
            }
        }
        redoing = __ballot(redo != 0);
        const uint64_t done = busy & ~over & ~redoing;
        popped = __ballot(pop);
        dirty = (dirty & ~popped) | __ballot(push);
        w_exp += (uint64_t)__popcll(done);
    }

    for (int o = 32; o > 0; o >>= 1)
        n_cut += __shfl_xor(n_cut, o);
    if (lane == 0) {
        atomicAdd((unsigned long long *)(cursor + 2), (unsigned long long)w_exp);
        if (n_cut)
            atomicAdd(cursor + 1, n_cut);
    }
    __syncthreads();
    if (tid == 0) {
        unsigned long long *count = args_again().expansions + (seg % kCountCopies) * kCountWords;
        atomicAdd(count, *(unsigned long long *)(cursor + 2));
        if (cursor[1]) {
            atomicAdd(count + 1, (unsigned long long)cursor[1]);
            if (args_again().set_cuts)
                atomicAdd(args_again().set_cuts + set_id, (unsigned long long)cursor[1]);
        }
    }
    if constexpr (Grad) {
        for (uint32_t i = tid; i < 3 * T; i += kWalkThreads) {
            // dL/dmean and dL/dsd carry p_j / beta
            double v = gsum[i];
            for (uint32_t k = 1; k < sums; ++k)
                v += gsum[k * 3 * T + i];
            v *= (i < 2 * T ? theta[2 * T + i % T] * ib : 1.0);
            if (v != 0.0)
                unsafeAtomicAdd(args_again().grad + set_again().theta_base + i, v);
        }
    } else {
        // p_j and 1 / beta multiply the sums.  Where p_j is not finite, an entry
        // whose records are all exactly 0 (the sigmoid 1) is not 0 either: the
        // product reaches every entry that the row's walks of type j may record
        // in.
        const uint32_t n_prolif_w = set_again().n_prolif;
        auto may_record = [&](uint32_t e) {
            const uint32_t gen = e % KT / T, info = args_again().row_info[w_lo + e / KT];
            bool walks = false;
            for (uint32_t q = 0; q < n_prolif_w; ++q)
                walks = walks || prolif[q] == e % T;
            return walks && gen <= (info & 255u) && (gen > 0 || ((info >> 8) & 1u) != 0);
        };
        for (uint32_t i = tid; i < kParts * win_n; i += kWalkThreads) {
            double v = win[i];
            for (uint32_t k = 1; k < copies; ++k)
                v += win[k * win_stride + i];
            const uint32_t e = i / kParts, part = i - e * kParts;
            const double p = theta[2 * T + e % T];
            if (v != 0.0 || (!(fabs(p) <= 0x1.fffffffffffffp1023) && may_record(e))) {
                double *dst = part == 0 ? args_again().h : args_again().jac + (uint64_t)(part - 1) * args_again().h_total;
                unsafeAtomicAdd(dst + h0 + e, v * p * (part ? ib : 1.0));
            }
        }
    }
}

// Clears up to three ranges in one launch.
__global__ __launch_bounds__(256) void relaxed_clear_kernel(unsigned long long *p0, uint64_t n0, unsigned long long *p1,
                                                            uint64_t n1, unsigned long long *p2, uint64_t n2)
{
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n0 + n1 + n2; i += (uint64_t)gridDim.x * 256) {
        if (i < n0)
            p0[i] = 0ull;
        else if (i < n0 + n1)
            p1[i - n0] = 0ull;
        else
            p2[i - n0 - n1] = 0ull;
    }
}

hipError_t clear_ranges(void *p0, uint64_t n0, void *p1, uint64_t n1, void *p2, uint64_t n2, hipStream_t st)
{
    const uint64_t blocks = (n0 + n1 + n2 + 255) / 256;
    if (blocks == 0)
        return hipSuccess;
    hipLaunchKernelGGL(relaxed_clear_kernel, dim3((unsigned)std::min<uint64_t>(blocks, 4096)), dim3(256), 0, st,
                       (unsigned long long *)p0, n0, (unsigned long long *)p1, n1, (unsigned long long *)p2, n2);
    return hipGetLastError();
}

thread_local hipError_t g_relaxed_hip = hipSuccess;

#define RELAX_TRY(expr)                      \
    do {                                     \
        hipError_t e_ = (expr);              \
        if (e_ != hipSuccess) {              \
            g_relaxed_hip = e_;              \
            return PROCELL_E_HIP;            \
        }                                    \
    } while (0)

// Expected expansions of one walk of a type in a row with this generation
// cap: its root and, per generation, the nodes whose completion time s lies at
// most 34.5 beta past t_max (beyond it d < 1e-15).  s_k is taken as normal (as
// in the plain method's cost_caps).  Only used to balance the segments.
double walk_cost(uint32_t kcap, double t_max, double beta, double mean, double sd)
{
    double e = 1.0;
    for (uint32_t k = 0; k < kcap; ++k) {
        const double mu = (1.5 + k) * mean;
        const double var = (7.0 / 3.0 + k) * sd * sd + mean * mean / 12.0;
        const double z = (t_max + 34.5 * beta - mu) / sqrt(var > 0.0 ? var : 1e-300);
        const double prob = 0.5 * erfc(-z * 0.70710678118654752);
        e += ldexp(prob, (int)k);
        if (!(prob >= 1e-12))
            break;
    }
    return e;
}

int relaxed_device(int device, int *n_cu)
{
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0 || device < 0 || device >= count)
        return PROCELL_E_NO_DEVICE;
    RELAX_TRY(hipSetDevice(device));
    hipDeviceProp_t prop;
    RELAX_TRY(hipGetDeviceProperties(&prop, device));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return PROCELL_E_NO_DEVICE;
    *n_cu = prop.multiProcessorCount;
    return PROCELL_OK;
}

using WalkKernel = void (*)(RelaxArgs);

// The kernel of a pass: 32-bit heap indices and level masks for trees of at
// most 31 generations.
WalkKernel walk_kernel_of(int mode, uint32_t kdim)
{
    static const WalkKernel narrow[3] = {walk_kernel<kForward, uint32_t>, walk_kernel<kAdjoint, uint32_t>,
                                         walk_kernel<kJacobian, uint32_t>};
    static const WalkKernel wide[3] = {walk_kernel<kForward, uint64_t>, walk_kernel<kAdjoint, uint64_t>,
                                       walk_kernel<kJacobian, uint64_t>};
    return kdim <= 32 ? narrow[mode] : wide[mode];
}

// Device tables of a relaxed plan over n parameter sets.
struct RelaxCore {
    int device = 0;
    uint32_t n_sets = 0;
    std::vector<Setup> setups;
    std::vector<RelaxSet> sets;
    std::vector<uint32_t> quiet_flag;  // per type of every set: 1 = quiescent
    uint32_t n_segments = 0;
    uint32_t per_launch = 0;   // segments that the stacks are for
    size_t lds_bytes[3] = {0, 0, 0};  // of the walk kernel, per WalkMode
    uint64_t h_total = 0;      // tally entries of all sets
    uint32_t types_total = 0;  // types of all sets
    RelaxArgs args{};
    void *d_block = nullptr;
    double *d_stack = nullptr;
};

void core_free(RelaxCore &c)
{
    (void)hipSetDevice(c.device);
    if (c.d_block)
        (void)hipFree(c.d_block);
    if (c.d_stack)
        (void)hipFree(c.d_stack);
    c.d_block = nullptr;
    c.d_stack = nullptr;
}

// Validates the sets, cuts their initial cells into the workgroups' segments
// and uploads the tables.
int core_build(RelaxCore &c, const procell_params *ps, uint32_t n, double beta, bool want_bins)
{
    if (!ps || n == 0)
        return PROCELL_E_INVALID;
    if (!(beta > 0.0) || !isfinite(beta))
        return PROCELL_E_INVALID;
    for (uint32_t i = 1; i < n; ++i)
        if (ps[i].device != ps[0].device)
            return PROCELL_E_INVALID;
    c.n_sets = n;
    c.setups.resize(n);
    for (uint32_t i = 0; i < n; ++i) {
        const int rc = build_setup(&ps[i], c.setups[i], want_bins, false);
        if (rc != PROCELL_OK)
            return rc;
    }
    int n_cu = 0;
    {
        const int rc = relaxed_device(ps[0].device, &n_cu);
        if (rc != PROCELL_OK)
            return rc;
    }
    c.device = ps[0].device;

    // ---- concatenation ----
    std::vector<uint32_t> prolif, quiet, row_start, row_info;
    c.sets.resize(n);
    uint64_t cells = 0;
    uint32_t rows = 0, kdim_max = 1, t_max_types = 1;
    std::vector<uint64_t> units(n);
    for (uint32_t i = 0; i < n; ++i) {
        const Setup &s = c.setups[i];
        RelaxSet &S = c.sets[i];
        memset(&S, 0, sizeof S);
        S.seed = ps[i].seed;
        S.t_max = ps[i].t_max;
        S.cell_base = cells;
        S.h_base = c.h_total;
        S.row_base = rows;
        S.n_rows = (uint32_t)s.v.size();
        S.kdim = (uint32_t)s.kmax + 1;
        S.n_types = std::max(1u, ps[i].n_types);
        S.theta_base = 3 * c.types_total;
        S.prolif_base = (uint32_t)prolif.size();
        S.quiet_base = (uint32_t)quiet.size();
        for (uint32_t j = 0; j < ps[i].n_types; ++j) {
            const bool q = ps[i].types[j].mean < 0.0;
            (q ? quiet : prolif).push_back(j);
            c.quiet_flag.push_back(q ? 1u : 0u);
        }
        for (uint32_t j = ps[i].n_types; j < S.n_types; ++j)
            c.quiet_flag.push_back(1u);
        S.n_prolif = (uint32_t)prolif.size() - S.prolif_base;
        S.n_quiet = (uint32_t)quiet.size() - S.quiet_base;
        for (uint32_t r = 0; r < S.n_rows; ++r) {
            row_start.push_back((uint32_t)(cells + s.start[r]));
            row_info.push_back(s.row_info[r]);
        }
        units[i] = s.n_cells * (uint64_t)S.n_prolif;
        cells += s.n_cells;
        if (cells > kMaxCells)
            return PROCELL_E_TOO_MANY_CELLS;
        rows += S.n_rows;
        c.h_total += (uint64_t)S.n_rows * S.kdim * S.n_types;
        c.types_total += S.n_types;
        kdim_max = std::max(kdim_max, S.kdim);
        t_max_types = std::max(t_max_types, S.n_types);
    }
    row_start.push_back((uint32_t)cells);

    // ---- segments ----
    // Windows: what is left of a workgroup's share of the LDS beside its
    // fixed part (kept to the rows that a segment has, below)
    uint32_t win_cap[3];
    int occ = 0;
    for (int m = 0; m < 3; ++m) {
        const size_t fixed = (size_t)walk_lds(t_max_types, m).fixed;
        win_cap[m] = fixed < kWalkLds ? (uint32_t)((kWalkLds - fixed) / 8) : 0u;
        int o = 0;
        RELAX_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&o, walk_kernel_of(m, kdim_max), (int)kWalkThreads,
                                                               fixed + win_cap[m] * 8));
        occ = m == 0 ? o : std::min(occ, o);
    }
    if (occ < 1)
        return PROCELL_E_HIP;
    if (ps[0].tuning.blocks_per_cu)
        occ = std::min(occ, (int)ps[0].tuning.blocks_per_cu);
    const uint32_t factor = n > 1 ? kMultiSetFactor : 1u;
    const uint64_t budget = (uint64_t)occ * (uint64_t)n_cu * factor;
    std::vector<std::vector<double>> cell_cost(n);
    std::vector<double> set_cost(n, 0.0);
    double all_cost = 0.0;
    for (uint32_t i = 0; i < n; ++i) {
        const Setup &s = c.setups[i];
        const RelaxSet &S = c.sets[i];
        cell_cost[i].assign(S.n_rows, 1.0);
        if (!units[i])
            continue;
        std::vector<double> by_cap(S.kdim, -1.0);
        for (uint32_t r = 0; r < S.n_rows; ++r) {
            const uint32_t cap = s.row_info[r] & 255u;
            double &cr = by_cap[cap];
            if (cr < 0.0) {
                cr = 0.0;
                for (uint32_t q = 0; q < S.n_prolif; ++q) {
                    const procell_type &ty = ps[i].types[prolif[S.prolif_base + q]];
                    cr += walk_cost(cap, ps[i].t_max, beta, ty.mean, ty.sd);
                }
            }
            cell_cost[i][r] = cr;
            set_cost[i] += cr * (double)(s.start[r + 1] - s.start[r]);
        }
        all_cost += set_cost[i];
        c.sets[i].deep = set_cost[i] >= kDeepWalk * (double)units[i] ? 1u : 0u;
    }
    std::vector<Segment> segs;
    for (uint32_t i = 0; i < n; ++i) {
        const Setup &s = c.setups[i];
        if (!units[i]) {
            // no walks: the quiescent types' records alone, 4096 rows a segment
            for (size_t r = 0; r < s.v.size(); r += 4096) {
                const size_t r1 = std::min(r + 4096, s.v.size());
                segs.push_back(Segment{i, (uint32_t)s.start[r], (uint32_t)(r1 < s.v.size() ? s.start[r1] : s.n_cells),
                                       c.sets[i].row_base + (uint32_t)r, c.sets[i].row_base + (uint32_t)r1 - 1});
            }
            continue;
        }
        const double share = all_cost > 0.0 ? set_cost[i] / all_cost * (double)budget : 1.0;
        const uint64_t most = (units[i] + kMinWalks - 1) / kMinWalks;
        split_set(s, cell_cost[i], std::max<uint64_t>(1, std::min((uint64_t)floor(share + 0.5), most)), i,
                  c.sets[i].row_base, kMaxSegmentUnits / ((c.sets[i].n_prolif + 63) / 64), segs);
    }
    if (segs.size() > 0x7FFFFFFFull)
        return PROCELL_E_TOO_MANY_CELLS;
    c.n_segments = (uint32_t)segs.size();
    c.args.even_ends = c.n_segments <= (uint64_t)occ * (uint64_t)n_cu ? 1u : 0u;
    std::vector<uint32_t> seg_set, seg_cell, seg_row;
    uint64_t entries = 0;  // most entries of a segment's rows
    for (const Segment &p : segs) {
        seg_set.push_back(p.set);
        seg_cell.insert(seg_cell.end(), {p.c0, p.c1});
        seg_row.insert(seg_row.end(), {p.r0, p.r1});
        entries = std::max<uint64_t>(entries, (uint64_t)(p.r1 - p.r0 + 1) * c.sets[p.set].kdim * c.sets[p.set].n_types);
    }
    // each segment's window over the rows that take most of its cost
    std::vector<uint32_t> seg_win;
    for (int m = 0; m < 3; ++m) {
        for (const Segment &p : segs) {
            const Setup &s = c.setups[p.set];
            const RelaxSet &S = c.sets[p.set];
            const uint32_t len = std::max(1u, win_cap[m] / (S.kdim * S.n_types * (m == kJacobian ? 3 : 1)));
            auto cost = [&](uint32_t row) {  // of the segment's cells in a row
                const uint32_t r = row - S.row_base;
                return cell_cost[p.set][r] * (double)(std::min<uint64_t>(s.start[r + 1], p.c1) - std::max<uint64_t>(s.start[r], p.c0));
            };
            uint32_t at = p.r0;
            double in = 0.0, best = -1.0;
            for (uint32_t r = p.r0; r <= p.r1; ++r) {
                in += cost(r);
                if (r - p.r0 >= len)
                    in -= cost(r - len);
                if (in > best && (r - p.r0 + 1 >= len || r == p.r1)) {
                    best = in;
                    at = r - p.r0 + 1 >= len ? r + 1 - len : p.r0;
                }
            }
            seg_win.push_back(at);
        }
    }
    for (int m = 0; m < 3; ++m) {
        c.args.win_doubles[m] = (uint32_t)std::min<uint64_t>(win_cap[m], (entries * (m == kJacobian ? 3 : 1) + 1) * (m == kAdjoint ? 1 : 8));
        c.lds_bytes[m] = (size_t)walk_lds(t_max_types, m).fixed + (size_t)c.args.win_doubles[m] * 8;
    }

    // ---- upload ----
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t o = off;
        off = (off + bytes + 255) / 256 * 256;
        return o;
    };
    const size_t o_sets = take(c.sets.size() * sizeof(RelaxSet));
    const size_t o_ss = take(seg_set.size() * 4 + 4), o_sc = take(seg_cell.size() * 4 + 4);
    const size_t o_sw = take(seg_win.size() * 4 + 4);
    const size_t o_sr = take(seg_row.size() * 4 + 4), o_rs = take(row_start.size() * 4);
    const size_t o_ri = take(row_info.size() * 4 + 4);
    const size_t o_pr = take(prolif.size() * 4 + 4), o_qu = take(quiet.size() * 4 + 4);
    const size_t o_ex = take((kCountCopies * kCountWords + (size_t)n) * 8);  // counters, walks cut per set
    if (hipMalloc(&c.d_block, off) != hipSuccess)
        return PROCELL_E_OUT_OF_MEMORY;
    char *base = (char *)c.d_block;
    auto up = [&](size_t o, const void *src, size_t bytes) {
        return bytes ? hipMemcpy(base + o, src, bytes, hipMemcpyHostToDevice) : hipSuccess;
    };
    RELAX_TRY(up(o_sets, c.sets.data(), c.sets.size() * sizeof(RelaxSet)));
    RELAX_TRY(up(o_ss, seg_set.data(), seg_set.size() * 4));
    RELAX_TRY(up(o_sc, seg_cell.data(), seg_cell.size() * 4));
    RELAX_TRY(up(o_sw, seg_win.data(), seg_win.size() * 4));
    RELAX_TRY(up(o_sr, seg_row.data(), seg_row.size() * 4));
    RELAX_TRY(up(o_rs, row_start.data(), row_start.size() * 4));
    RELAX_TRY(up(o_ri, row_info.data(), row_info.size() * 4));
    RELAX_TRY(up(o_pr, prolif.data(), prolif.size() * 4));
    RELAX_TRY(up(o_qu, quiet.data(), quiet.size() * 4));
    RelaxArgs &a = c.args;
    a.beta = beta;
    a.n_sets = n;
    a.n_rows = rows;
    a.n_segments = c.n_segments;
    a.kdim_max = kdim_max;
    a.sets = (const RelaxSet *)(base + o_sets);
    a.seg_set = (const uint32_t *)(base + o_ss);
    a.seg_cell = (const uint32_t *)(base + o_sc);
    a.seg_win = (const uint32_t *)(base + o_sw);
    a.seg_row = (const uint32_t *)(base + o_sr);
    a.row_start = (const uint32_t *)(base + o_rs);
    a.row_info = (const uint32_t *)(base + o_ri);
    a.prolif = (const uint32_t *)(base + o_pr);
    a.quiet = (const uint32_t *)(base + o_qu);
    a.expansions = (unsigned long long *)(base + o_ex);
    a.set_cuts = a.expansions + kCountCopies * kCountWords;
    a.h_total = c.h_total;
    if (c.n_segments) {
        const size_t seg_bytes = (size_t)kWalkThreads * (kdim_max + 1) * kFrameBytes;
        c.per_launch = (uint32_t)std::min<uint64_t>(c.n_segments, kStackBytes / seg_bytes);
        if (hipMalloc((void **)&c.d_stack, c.per_launch * seg_bytes) != hipSuccess)
            return PROCELL_E_OUT_OF_MEMORY;
        a.stack = c.d_stack;
    }
    return PROCELL_OK;
}

// Enqueues one pass of a WalkMode (the caller has cleared h, the Jacobian or
// the gradient, and the expansion counter).
hipError_t core_launch(const RelaxCore &c, const RelaxArgs &a, int mode, hipStream_t st)
{
    RelaxArgs part = a;
    for (part.seg_first = 0; part.seg_first < c.n_segments; part.seg_first += c.per_launch) {
        const uint32_t n = std::min(c.per_launch, c.n_segments - part.seg_first);
        hipLaunchKernelGGL(walk_kernel_of(mode, a.kdim_max), dim3(n), dim3(kWalkThreads), c.lds_bytes[mode], st, part);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// Batched calibration: per set, the squared L2 distance between the
// normalised relaxed histogram (h summed over types, (row, generation)
// entries merged into the output bins value / 2^k) and a normalised target,
// its cotangent dL/dh, and an Adam step on (log mean, log sd, proportion
// logits).
// ---------------------------------------------------------------------------
struct CalibSet {
    uint32_t bin_base;   // first output bin of the set (targets, per-bin scratch)
    uint32_t n_bins;
    uint32_t ptr_base;   // first entry of the set's bin -> entries CSR offsets (n_bins + 1 of them)
    uint32_t ent_base;   // first (row, generation) entry of the set in ent_bin
    uint32_t n_ent;      // rows x kdim
    uint32_t pad[3];
};

struct CalibArgs {
    uint32_t n_sets;
    uint32_t pad;
    double lr, beta1, beta2, eps;
    const RelaxSet *sets;
    const CalibSet *csets;
    const uint32_t *bin_ptr;   // CSR offsets into bin_ent, per set
    const uint32_t *bin_ent;   // set-local entry ids (row * kdim + k) of each bin
    const int32_t *ent_bin;    // bin of each (row, generation) entry, or -1
    const double *q;           // normalised targets per bin
    const uint32_t *quiet_flag;  // per type of every set
    double *hb;                // per-bin scratch: relaxed histogram, then dL/dhb
    double *loss;              // [n_sets]
    const double *h;
    double *g;                 // dL/dh, written for the adjoint pass (null with jac)
    double *grad;              // dL/dtheta per set [3][T]
    const double *jac;         // dh/dmean | dh/dsd, each laid out like h; null: adjoint route
    uint64_t h_total;
    double *x;                 // per set [3][T]: log mean, log sd, logits
    double *m1, *m2;           // Adam moments, layout of x
    double *theta;             // per set [3][T]
    unsigned long long *step;  // [1] Adam steps taken
};

__device__ double block_sum_256(double v, double *red)
{
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o);
    const uint32_t wv = threadIdx.x >> 6, ln = threadIdx.x & 63u;
    __syncthreads();
    if (ln == 0)
        red[wv] = v;
    __syncthreads();
    double s = 0.0;
    for (uint32_t i = 0; i < (blockDim.x >> 6); ++i)
        s += red[i];
    return s;
}

// One workgroup (256 threads) per set.  L = sum_b (hb_b / S - q_b)^2 with
// S = sum_b hb_b; dL/dhb_a = (2 / S) (r_a - sum_b r_b hb_b / S), r = hb / S - q.
__global__ __launch_bounds__(256) void calib_loss_kernel(CalibArgs c)
{
    __shared__ double red[4];
    const uint32_t set = blockIdx.x;
    const RelaxSet &S = c.sets[set];
    const CalibSet &C = c.csets[set];
    const uint32_t T = S.n_types;
    const double *h = c.h + S.h_base;
    double *hb = c.hb + C.bin_base;
    const uint32_t *ptr = c.bin_ptr + C.ptr_base;
    double part = 0.0;
    for (uint32_t b = threadIdx.x; b < C.n_bins; b += blockDim.x) {
        double v = 0.0;
        for (uint32_t e = ptr[b]; e < ptr[b + 1]; ++e) {
            const uint64_t at = (uint64_t)c.bin_ent[e] * T;
            for (uint32_t j = 0; j < T; ++j)
                v += h[at + j];
        }
        hb[b] = v;
        part += v;
    }
    const double tot = block_sum_256(part, red);
    const double inv = tot > 0.0 ? 1.0 / tot : 0.0;
    double pl = 0.0, pc = 0.0;
    for (uint32_t b = threadIdx.x; b < C.n_bins; b += blockDim.x) {
        const double p = hb[b] * inv;
        const double r = p - c.q[C.bin_base + b];
        pl += r * r;
        pc += r * p;
        hb[b] = r;
    }
    const double L = block_sum_256(pl, red);
    const double Cc = block_sum_256(pc, red);
    for (uint32_t b = threadIdx.x; b < C.n_bins; b += blockDim.x)
        hb[b] = tot > 0.0 ? 2.0 * inv * (hb[b] - Cc) : 0.0;
    __syncthreads();
    if (threadIdx.x == 0)
        c.loss[set] = L;
    if (!c.jac) {
        double *g = c.g + S.h_base;
        for (uint32_t e = threadIdx.x; e < C.n_ent; e += blockDim.x) {
            const int32_t b = c.ent_bin[C.ent_base + e];
            const double gv = b >= 0 ? hb[b] : 0.0;
            for (uint32_t j = 0; j < T; ++j)
                g[(uint64_t)e * T + j] = gv;
        }
        return;
    }
    // Jacobian route: dL/dtheta = J^T dL/dh.  An entry depends on its own
    // type's parameters only, and h is linear in p_j (dh/dp_j = h / p_j; at
    // p_j = 0 the entry is left 0: the Adam step multiplies it by p_j).
    const double *jm = c.jac + S.h_base, *js = c.jac + c.h_total + S.h_base;
    const double *th = c.theta + S.theta_base;
    double *gr = c.grad + S.theta_base;
    for (uint32_t j = 0; j < T; ++j) {
        double sm = 0.0, ss = 0.0, sp = 0.0;
        for (uint32_t e = threadIdx.x; e < C.n_ent; e += blockDim.x) {
            const int32_t b = c.ent_bin[C.ent_base + e];
            if (b < 0)
                continue;
            const double gv = hb[b];
            const uint64_t at = (uint64_t)e * T + j;
            sm += gv * jm[at];
            ss += gv * js[at];
            sp += gv * h[at];
        }
        sm = block_sum_256(sm, red);
        ss = block_sum_256(ss, red);
        sp = block_sum_256(sp, red);
        if (threadIdx.x == 0) {
            const double pj = th[2 * T + j];
            gr[j] = sm;
            gr[T + j] = ss;
            gr[2 * T + j] = pj > 0.0 ? sp / pj : 0.0;
        }
    }
}

// theta of one set from its unconstrained parameters.
__device__ void calib_theta(const CalibArgs &c, const RelaxSet &S)
{
    const uint32_t T = S.n_types, tb = S.theta_base;
    const uint32_t *qf = c.quiet_flag + tb / 3;
    double mx = c.x[tb + 2 * T];
    for (uint32_t j = 1; j < T; ++j)
        mx = fmax(mx, c.x[tb + 2 * T + j]);
    double sum = 0.0;
    for (uint32_t j = 0; j < T; ++j)
        sum += exp(c.x[tb + 2 * T + j] - mx);
    for (uint32_t j = 0; j < T; ++j) {
        c.theta[tb + j] = qf[j] ? -1.0 : exp(c.x[tb + j]);
        c.theta[tb + T + j] = qf[j] ? -1.0 : exp(c.x[tb + T + j]);
        c.theta[tb + 2 * T + j] = exp(c.x[tb + 2 * T + j] - mx) / sum;
    }
}

__device__ __forceinline__ void adam_update(double &x, double &m, double &v, double gr, const CalibArgs &c,
                                            double bc1, double bc2)
{
    m = c.beta1 * m + (1.0 - c.beta1) * gr;
    v = c.beta2 * v + (1.0 - c.beta2) * gr * gr;
    const double denom = sqrt(v) / sqrt(bc2) + c.eps;
    x = x - (c.lr / bc1) * (m / denom);
}

// One workgroup; thread s updates set s (and s + blockDim, ...).  Chain rule
// to the unconstrained parameters: d/dlog mean = dL/dmean mean, d/dlog sd =
// dL/dsd sd, d/dlogit_j = p_j (dL/dp_j - sum_k p_k dL/dp_k).
__global__ __launch_bounds__(256) void calib_adam_kernel(CalibArgs c)
{
    const unsigned long long t = c.step[0] + 1ull;
    const double bc1 = 1.0 - pow(c.beta1, (double)t), bc2 = 1.0 - pow(c.beta2, (double)t);
    for (uint32_t set = threadIdx.x; set < c.n_sets; set += blockDim.x) {
        const RelaxSet &S = c.sets[set];
        const uint32_t T = S.n_types, tb = S.theta_base;
        const uint32_t *qf = c.quiet_flag + tb / 3;
        const double *th = c.theta + tb;
        const double *gr = c.grad + tb;
        double dot = 0.0;
        for (uint32_t j = 0; j < T; ++j)
            dot += th[2 * T + j] * gr[2 * T + j];
        for (uint32_t j = 0; j < T; ++j) {
            if (!qf[j]) {
                adam_update(c.x[tb + j], c.m1[tb + j], c.m2[tb + j], gr[j] * th[j], c, bc1, bc2);
                adam_update(c.x[tb + T + j], c.m1[tb + T + j], c.m2[tb + T + j], gr[T + j] * th[T + j], c, bc1,
                            bc2);
                // keep sd <= 0.8 mean (kLogMaxSdRatio): the expected tree
                // grows quickly beyond it
                c.x[tb + T + j] = fmin(c.x[tb + T + j], c.x[tb + j] + kLogMaxSdRatio);
            }
            const uint32_t z = tb + 2 * T + j;
            adam_update(c.x[z], c.m1[z], c.m2[z], th[2 * T + j] * (gr[2 * T + j] - dot), c, bc1, bc2);
        }
        calib_theta(c, S);
    }
    __syncthreads();
    if (threadIdx.x == 0)
        c.step[0] = t;
}

__global__ void calib_init_kernel(CalibArgs c)
{
    for (uint32_t set = blockIdx.x * blockDim.x + threadIdx.x; set < c.n_sets; set += gridDim.x * blockDim.x)
        calib_theta(c, c.sets[set]);
}

}  // namespace
}  // namespace procell

using namespace procell;

struct procell_relaxed {
    RelaxCore core;
};

struct procell_calib {
    RelaxCore core;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    CalibArgs cargs{};
    RelaxArgs fwd{}, bwd{};  // fwd is the Jacobian pass without a cell stride
    bool jac_route = false;
    void *d_calib = nullptr;        // tables of the loss kernel
    void *d_state = nullptr;        // x, m1, m2, theta, grad, h, g, per-bin scratch, loss, step
    unsigned long long *d_clear = nullptr;  // h | grad | expansion counter: cleared every step
    size_t clear_words = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
};

namespace {

void destroy_relaxed(procell_relaxed *r)
{
    if (!r)
        return;
    core_free(r->core);
    delete r;
}

void destroy_calib(procell_calib *c)
{
    if (!c)
        return;
    (void)hipSetDevice(c->core.device);
    if (c->graph_exec)
        (void)hipGraphExecDestroy(c->graph_exec);
    if (c->graph)
        (void)hipGraphDestroy(c->graph);
    if (c->d_calib)
        (void)hipFree(c->d_calib);
    if (c->d_state)
        (void)hipFree(c->d_state);
    if (c->own_stream && c->stream)
        (void)hipStreamDestroy(c->stream);
    core_free(c->core);
    delete c;
}

// Expansions and walks cut of a pass, from its device counters.
hipError_t read_counts(const unsigned long long *counts, uint64_t &expansions, uint64_t &cut)
{
    unsigned long long c[kCountCopies * kCountWords];
    const hipError_t e = hipMemcpy(c, counts, sizeof c, hipMemcpyDeviceToHost);
    expansions = cut = 0;
    for (uint32_t i = 0; i < kCountCopies && e == hipSuccess; ++i) {
        expansions += c[i * kCountWords];
        cut += c[i * kCountWords + 1];
    }
    return e;
}

int relaxed_call(procell_relaxed *r, int mode, const double *theta, double *h, const double *g, double *gr,
                 double *jac, void *stream)
{
    RELAX_TRY(hipSetDevice(r->core.device));
    hipStream_t st = (hipStream_t)stream;  // NULL: the default stream
    RelaxArgs a = r->core.args;
    a.theta = theta;
    a.h = h;
    a.g = g;
    a.grad = gr;
    a.jac = jac;
    const uint64_t n_h = r->core.h_total, n_counts = kCountCopies * kCountWords + a.n_sets;
    if (mode == kAdjoint)
        RELAX_TRY(clear_ranges(a.expansions, n_counts, gr, 3ull * r->core.types_total, nullptr, 0, st));
    else
        RELAX_TRY(clear_ranges(a.expansions, n_counts, h, n_h, jac, mode == kJacobian ? 2 * n_h : 0, st));
    RELAX_TRY(core_launch(r->core, a, mode, st));
    return PROCELL_OK;
}

// One calibration step.  Without a cell stride: clear, the Jacobian pass (h
// and dh/dtheta in one walk), loss and gradient J^T dL/dh, Adam.  With one:
// clear, forward, loss and cotangent, adjoint on the next class of cells,
// Adam.
hipError_t calib_enqueue(procell_calib *c, hipStream_t st)
{
    hipError_t e = launch_zero(c->d_clear, c->clear_words, st);
    if (e != hipSuccess)
        return e;
    if ((e = core_launch(c->core, c->fwd, c->jac_route ? kJacobian : kForward, st)) != hipSuccess)
        return e;
    hipLaunchKernelGGL(calib_loss_kernel, dim3(c->core.n_sets), dim3(256), 0, st, c->cargs);
    if ((e = hipGetLastError()) != hipSuccess)
        return e;
    if (!c->jac_route && (e = core_launch(c->core, c->bwd, kAdjoint, st)) != hipSuccess)
        return e;
    hipLaunchKernelGGL(calib_adam_kernel, dim3(1), dim3(256), 0, st, c->cargs);
    return hipGetLastError();
}

}  // namespace

extern "C" {

int procell_relaxed_create(const procell_params *p, double beta, procell_relaxed **out)
{
    if (!p || !out)
        return PROCELL_E_INVALID;
    *out = nullptr;
    if (!(beta > 0.0) || !isfinite(beta))
        return PROCELL_E_INVALID;
    procell_relaxed *r = new (std::nothrow) procell_relaxed();
    if (!r)
        return PROCELL_E_OUT_OF_MEMORY;
    const int rc = core_build(r->core, p, 1, beta, false);
    if (rc != PROCELL_OK) {
        destroy_relaxed(r);
        return rc;
    }
    *out = r;
    return PROCELL_OK;
}

int procell_relaxed_create_batch(const procell_params *sets, uint32_t n_sets, double beta, procell_relaxed **out)
{
    if (!sets || !out || n_sets == 0)
        return PROCELL_E_INVALID;
    *out = nullptr;
    procell_relaxed *r = new (std::nothrow) procell_relaxed();
    if (!r)
        return PROCELL_E_OUT_OF_MEMORY;
    const int rc = core_build(r->core, sets, n_sets, beta, false);
    if (rc != PROCELL_OK) {
        destroy_relaxed(r);
        return rc;
    }
    *out = r;
    return PROCELL_OK;
}

int procell_relaxed_set_shape(const procell_relaxed *r, uint32_t set, uint64_t *h_base, uint64_t *n_rows,
                              uint32_t *kdim, uint32_t *n_types)
{
    if (!r || set >= r->core.n_sets)
        return PROCELL_E_INVALID;
    const RelaxSet &S = r->core.sets[set];
    if (h_base)
        *h_base = S.h_base;
    if (n_rows)
        *n_rows = S.n_rows;
    if (kdim)
        *kdim = S.kdim;
    if (n_types)
        *n_types = S.n_types;
    return PROCELL_OK;
}

int procell_relaxed_shape(const procell_relaxed *r, uint64_t *n_rows, uint32_t *kdim, uint32_t *n_types)
{
    if (!r)
        return PROCELL_E_INVALID;
    const RelaxSet &S = r->core.sets[0];
    if (n_rows)
        *n_rows = S.n_rows;
    if (kdim)
        *kdim = S.kdim;
    if (n_types)
        *n_types = S.n_types;
    return PROCELL_OK;
}

int procell_relaxed_forward(procell_relaxed *r, const double *theta, double *h, void *stream)
{
    if (!r || !theta || !h)
        return PROCELL_E_INVALID;
    return relaxed_call(r, kForward, theta, h, nullptr, nullptr, nullptr, stream);
}

int procell_relaxed_backward(procell_relaxed *r, const double *theta, const double *g, double *grad,
                             void *stream)
{
    if (!r || !theta || !g || !grad)
        return PROCELL_E_INVALID;
    return relaxed_call(r, kAdjoint, theta, nullptr, g, grad, nullptr, stream);
}

int procell_relaxed_jacobian(procell_relaxed *r, const double *theta, double *h, double *jac, void *stream)
{
    if (!r || !theta || !h || !jac)
        return PROCELL_E_INVALID;
    return relaxed_call(r, kJacobian, theta, h, nullptr, nullptr, jac, stream);
}

int procell_relaxed_set_stride(procell_relaxed *r, uint32_t stride, uint32_t phase)
{
    if (!r || stride == 0 || (stride & (stride - 1)) != 0 || stride > (1u << 16))
        return PROCELL_E_INVALID;
    r->core.args.stride_mask = stride - 1;
    r->core.args.phase = phase & (stride - 1);
    return PROCELL_OK;
}

int procell_relaxed_expansions(procell_relaxed *r, uint64_t *n)
{
    if (!r || !n)
        return PROCELL_E_INVALID;
    RELAX_TRY(hipSetDevice(r->core.device));
    RELAX_TRY(hipDeviceSynchronize());
    uint64_t cut = 0;
    RELAX_TRY(read_counts(r->core.args.expansions, *n, cut));
    return cut ? PROCELL_E_DEPTH : PROCELL_OK;
}

int procell_relaxed_set_cuts(procell_relaxed *r, uint64_t *cuts, void *stream)
{
    if (!r || !cuts)
        return PROCELL_E_INVALID;
    RELAX_TRY(hipSetDevice(r->core.device));
    RELAX_TRY(hipMemcpyAsync(cuts, r->core.args.set_cuts, (size_t)r->core.args.n_sets * 8, hipMemcpyDeviceToDevice,
                             (hipStream_t)stream));
    return PROCELL_OK;
}

int procell_relaxed_destroy(procell_relaxed *r)
{
    destroy_relaxed(r);
    return PROCELL_OK;
}

int procell_calib_create(const procell_params *sets, uint32_t n_sets, double beta, const procell_result *targets,
                         const procell_adam *adam, uint32_t cell_stride, procell_calib **out)
{
    if (!sets || !targets || !adam || !out || n_sets == 0)
        return PROCELL_E_INVALID;
    if (cell_stride == 0 || (cell_stride & (cell_stride - 1)) != 0 || cell_stride > (1u << 16))
        return PROCELL_E_INVALID;
    *out = nullptr;
    if (!(adam->lr > 0.0) || !(adam->beta1 >= 0.0 && adam->beta1 < 1.0) || !(adam->beta2 >= 0.0 && adam->beta2 < 1.0) ||
        !(adam->eps > 0.0))
        return PROCELL_E_INVALID;
    procell_calib *c = new (std::nothrow) procell_calib();
    if (!c)
        return PROCELL_E_OUT_OF_MEMORY;
    auto fail = [&](int code) {
        destroy_calib(c);
        return code;
    };
#define CALIB_TRY(expr)                       \
    do {                                      \
        hipError_t e_ = (expr);               \
        if (e_ != hipSuccess) {               \
            g_relaxed_hip = e_;               \
            return fail(PROCELL_E_HIP);       \
        }                                     \
    } while (0)
    int rc = core_build(c->core, sets, n_sets, beta, true);
    if (rc != PROCELL_OK)
        return fail(rc);
    RelaxCore &core = c->core;
    for (uint32_t i = 0; i < n_sets; ++i)
        for (uint32_t j = 0; j < sets[i].n_types; ++j)
            if (sets[i].types[j].mean >= 0.0 && !(sets[i].types[j].mean > 0.0 && sets[i].types[j].sd > 0.0 &&
                                                  sets[i].types[j].proportion > 0.0))
                return fail(PROCELL_E_INVALID);  // log parameters need mean, sd, proportion > 0

    // ---- bins, targets, (row, generation) -> bin maps ----
    std::vector<CalibSet> cs(n_sets);
    std::vector<uint32_t> bin_ptr, bin_ent;
    std::vector<int32_t> ent_bin;
    std::vector<double> q;
    for (uint32_t i = 0; i < n_sets; ++i) {
        const Setup &s = core.setups[i];
        const RelaxSet &S = core.sets[i];
        CalibSet &C = cs[i];
        memset(&C, 0, sizeof C);
        C.bin_base = (uint32_t)q.size();
        C.n_bins = (uint32_t)s.bins.size();
        C.ptr_base = (uint32_t)bin_ptr.size();
        C.ent_base = (uint32_t)ent_bin.size();
        C.n_ent = S.n_rows * S.kdim;
        const procell_result &tr = targets[i];
        if (tr.n_out && (!tr.value || !tr.count))
            return fail(PROCELL_E_INVALID);
        std::vector<double> tq(C.n_bins, 0.0);
        double tsum = 0.0;
        for (uint64_t r = 0; r < tr.n_out; ++r) {
            auto it = std::lower_bound(s.bins.begin(), s.bins.end(), tr.value[r]);
            if (it == s.bins.end() || *it != tr.value[r] || tr.count[r] < 0)
                return fail(PROCELL_E_INVALID);  // a target value outside the set's output bins
            tq[it - s.bins.begin()] += (double)tr.count[r];
            tsum += (double)tr.count[r];
        }
        for (double &x : tq)
            q.push_back(tsum > 0.0 ? x / tsum : 0.0);
        std::vector<std::vector<uint32_t>> members(C.n_bins);
        for (uint32_t r = 0; r < S.n_rows; ++r) {
            const uint32_t kc = s.row_info[r] & 255u;
            const bool ge = ((s.row_info[r] >> 8) & 1u) != 0;
            double f = s.v[r];
            for (uint32_t k = 0; k < S.kdim; ++k) {
                int32_t b = -1;
                if (k <= kc && (k > 0 || ge)) {
                    auto it = std::lower_bound(s.bins.begin(), s.bins.end(), f);
                    if (it != s.bins.end() && *it == f) {
                        b = (int32_t)(it - s.bins.begin());
                        members[b].push_back(r * S.kdim + k);
                    }
                }
                ent_bin.push_back(b);
                f = f / 2;
            }
        }
        for (uint32_t b = 0; b < C.n_bins; ++b) {
            bin_ptr.push_back((uint32_t)bin_ent.size());
            for (uint32_t e : members[b])
                bin_ent.push_back(e);
        }
        bin_ptr.push_back((uint32_t)bin_ent.size());
    }
    // CSR offsets are relative to the whole bin_ent array
    const size_t n_bins_total = q.size();

    // ---- device memory ----
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t o = off;
        off = (off + bytes + 255) / 256 * 256;
        return o;
    };
    const size_t o_cs = take(cs.size() * sizeof(CalibSet)), o_bp = take(bin_ptr.size() * 4 + 4);
    const size_t o_be = take(bin_ent.size() * 4 + 4), o_eb = take(ent_bin.size() * 4 + 4);
    const size_t o_q = take(q.size() * 8 + 8), o_qf = take(core.quiet_flag.size() * 4 + 4);
    if (hipMalloc(&c->d_calib, off) != hipSuccess)
        return fail(PROCELL_E_OUT_OF_MEMORY);
    char *base = (char *)c->d_calib;
    auto up = [&](size_t o, const void *src, size_t bytes) {
        return bytes ? hipMemcpy(base + o, src, bytes, hipMemcpyHostToDevice) : hipSuccess;
    };
    CALIB_TRY(up(o_cs, cs.data(), cs.size() * sizeof(CalibSet)));
    CALIB_TRY(up(o_bp, bin_ptr.data(), bin_ptr.size() * 4));
    CALIB_TRY(up(o_be, bin_ent.data(), bin_ent.size() * 4));
    CALIB_TRY(up(o_eb, ent_bin.data(), ent_bin.size() * 4));
    CALIB_TRY(up(o_q, q.data(), q.size() * 8));
    CALIB_TRY(up(o_qf, core.quiet_flag.data(), core.quiet_flag.size() * 4));

    const size_t P = 3ull * core.types_total;
    size_t so = 0;
    auto stake = [&](size_t bytes) {
        const size_t o = so;
        so = (so + bytes + 255) / 256 * 256;
        return o;
    };
    // cleared every step: h | Jacobian (without a stride) | grad | expansions
    // (one contiguous block)
    c->jac_route = cell_stride == 1;
    const size_t jac_words = c->jac_route ? 2ull * core.h_total : 0;
    const size_t s_h = stake(0);
    const size_t clear_bytes = (core.h_total + jac_words + P + kCountCopies * kCountWords) * 8;
    so = (clear_bytes + 255) / 256 * 256;
    const size_t s_x = stake(P * 8), s_m1 = stake(P * 8), s_m2 = stake(P * 8), s_th = stake(P * 8);
    const size_t s_g = stake(c->jac_route ? 8 : core.h_total * 8 + 8), s_hb = stake(n_bins_total * 8 + 8);
    const size_t s_loss = stake(n_sets * 8), s_step = stake(8);
    if (hipMalloc(&c->d_state, so) != hipSuccess)
        return fail(PROCELL_E_OUT_OF_MEMORY);
    char *sb = (char *)c->d_state;
    std::vector<double> x(P, 0.0);
    for (uint32_t i = 0; i < n_sets; ++i) {
        const RelaxSet &S = core.sets[i];
        const uint32_t T = S.n_types;
        for (uint32_t j = 0; j < sets[i].n_types; ++j) {
            const procell_type &ty = sets[i].types[j];
            if (ty.mean >= 0.0) {
                x[S.theta_base + j] = log(ty.mean);
                x[S.theta_base + T + j] = log(ty.sd);
            }
            x[S.theta_base + 2 * T + j] = ty.proportion > 0.0 ? log(ty.proportion) : -745.0;
        }
        for (uint32_t j = sets[i].n_types; j < T; ++j)
            x[S.theta_base + 2 * T + j] = -745.0;  // padding type of an empty type table
    }
    CALIB_TRY(hipMemcpy(sb + s_x, x.data(), P * 8, hipMemcpyHostToDevice));
    CALIB_TRY(hipMemset(sb + s_m1, 0, P * 8));
    CALIB_TRY(hipMemset(sb + s_m2, 0, P * 8));
    CALIB_TRY(hipMemset(sb + s_step, 0, 8));
    CALIB_TRY(hipMemset(sb, 0, clear_bytes));
    c->d_clear = (unsigned long long *)(sb + s_h);
    c->clear_words = clear_bytes / 8;
    double *d_h = (double *)(sb + s_h);
    double *d_jac = c->jac_route ? d_h + core.h_total : nullptr;
    double *d_grad = d_h + core.h_total + jac_words;
    unsigned long long *d_exp = (unsigned long long *)(d_grad + P);

    CalibArgs &ca = c->cargs;
    ca.n_sets = n_sets;
    ca.lr = adam->lr;
    ca.beta1 = adam->beta1;
    ca.beta2 = adam->beta2;
    ca.eps = adam->eps;
    ca.sets = core.args.sets;
    ca.csets = (const CalibSet *)(base + o_cs);
    ca.bin_ptr = (const uint32_t *)(base + o_bp);
    ca.bin_ent = (const uint32_t *)(base + o_be);
    ca.ent_bin = (const int32_t *)(base + o_eb);
    ca.q = (const double *)(base + o_q);
    ca.quiet_flag = (const uint32_t *)(base + o_qf);
    ca.hb = (double *)(sb + s_hb);
    ca.loss = (double *)(sb + s_loss);
    ca.h = d_h;
    ca.g = (double *)(sb + s_g);
    ca.grad = d_grad;
    ca.jac = d_jac;
    ca.h_total = core.h_total;
    ca.x = (double *)(sb + s_x);
    ca.m1 = (double *)(sb + s_m1);
    ca.m2 = (double *)(sb + s_m2);
    ca.theta = (double *)(sb + s_th);
    ca.step = (unsigned long long *)(sb + s_step);
    c->fwd = core.args;
    c->fwd.step = ca.step;
    c->fwd.stride_mask = cell_stride - 1;
    c->fwd.theta = ca.theta;
    c->fwd.h = d_h;
    c->fwd.expansions = d_exp;
    c->fwd.set_cuts = nullptr;  // a calibration reports the step's total only
    c->fwd.jac = d_jac;
    c->bwd = c->fwd;
    // with a stride, the adjoint walks the next class of cells: the residual
    // (from the forward pass) and the Jacobian then come from independent
    // cells, so their product is an unbiased gradient of the squared loss
    c->bwd.phase = cell_stride > 1 ? 1u : 0u;
    c->bwd.h = nullptr;
    c->bwd.g = ca.g;
    c->bwd.grad = d_grad;

    if (sets[0].stream) {
        c->stream = (hipStream_t)sets[0].stream;
    } else {
        CALIB_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
        c->own_stream = true;
    }
    hipLaunchKernelGGL(calib_init_kernel, dim3((n_sets + 255) / 256), dim3(256), 0, c->stream, ca);
    CALIB_TRY(hipGetLastError());
    CALIB_TRY(hipStreamSynchronize(c->stream));
    *out = c;
    return PROCELL_OK;
#undef CALIB_TRY
}

int procell_calib_step(procell_calib *c, uint32_t n_steps)
{
    if (!c)
        return PROCELL_E_INVALID;
    RELAX_TRY(hipSetDevice(c->core.device));
    if (!c->graph_exec) {
        RELAX_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        const hipError_t e = calib_enqueue(c, c->stream);
        hipGraph_t g = nullptr;
        const hipError_t e2 = hipStreamEndCapture(c->stream, &g);
        if (e != hipSuccess || e2 != hipSuccess) {
            if (g)
                (void)hipGraphDestroy(g);
            g_relaxed_hip = e != hipSuccess ? e : e2;
            return PROCELL_E_HIP;
        }
        const hipError_t e3 = hipGraphInstantiate(&c->graph_exec, g, nullptr, nullptr, 0);
        if (e3 != hipSuccess) {
            (void)hipGraphDestroy(g);
            c->graph_exec = nullptr;
            g_relaxed_hip = e3;
            return PROCELL_E_HIP;
        }
        c->graph = g;
    }
    for (uint32_t i = 0; i < n_steps; ++i)
        RELAX_TRY(hipGraphLaunch(c->graph_exec, c->stream));
    return PROCELL_OK;
}

int procell_calib_theta(procell_calib *c, double *theta, uint64_t capacity)
{
    if (!c || !theta || capacity < 3ull * c->core.types_total)
        return PROCELL_E_INVALID;
    RELAX_TRY(hipSetDevice(c->core.device));
    RELAX_TRY(hipStreamSynchronize(c->stream));
    RELAX_TRY(hipMemcpy(theta, c->cargs.theta, 3ull * c->core.types_total * 8, hipMemcpyDeviceToHost));
    return PROCELL_OK;
}

int procell_calib_loss(procell_calib *c, double *loss, uint32_t capacity, uint64_t *steps, uint64_t *expansions)
{
    if (!c || !loss || capacity < c->core.n_sets)
        return PROCELL_E_INVALID;
    RELAX_TRY(hipSetDevice(c->core.device));
    RELAX_TRY(hipStreamSynchronize(c->stream));
    RELAX_TRY(hipMemcpy(loss, c->cargs.loss, c->core.n_sets * 8ull, hipMemcpyDeviceToHost));
    if (steps) {
        unsigned long long s = 0;
        RELAX_TRY(hipMemcpy(&s, c->cargs.step, 8, hipMemcpyDeviceToHost));
        *steps = s;
    }
    uint64_t ex = 0, cut = 0;
    RELAX_TRY(read_counts(c->fwd.expansions, ex, cut));
    if (expansions)
        *expansions = ex;
    return cut ? PROCELL_E_DEPTH : PROCELL_OK;
}

void *procell_calib_stream(procell_calib *c) { return c ? (void *)c->stream : nullptr; }

int procell_calib_destroy(procell_calib *c)
{
    destroy_calib(c);
    return PROCELL_OK;
}

}  // extern "C"
