// procell_setup.cpp -- host-only part of libprocell: validation and set-up
// (the reference's parse-time rules, src/io/parser.cu:46-151), the cost
// model behind the segment split, the merge of a raw tally into the output
// histogram (src/simulation/proliferation.cu:353-380), and the sizing entry
// points of the C ABI.  Compiled by the host compiler.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "procell_filter.hpp"
#include "procell_setup.hpp"

namespace procell {

// ---------------------------------------------------------------------------
// Validation and set-up (mirrors the reference's parse-time rules).
// ---------------------------------------------------------------------------
int generation_cap(double v, double phi)
{
    // proliferation.cu:323: divide only while f/2 > phi; f halves exactly.
    int k = 0;
    double f = v;
    while (f / 2 > phi) {
        f = f / 2;
        if (++k > kMaxGeneration)
            return k;
    }
    return k;
}

double resolve_phi(const procell_params *p)
{
    if (p->phi > 0.0)
        return p->phi;
    // parser.cu:80-96: smallest value among rows with a nonzero count.
    double best = 0.0;
    bool have = false;
    for (uint64_t i = 0; i < p->n_rows; ++i) {
        const procell_row &r = p->rows[i];
        if (r.count > 0 && (!have || r.value < best)) {
            best = r.value;
            have = true;
        }
    }
    return best;
}

// Bits, biased exponent and mantissa of a double.
static uint64_t double_bits(double x)
{
    uint64_t u;
    memcpy(&u, &x, 8);
    return u;
}
static uint64_t exponent(double x) { return double_bits(x) >> 52; }
static uint64_t mantissa(double x) { return double_bits(x) & ((1ull << 52) - 1); }

// Rows with value >= phi by mantissa.  Halving a normal number keeps its
// mantissa, so the values v / 2^k of one exponent come in this order.
static std::vector<std::pair<uint64_t, uint32_t>> rows_by_mantissa(const Setup &s)
{
    std::vector<std::pair<uint64_t, uint32_t>> rows;  // mantissa, row
    rows.reserve(s.v.size());
    for (size_t r = 0; r < s.v.size(); ++r)
        if (s.v[r] >= s.phi)
            rows.emplace_back(mantissa(s.v[r]), (uint32_t)r);
    std::sort(rows.begin(), rows.end());
    return rows;
}

// Output bin set (parser.cu:126-151): every v / 2^k >= phi, exact halving,
// distinct, ascending.
static void build_bins(Setup &s)
{
    if (exponent(s.phi) == 0) {
        // phi below the smallest normal number: sorted as they come
        for (double v : s.v) {
            double f = v;
            while (f >= s.phi) {
                s.bins.push_back(f);
                f = f / 2;
            }
        }
        std::sort(s.bins.begin(), s.bins.end());
        s.bins.erase(std::unique(s.bins.begin(), s.bins.end()), s.bins.end());
        return;
    }
    // one exponent after the other, each in the order of the distinct
    // mantissas (sorting the rows, not the several bins of each: 175 -> 50 us
    // at 796 rows and 3706 bins)
    std::vector<std::pair<uint64_t, uint64_t>> values;  // mantissa, largest exponent
    uint64_t top = 0;
    for (const auto &mr : rows_by_mantissa(s)) {
        const uint64_t e = exponent(s.v[mr.second]);
        top = std::max(top, e);
        if (values.empty() || values.back().first != mr.first)
            values.emplace_back(mr.first, e);
        else
            values.back().second = std::max(values.back().second, e);
    }
    const uint64_t first = exponent(s.phi);
    for (uint64_t e = first; e <= top; ++e)
        for (const auto &me : values)
            if (me.second >= e && (e > first || me.first >= mantissa(s.phi))) {
                const uint64_t u = e << 52 | me.first;
                double f;
                memcpy(&f, &u, 8);
                s.bins.push_back(f);
            }
}

static void cost_caps(Setup &s);

int build_setup(const procell_params *p, Setup &s, bool want_bins, bool want_costs)
{
    if (!p || (p->n_rows && !p->rows) || (p->n_types && !p->types))
        return PROCELL_E_INVALID;
    if (isnan(p->t_max) || p->t_max < 0.0)
        return PROCELL_E_INVALID;
    s = Setup();
    s.t_max = p->t_max;
    uint64_t total = 0, n_nz = 0;
    for (uint64_t i = 0; i < p->n_rows; ++i) {
        if (!isfinite(p->rows[i].value))
            return PROCELL_E_NONFINITE;
        const uint64_t c = p->rows[i].count;
        if (c == 0)
            continue;
        ++n_nz;
        if (total + c < total || total + c > kMaxCells)
            return PROCELL_E_TOO_MANY_CELLS;
        total += c;
    }
    if (n_nz > kMaxRows)
        return PROCELL_E_TOO_MANY_CELLS;
    if (p->n_types == 0)
        return total ? PROCELL_E_PROPORTIONS : PROCELL_OK;
    if (p->n_types > kMaxTypes)
        return PROCELL_E_TOO_MANY_CELLS;
    // parser.cu:46-66: proportions (left fold, file order) must sum to 1.
    double sum = 0.0;
    for (uint32_t j = 0; j < p->n_types; ++j) {
        const procell_type &t = p->types[j];
        if (!isfinite(t.proportion) || !isfinite(t.mean) || !isfinite(t.sd))
            return PROCELL_E_NONFINITE;
        sum = sum + t.proportion;
    }
    if (fabs(1.0 - sum) > 1.0 / pow(10.0, 8.0))
        return PROCELL_E_PROPORTIONS;
    for (uint32_t j = 0; j < p->n_types; ++j)
        if (p->types[j].mean == 0.0)
            return PROCELL_E_ZERO_MEAN;  // cell.cu:110 would leave the timer unset
    const double phi = resolve_phi(p);
    if (total > 0 && !(phi > 0.0))
        return PROCELL_E_PHI;
    s.phi = phi;
    s.n_cells = total;
    s.n_types = p->n_types;
    s.v.reserve(n_nz);
    s.start.reserve(n_nz + 1);
    s.row_info.reserve(n_nz);
    uint64_t acc = 0;
    for (uint64_t i = 0; i < p->n_rows; ++i) {
        const procell_row &r = p->rows[i];
        if (r.count == 0)
            continue;
        const int kc = generation_cap(r.value, phi);
        if (kc > kMaxGeneration)
            return PROCELL_E_DEPTH;
        s.kmax = std::max(s.kmax, kc);
        s.v.push_back(r.value);
        s.start.push_back(acc);
        s.row_info.push_back((uint32_t)kc | ((r.value >= phi ? 1u : 0u) << 8));
        acc += r.count;
    }
    s.start.push_back(acc);
    // parser.cu:184: descending proportion; ties keep file order.
    s.type_file.resize(s.n_types);
    for (uint32_t j = 0; j < s.n_types; ++j)
        s.type_file[j] = j;
    std::stable_sort(s.type_file.begin(), s.type_file.end(), [&](uint32_t x, uint32_t y) {
        return p->types[x].proportion > p->types[y].proportion;
    });
    // cell.cu:86-101: running sum in sorted order.
    double c = 0.0;
    for (uint32_t j = 0; j < s.n_types; ++j) {
        const procell_type &t = p->types[s.type_file[j]];
        c = c + t.proportion;
        s.type_cum.push_back(c);
        s.type_mean.push_back(t.mean);
        s.type_sd.push_back(t.sd);
    }
    if (want_costs)
        cost_caps(s);
    if (want_bins)
        build_bins(s);
    return PROCELL_OK;
}

static double normal_cdf(double z) { return 0.5 * erfc(-z / sqrt(2.0)); }

// Mean and variance of the completion time D = tau0 (1 + U) + tau_1 + ... +
// tau_k of a type's division k+1, approximated as normal (truncation ignored).
static void completion(double m, double sd, int k, double &mu, double &var)
{
    mu = 1.5 * m + k * m;
    var = (7.0 / 3.0) * sd * sd + m * m / 12.0 + k * sd * sd;
    if (!(var > 0.0))
        var = 1e-300;
}

// Lane-steps of one initial cell of a row: its root step (one lane of a
// full-width step, about what a division costs) plus the expected number of
// divisions.  Only used to balance the workgroups' segments (claims and
// stealing even out its errors) and to choose the kernel.  It depends on the
// row through its generation cap alone, and on the type through prefix sums
// over the levels, so every completion probability is evaluated once (1024
// rows, 5 types, 11 caps: 0.3 ms of erfc evaluations by row, 30 us by cap).
constexpr double kRootCost = 1.0;
static void cost_caps(Setup &s)
{
    s.cap_cost.assign((size_t)s.kmax + 1, kRootCost);
    s.in_time.assign((size_t)s.n_types * (size_t)s.kmax, 0.0);
    double p_prev = 0.0;
    for (uint32_t j = 0; j < s.n_types; ++j) {
        const double m = s.type_mean[j], sd = fabs(s.type_sd[j]), p = s.type_cum[j] - p_prev;
        p_prev = s.type_cum[j];
        if (m < 0.0)
            continue;
        double e = 0.0, prob = 1.0;
        for (int cap = 1; cap <= s.kmax; ++cap) {
            if (!(prob < 1e-12)) {
                double mu, var;
                completion(m, sd, cap - 1, mu, var);
                prob = normal_cdf((s.t_max - mu) / sqrt(var));
                s.in_time[(size_t)j * s.kmax + cap - 1] = prob;
                e += ldexp(prob, cap - 1);
            }
            s.cap_cost[cap] += p * e;
        }
    }
}

// Expected work of a set on the filtered kernel, in lane-steps (normal
// approximation as in cost_caps).
struct FilterWork {
    double divisions = 0.0;
    double redraws = 0.0;  // steps that draw a refused timer again
    double unsure = 0.0;   // divisions with a test within the error bound, evaluated again in 64 bits
    double levels = 0.0;   // divisions, each times its level
    double chain = 0.0;    // expected longest chain of such evaluations on one lane, in levels
};

static FilterWork filter_work(const Setup &s)
{
    FilterWork f;
    std::vector<double> cells((size_t)s.kmax + 1, 0.0);  // by generation cap
    for (size_t r = 0; r < s.v.size(); ++r)
        cells[s.row_info[r] & 0xFFu] += (double)(s.start[r + 1] - s.start[r]);
    double p_prev = 0.0;
    for (uint32_t j = 0; j < s.n_types && !s.v.empty(); ++j) {
        const double m = s.type_mean[j], sd = fabs(s.type_sd[j]), p = s.type_cum[j] - p_prev;
        p_prev = s.type_cum[j];
        if (m < 0.0 || !(p > 0.0))
            continue;
        const double refused = sd > 0.0 ? normal_cdf(-m / sd) : 0.0;
        const double redraws = 2.0 * refused / (1.0 - refused * refused);  // per division; two candidates a block
        const double terr = filter_type_err(m, sd, s.t_max);
        const double at0 = sd > 0.0 ? 0.3989422804014327 * exp(-0.5 * (m / sd) * (m / sd)) / sd : 0.0;  // timers' density there
        // over the levels above a cap: divisions, levels; over its daughters'
        // levels: density of completion times at t_max, of all and of one per level
        double e = 0.0, lv = 0.0, dens = 0.0, dens1 = 0.0;
        for (int cap = 1; cap <= s.kmax; ++cap) {
            const double prob = s.in_time[(size_t)j * s.kmax + cap - 1];
            if (prob > 0.0) {
                e += ldexp(prob, cap - 1);
                lv += ldexp(prob, cap - 1) * cap;
                double mu, var;
                completion(m, sd, cap, mu, var);
                const double z = (s.t_max - mu) / sqrt(var), d = 0.3989422804014327 * exp(-0.5 * z * z) / sqrt(var);
                dens += ldexp(d, cap);
                dens1 += d;
            }
            const double n = cells[cap] * p, err = (cap + 4.0) * terr;
            if (!(n > 0.0) || !(e > 0.0))
                continue;
            const double near0 = err < 0.1 * sd ? 2.0 * err * at0
                                 : sd > 0.0     ? normal_cdf((err - m) / sd) - normal_cdf((-err - m) / sd)
                                                : (m < err ? 1.0 : 0.0);
            f.divisions += n * e;
            f.redraws += n * e * redraws;
            f.unsure += n * (std::min(1.0, 2.0 * near0) * e + std::min(e, 2.0 * err * dens));
            f.levels += n * lv;
            // a cell within the bound of t_max, and the share of its last
            // daughters that then are
            const double chain = std::min(1.0, 2.5 * err / (sd * sqrt(lv / e) + 1e-300)) * 0.5 * lv;
            if (chain > f.chain)
                f.chain = std::max(f.chain, chain * (1.0 - exp(-2.0 * err * n * dens1)));
        }
    }
    return f;
}

// A step of a wavefront, in steps of the filtered kernel without any of the
// following:
//  * with a lane whose refused timer is drawn again, both kernels take their
//    longer branch, the filtered one a longer one (the more such lanes);
//  * an unsure division walks its path from the root again in 64 bits, about
//    1.8 steps per level, while the wavefront's other lanes wait;
//  * where a type's timers hardly differ, a cell within the bound of t_max has
//    many daughters that are, evaluated one after the other on its lane.
// With fewer than 3 wavefronts of initial cells per SIMD a run is as long as
// its wavefronts' own instruction streams take, with more the vector units'
// issue limits it; there the filtered kernel gains more and loses less.
// Measured, 64-bit against filtered kernel, microseconds per run (two rows of
// 11 generations; t_max / mean, sd / mean): 3e4 cells at 8.3, 0.3: 172 / 135;
// 0.4: 202 / 194; 0.45: 217 / 228; 0.6: 221 / 264; 1: 156 / 230; 8.0, 0:
// 99 / 395; 8.0, 1e-3: 97 / 74; 4e4, 0.25: 802 / 680; 1.6e5, 0.25: 801 / 2091;
// 1e4, 0.4: 887 / 2403.  3e5 cells at 3.3, 0.4: 46 / 32; 1: 60 / 60; 1.5:
// 57 / 61.  1024 rows and 1e7 cells of four types, 0.25: 542 / 305; 0.6: 619 /
// 494; 1: 722 / 683.
bool filter_pays(const std::vector<Setup> &sets)
{
    constexpr double kSimds = 1024.0, kResident = 6.0 * kSimds;  // filtered kernel: wavefronts
    double cells = 0.0;
    for (const Setup &s : sets)
        cells += (double)s.n_cells;
    const double waves = std::max(1.0, cells / 64.0);
    const bool few = waves < 3.0 * kSimds;
    double all = 0.0, filter = 0.0, wide = 0.0, chain = 0.0;
    for (const Setup &s : sets) {
        const FilterWork f = filter_work(s);
        const double steps = f.divisions + f.redraws;
        if (!(steps > 0.0))
            continue;
        const double r = f.redraws / steps, redo = 1.0 - pow(1.0 - r, 64.0);
        const double unsure = 1.8 * f.levels / f.divisions * (1.0 - pow(1.0 - std::min(1.0, f.unsure / steps), 64.0));
        filter += steps * (few ? 1.0 + 0.75 * redo + 3.2 * r + unsure : 1.0 + 0.1 * redo + 2.2 * r + unsure);
        wide += steps * (few ? 1.42 + 0.23 * redo : 1.78);
        all += steps;
        chain = std::max(chain, f.chain);
    }
    if (!(all > 0.0))
        return true;
    // the run in a wavefront's steps: six wavefronts of a SIMD take 2.5 times
    // as long for one as one alone
    const double run = all / 64.0 / std::min(waves, kResident) * (few ? 1.0 : 2.5);
    return !(filter + all * 1.8 * chain / run > wide);
}

static std::vector<double> row_costs(const Setup &s)
{
    std::vector<double> w(s.v.size());
    for (uint32_t r = 0; r < (uint32_t)w.size(); ++r)
        w[r] = s.cap_cost[s.row_info[r] & 0xFFu];
    return w;
}

Setup order_rows(const Setup &s, std::vector<uint32_t> &file_row)
{
    const std::vector<double> w = row_costs(s);
    const size_t n = w.size();
    file_row.resize(n);
    for (size_t i = 0; i < n; ++i)
        file_row[i] = (uint32_t)i;
    std::stable_sort(file_row.begin(), file_row.end(), [&](uint32_t x, uint32_t y) { return w[x] > w[y]; });
    Setup o = s;
    uint64_t at = 0;
    for (size_t i = 0; i < n; ++i) {
        const uint32_t r = file_row[i];
        o.v[i] = s.v[r];
        o.row_info[i] = s.row_info[r];
        o.start[i] = at;
        at += s.start[r + 1] - s.start[r];
    }
    return o;
}

// Split the initial cells into contiguous segments whose cumulative costs end
// at the fractions cum[0] < cum[1] < ... < cum[g-1] = 1 of the total.
void split_segments(const Setup &s, const std::vector<double> &cum, std::vector<uint64_t> &begin,
                    std::vector<uint32_t> &row_of)
{
    const uint32_t g = (uint32_t)cum.size();
    const uint32_t n_rows = (uint32_t)s.v.size();
    begin.assign(g + 1, s.n_cells);
    row_of.assign(g, n_rows ? n_rows - 1 : 0);
    begin[0] = 0;
    const std::vector<double> w = row_costs(s);
    double total = 0.0;
    for (uint32_t r = 0; r < n_rows; ++r)
        total += w[r] * (double)(s.start[r + 1] - s.start[r]);
    uint32_t next = 1;
    double acc = 0.0;
    for (uint32_t r = 0; r < n_rows && next < g; ++r) {
        const uint64_t n = s.start[r + 1] - s.start[r];
        const double row_total = w[r] * (double)n;
        while (next < g && acc + row_total >= total * cum[next - 1]) {
            const double want = total * cum[next - 1] - acc;
            uint64_t cut = s.start[r] + (uint64_t)(want / w[r]);
            if (cut > s.start[r + 1])
                cut = s.start[r + 1];
            if (cut < begin[next - 1])
                cut = begin[next - 1];
            begin[next++] = cut;
        }
        acc += row_total;
    }
    for (uint32_t i = 0; i < g; ++i) {
        const uint64_t c = begin[i] < s.n_cells ? begin[i] : (s.n_cells ? s.n_cells - 1 : 0);
        row_of[i] = (uint32_t)(std::upper_bound(s.start.begin(), s.start.end() - 1, c) - s.start.begin()) - 1;
    }
}

// Expected work of a set (sum of row costs over its cells).
double set_cost(const Setup &s)
{
    const std::vector<double> w = row_costs(s);
    double total = 0.0;
    for (uint32_t r = 0; r < (uint32_t)s.v.size(); ++r)
        total += w[r] * (double)(s.start[r + 1] - s.start[r]);
    return total;
}

void fill_stats(const unsigned long long *cnt, const int64_t *tally, size_t tally_len, procell_stats &st)
{
    memset(&st, 0, sizeof st);
    st.divisions = cnt[kDivisions];
    // recorded = tally sum; dropped from the event balance (every division
    // adds one cell; every cell ends recorded, dropped or lost)
    uint64_t recorded = 0;
    for (size_t i = 0; i < tally_len; ++i)
        recorded += (uint64_t)tally[i];
    st.recorded = recorded;
    st.dropped = cnt[kCells] + cnt[kDivisions] - recorded - cnt[kLost];
    st.lost = cnt[kLost];
    st.rejected = cnt[kRejected];
    st.cells = cnt[kCells];
    st.pool = cnt[kPoolCount];
}

std::vector<int32_t> index_bins(const Setup &s)
{
    const uint64_t n_rows = s.v.size();
    const uint32_t kdim = (uint32_t)s.kmax + 1;
    std::vector<int32_t> bin_of(n_rows * kdim, -1);
    if (s.bins.empty())
        return bin_of;
    if (exponent(s.bins.front()) == 0) {
        // subnormal bins (phi below the smallest normal number): searched
        for (uint64_t r = 0; r < n_rows; ++r) {
            double f = s.v[r];
            for (uint32_t k = 0; k < kdim; ++k, f = f / 2) {
                auto it = std::lower_bound(s.bins.begin(), s.bins.end(), f);
                if (it != s.bins.end() && *it == f)
                    bin_of[r * kdim + k] = (int32_t)(it - s.bins.begin());
            }
        }
        return bin_of;
    }
    // the bins of each exponent beside the rows, both by mantissa (a search per
    // entry took most of the merge)
    const auto rows = rows_by_mantissa(s);
    for (size_t b = 0; b < s.bins.size();) {
        const uint64_t e = exponent(s.bins[b]);
        size_t end = b;
        while (end < s.bins.size() && exponent(s.bins[end]) == e)
            ++end;
        for (const auto &mr : rows) {
            const uint64_t er = exponent(s.v[mr.second]);
            if (er < e || er - e >= kdim)
                continue;
            while (b < end && mantissa(s.bins[b]) < mr.first)
                ++b;
            if (b < end && mantissa(s.bins[b]) == mr.first)
                bin_of[(uint64_t)mr.second * kdim + (er - e)] = (int32_t)b;
        }
        b = end;
    }
    return bin_of;
}

int merge_tally(const Setup &s, const int64_t *tally, procell_result *r)
{
    return merge_tally(s, index_bins(s), tally, r);
}

int merge_tally(const Setup &s, const std::vector<int32_t> &bin_of, const int64_t *tally, procell_result *r)
{
    const uint32_t T = s.n_types ? s.n_types : 1;
    const uint32_t kdim = (uint32_t)s.kmax + 1;
    const uint64_t n_ent = s.v.size() * kdim;
    const uint64_t n_bins = s.bins.size();
    if (!r || (r->capacity && !(r->value && r->count)))
        return PROCELL_E_INVALID;
    // (row, generation) -> output value row_value * 2^-generation, exact
    // equality merge into the bin set (proliferation.cu:353-380 searches the
    // same set by exact equality).
    std::vector<int64_t> bt((size_t)n_bins * (T + 1), 0);  // per bin: all types, then each
    for (uint64_t e = 0; e < n_ent; ++e) {
        const int64_t *cell = &tally[(size_t)e * T];
        int64_t tot = 0;
        for (uint32_t j = 0; j < T; ++j)
            tot += cell[j];
        if (!tot || bin_of[e] < 0)  // (recorded values are >= phi)
            continue;
        int64_t *bin = &bt[(size_t)bin_of[e] * (T + 1)];
        bin[0] += tot;
        for (uint32_t j = 0; j < T; ++j)
            bin[1 + j] += cell[j];
    }
    uint64_t n_out = 0;
    for (uint64_t b = 0; b < n_bins; ++b)
        n_out += bt[b * (T + 1)] > 0;
    r->n_out = n_out;
    if (n_out > r->capacity)
        return PROCELL_E_CAPACITY;
    uint64_t o = 0;
    for (uint64_t b = 0; b < n_bins; ++b) {
        const int64_t *bin = &bt[b * (T + 1)];
        if (bin[0] <= 0)
            continue;
        r->value[o] = s.bins[b];
        r->count[o] = bin[0];
        if (r->type_count)
            for (uint32_t j = 0; j < s.n_types; ++j)
                r->type_count[o * s.n_types + j] = bin[1 + j];
        ++o;
    }
    return PROCELL_OK;
}

}  // namespace procell

using namespace procell;

extern "C" {

int procell_output_capacity(const procell_params *p, uint64_t *capacity)
{
    if (!capacity)
        return PROCELL_E_INVALID;
    Setup s;
    const int rc = build_setup(p, s, true, false);
    if (rc != PROCELL_OK)
        return rc;
    *capacity = s.bins.size();
    return PROCELL_OK;
}

int procell_tally_shape(const procell_params *p, uint64_t *nonzero_rows, uint32_t *kdim)
{
    if (!nonzero_rows || !kdim)
        return PROCELL_E_INVALID;
    Setup s;
    const int rc = build_setup(p, s, false, false);
    if (rc != PROCELL_OK)
        return rc;
    *nonzero_rows = s.v.size();
    *kdim = (uint32_t)s.kmax + 1;
    return PROCELL_OK;
}

int procell_resolve_phi(const procell_params *p, double *phi)
{
    if (!p || !phi || (p->n_rows && !p->rows))
        return PROCELL_E_INVALID;
    *phi = resolve_phi(p);
    return PROCELL_OK;
}

}  // extern "C"
