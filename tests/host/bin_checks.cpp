// bin_checks.cpp -- the output bin set and the bin of every (row, generation)
// (procell_setup.cpp: build_bins, index_bins) against their definition: every
// v / 2^k >= phi, exact halving, distinct, ascending; the bin of an entry is
// the one that equals its value, -1 below phi.  Exit status 0 when it held.
#include <math.h>
#include <stdio.h>

#include <random>
#include <set>

#include "procell_setup.hpp"

using namespace procell;

static int g_failures = 0, g_entries = 0;

static void check(const char *what, const std::vector<double> &values, const std::vector<uint64_t> &counts, double phi)
{
    std::vector<procell_row> rows;
    for (size_t i = 0; i < values.size(); ++i)
        rows.push_back({values[i], counts[i]});
    const procell_type type{1.0, 10.0, 1.0};
    procell_params p{};
    p.rows = rows.data();
    p.n_rows = rows.size();
    p.types = &type;
    p.n_types = 1;
    p.t_max = 10.0;
    p.phi = phi;
    Setup s;
    bool ok = build_setup(&p, s, true) == PROCELL_OK;
    std::set<double> want;
    for (double v : s.v)
        for (double f = v; ok && f >= s.phi; f = f / 2)
            want.insert(f);
    ok = ok && s.bins == std::vector<double>(want.begin(), want.end());
    const std::vector<int32_t> bin_of = index_bins(s);
    const size_t kdim = (size_t)s.kmax + 1;
    ok = ok && bin_of.size() == s.v.size() * kdim;
    for (size_t r = 0; ok && r < s.v.size(); ++r) {
        double f = s.v[r];
        for (size_t k = 0; k < kdim; ++k, f = f / 2, ++g_entries) {
            const int32_t b = bin_of[r * kdim + k];
            ok = ok && (want.count(f) ? b >= 0 && (size_t)b < s.bins.size() && s.bins[(size_t)b] == f : b == -1);
        }
    }
    if (!ok) {
        fprintf(stderr, "%s: %zu rows, phi %g\n", what, values.size(), phi);
        ++g_failures;
    }
}

int main()
{
    const struct {
        std::vector<double> v;
        double phi;
    } tables[] = {
        {{8.0, 16.0, 12.0, 3.0, 6.0}, 1.0},       {{8.0, 16.0, 12.0, 3.0, 6.0}, 1.5}, {{8.0, 16.0}, 8.0},
        {{5.0, 2.0, -7.0, 0.0, 10.0}, 2.5},       {{1.0}, 0.0},                       {{1e-307, 3e-308, 7e-307}, 2.5e-308},
        {{1e-307, 3e-308, 7e-308}, 1e-310},       {{4e-324, 8e-324}, 4e-324},         {{1.75, 1.75, 3.5, 7.0, 1.0}, 0.4},
        {{1e-300, 2.2250738585072014e-308}, 2.2250738585072014e-308},                 {{1e-310, -0.0, 1e-320}, 1e-322},
        {{1.7976931348623157e308, 1e300}, 1e290}, {{-4.0, -8.0}, 1.0},
    };
    for (const auto &t : tables) {
        std::vector<uint64_t> counts;
        for (size_t i = 0; i < t.v.size(); ++i)
            counts.push_back(1 + i % 3);
        check("table", t.v, counts, t.phi);
    }
    std::mt19937_64 rng(7);
    for (int seed = 0; seed < 400; ++seed) {
        const size_t n = 1 + rng() % 200;
        const int low = seed % 5 == 4 ? -1070 : -3, span = seed % 5 == 4 ? 60 : 17;
        std::vector<double> v;
        std::vector<uint64_t> counts;
        for (size_t i = 0; i < n; ++i) {  // shared mantissas, and any
            const double m = seed % 2 ? (double)(8 + rng() % 8) / 8.0 : 1.0 + (double)rng() / 18446744073709551616.0;
            v.push_back((rng() % 50 ? 1.0 : -1.0) * ldexp(m, low + (int)(rng() % (unsigned)span)));
            counts.push_back(i ? rng() % 3 : 1);
        }
        v[0] = fabs(v[0]);
        const double phi = seed % 3 == 0 ? v[0] : ldexp(1.0 + (double)(rng() % 1000) / 1000.0, low + (int)(rng() % 4));
        check("random", v, counts, phi);
    }
    printf("%d entries, %d failed\n", g_entries, g_failures);
    return g_failures ? 1 : 0;
}
