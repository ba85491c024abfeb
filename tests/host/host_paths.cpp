// host_paths.cpp -- libprocell's host code over the stand-in HIP runtime
// (fake_hip.cpp): which device memory, streams and launches the entry points
// use, and which run their results come from.  usage: host_paths <check>; exit
// status 0 when it held.
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>

#include "fake_hip.hpp"
#include "procell.h"

static int g_failures = 0;

#define CHECK(c)                                                                    \
    do {                                                                            \
        if (!(c)) {                                                                 \
            fprintf(stderr, "CHECK failed at %s:%d: %s\n", __FILE__, __LINE__, #c); \
            ++g_failures;                                                           \
        }                                                                           \
    } while (0)

// A problem and room for its result.
struct Case {
    std::vector<procell_row> rows;
    std::vector<procell_type> types;
    std::vector<double> value;
    std::vector<int64_t> count;
    procell_params p{};
    procell_result r{};
    Case(std::vector<procell_row> rows_, std::vector<procell_type> types_, double t_max, double phi)
        : rows(std::move(rows_)), types(std::move(types_))
    {
        p.rows = rows.data();
        p.n_rows = rows.size();
        p.types = types.data();
        p.n_types = (uint32_t)types.size();
        p.t_max = t_max;
        p.phi = phi;
        uint64_t cap = 0;
        CHECK(procell_output_capacity(&p, &cap) == PROCELL_OK);
        value.resize(cap + 1);
        count.resize(cap + 1);
        r.capacity = cap;
        r.value = value.data();
        r.count = count.data();
    }
    Case(const Case &) = delete;
};

// A run that fails after its kernels were enqueued: every set's result then
// comes from that run, also those that an earlier download had brought along.
static void check_stage()
{
    Case c({{100.0, 500}, {30.0, 300}}, {{1.0, 20.0, 5.0}}, 90.0, 1.0);
    c.p.tuning.flags = PROCELL_FLAG_TIMING;
    std::vector<procell_params> sets(8, c.p);
    std::vector<uint64_t> seeds(8, 1);
    procell_plan *b = nullptr;
    CHECK(procell_batch_create(sets.data(), 8, &b) == PROCELL_OK);
    CHECK(procell_batch_run(b, seeds.data()) == PROCELL_OK);
    for (uint32_t i = 0; i < 2; ++i) {  // the second brings its successor along
        CHECK(procell_batch_result(b, i, &c.r) == PROCELL_OK);
        CHECK(c.r.stats.divisions == 1);
    }
    fake::fail_event_record = 3;  // the seeds' event, the run's first, the run's last
    CHECK(procell_batch_run(b, seeds.data()) == PROCELL_E_HIP);
    CHECK(fake::fail_event_record == 0 && fake::sim_runs == 2);
    for (uint32_t i : {2u, 7u, 1u, 3u}) {
        CHECK(procell_batch_result(b, i, &c.r) == PROCELL_OK);
        CHECK(c.r.stats.divisions == 2);
    }
    CHECK(procell_plan_destroy(b) == PROCELL_OK);
}

// procell_simulate_noalloc: 16 MiB of static memory for the counters, 8 bytes
// per tally entry and 8 of tables per row, so some 1.04e6 rows of one
// generation and one type, and not many more.
static void check_noalloc()
{
    for (uint64_t n : {1000ull, 835000ull, 900000ull, 1040000ull, 1060000ull}) {
        std::vector<procell_row> rows(n);
        for (uint64_t i = 0; i < n; ++i)
            rows[i] = {1.0 + (double)i / (double)(2 * n), 1};
        Case c(rows, {{1.0, 20.0, 5.0}}, 90.0, 1.0);
        const uint64_t before = fake::sim_runs;
        const int rc = procell_simulate_noalloc(&c.p, &c.r);
        CHECK(rc == (n > 1050000 ? PROCELL_E_SCRATCH : PROCELL_OK));
        CHECK(fake::sim_runs == before + (rc == PROCELL_OK) && fake::memory_alive == 0);
    }
}

// What procell_simulate keeps between calls (a few streams, one small
// allocation) does not outlive a reset of the device: the next call uses
// neither the handles from before, nor streams that the host program has got
// under the same handles since, nor memory under the old address.
static void check_reset()
{
    Case c({{100.0, 500}, {30.0, 300}}, {{1.0, 20.0, 5.0}}, 90.0, 1.0);
    uint64_t runs = 0;
    for (int i = 0; i < 4; ++i) {
        for (int k = 0; k < 2; ++k) {
            CHECK(procell_simulate(&c.p, &c.r) == PROCELL_OK);
            CHECK(c.r.stats.divisions == ++runs);
            CHECK(fake::streams_alive <= 4 + (i > 0) && fake::memory_alive <= 1 + (i > 0));
        }
        CHECK(fake::foreign_stream_uses == 0);
        fake::device_reset();  // from here on the first handles and addresses come again
        fake::take_stream();
        if (i > 0)
            fake::take_memory();
    }
    CHECK(fake::dead_stream_uses == 0);
}

// The kernel of a run: the filtered one, unless the sets' times leave what its
// error bound covers or make it the slower one (each case measured on both).
static void check_kernel()
{
    // two rows of 11 generations, t_max 240; cells, t_max / mean, sd / mean
    struct {
        uint64_t cells;
        double ratio, sd;
        bool filter;
    } const cases[] = {
        {30000, 3.3, 0.2, true},     {30000, 8.3, 0.3, true},    {30000, 50.0, 0.3, true},   {30000, 8.3, 0.45, false},
        {30000, 50.0, 0.5, false},   {30000, 8.3, 1.0, false},   {30000, 50.0, 3.0, false},  {30000, 5.3, 2.0, false},
        {300000, 3.3, 0.3, true},    {300000, 3.3, 0.6, true},   {300000, 3.3, 1.5, false},  {300000, 3.3, 2.0, false},
        {30000, 5e3, 0.25, true},    {30000, 1.6e5, 0.25, false}, {30000, 5e5, 0.25, false}, {30000, 5e6, 0.25, false},
        {30000, 1e4, 0.4, false},    {30000, 4e4, 0.1, true},    {30000, 1e6, 0.05, false},  {30000, 5e6, 0.0, false},
        {30000, 8.0, 0.0, false},    {30000, 8.0, 1e-5, false},  {30000, 8.0, 1e-3, true},   {30000, 8.0, 0.03, true},
        {30000, 50.0, 0.0, true},    {300000, 8.0, 0.0, false},
    };
    auto filtered = [] { return fake::launches.back().kernel.find("sim_filter") != std::string::npos; };
    auto types = [](double ratio, double sd) {
        const double m = 240.0 / ratio;
        return std::vector<procell_type>{{0.6, m, sd * m}, {0.4, 1.3 * m, sd * 1.3 * m}};
    };
    for (const auto &k : cases) {
        Case c({{1500.0, k.cells * 2 / 3}, {1050.0, k.cells / 3}}, types(k.ratio, k.sd), 240.0, 1.0);
        CHECK(procell_simulate(&c.p, &c.r) == PROCELL_OK);
        CHECK(filtered() == k.filter);
        if (filtered() != k.filter)
            fprintf(stderr, "  %llu cells, t_max / mean %g, sd / mean %g\n", (unsigned long long)k.cells, k.ratio, k.sd);
    }
    // times outside the bound's range
    for (double t_max : {0.0, 1e-10, 2e12, (double)INFINITY}) {
        Case c({{1500.0, 1000}}, {{1.0, 20.0, 4.0}}, t_max, 1.0);
        CHECK(procell_simulate(&c.p, &c.r) == PROCELL_OK && !filtered());
    }
    // a batch: by what its sets cost together
    for (bool small : {true, false}) {
        Case a({{1500.0, 200000}}, types(4.0, 0.25), 240.0, 1.0), b({{1500.0, small ? 5u : 20000u}}, types(5e5, 0.25), 240.0, 1.0);
        std::vector<procell_params> sets(16, a.p);
        sets[3] = b.p;
        std::vector<uint64_t> seeds(16, 1);
        procell_plan *pl = nullptr;
        CHECK(procell_batch_create(sets.data(), 16, &pl) == PROCELL_OK);
        CHECK(procell_batch_run(pl, seeds.data()) == PROCELL_OK && filtered() == small);
        CHECK(procell_plan_destroy(pl) == PROCELL_OK);
    }
}

// The tally window: rows of many generations and types, of which three
// workgroups of 512 per CU leave no room for as many as a segment spans, get
// fewer workgroups per CU; the others keep three.
static void check_window()
{
    const std::vector<procell_type> five{{0.2, 35, 9}, {0.2, 55, 14}, {0.2, 75, 19}, {0.2, 95, 24}, {0.2, -1, -1}};
    const std::vector<procell_type> two{{0.5, 35, 9}, {0.5, 95, 24}};
    struct {
        const std::vector<procell_type> &types;
        double top, phi;  // values from 1 to top
        uint32_t rows;
        double cells;
        uint32_t per_cu, window;  // workgroups; least rows
    } const cases[] = {
        {five, 1e5, 50.0, 1024, 1e7, 3, 4},  {five, 1e4, 1.0, 1500, 1e6, 3, 3},  {five, 1e4, 1.0, 6000, 1e7, 2, 10},
        {five, 1e4, 1.0, 100000, 1e7, 1, 100}, {two, 1e4, 1.0, 100, 1e6, 3, 2},  {two, 1e4, 1.0, 25000, 1e7, 2, 50},
        {two, 1e4, 1.0, 25000, 1e5, 3, 10},  {two, 1e3, 1.0, 25000, 1e7, 3, 20},
    };
    for (const auto &k : cases) {
        std::vector<procell_row> rows(k.rows);
        for (uint32_t i = 0; i < k.rows; ++i)
            rows[i] = {pow(k.top, (double)i / (k.rows - 1)), (uint64_t)(k.cells / k.rows)};
        Case c(rows, k.types, 168.0, k.phi);
        CHECK(procell_simulate(&c.p, &c.r) == PROCELL_OK);
        const uint32_t per_cu = (uint32_t)(163840 / c.r.stats.lds_bytes);
        CHECK((per_cu > 3 ? 3 : per_cu) == k.per_cu && c.r.stats.window_rows >= k.window);
        printf("%u types to %g, %u rows, %g cells: %u per CU, %u window rows\n", c.p.n_types, k.top, k.rows, k.cells,
               per_cu, c.r.stats.window_rows);
    }
}

// The autotuner times no layout twice and reports the workgroups per CU that
// the plan runs with, also where later candidates are the faster ones.
static float g_ms = 100.0f;
static void check_autotune()
{
    fake::elapsed_ms = [] { return g_ms -= 0.5f; };
    for (double top : {1e5, 1e15}) {  // the second: trees so deep that a CU holds one or two workgroups
        std::vector<procell_row> rows(1024);
        for (int i = 0; i < 1024; ++i)
            rows[i] = {pow(top, i / 1023.0), 9765};
        Case c(rows, {{0.4, 35, 9}, {0.3, 55, 14}, {0.3, -1, -1}}, 240.0, 50.0);
        procell_plan *pl = nullptr;
        CHECK(procell_plan_create(&c.p, &pl) == PROCELL_OK);
        fake::launches.clear();
        const uint64_t seed = 1;
        procell_tuning t{};
        CHECK(procell_plan_autotune(pl, &seed, 1, &t) == PROCELL_OK);
        std::map<std::pair<unsigned, size_t>, int> runs;  // of each layout: four idle-lane thresholds, a warm-up and a run each
        for (const fake::Launch &l : fake::launches)
            if (l.kernel.find("sim_") != std::string::npos)
                ++runs[{l.grid, l.lds}];
        for (const auto &r : runs)
            CHECK(r.second == 8);
        CHECK(procell_plan_run(pl, 1) == PROCELL_OK && procell_plan_result(pl, &c.r) == PROCELL_OK);
        const uint32_t fit = std::min<uint32_t>(24 * 64 / c.r.stats.block_size, (uint32_t)(163840 / c.r.stats.lds_bytes));
        CHECK(t.blocks_per_cu >= 1 && t.blocks_per_cu <= fit);
        CHECK(procell_plan_destroy(pl) == PROCELL_OK);
    }
}

// A relaxed plan over very many sets: bounded lane stacks, every segment
// walked by one of a pass's launches.
static void check_stacks()
{
    for (uint32_t n : {1000u, 120000u}) {
        Case c({{8000.0, 1}}, {{1.0, 20.0, 5.0}}, 90.0, 1.0);
        std::vector<procell_params> sets(n, c.p);
        procell_relaxed *r = nullptr;
        fake::memory_bytes = 0;
        CHECK(procell_relaxed_create_batch(sets.data(), n, 0.5, &r) == PROCELL_OK);
        CHECK(fake::memory_bytes <= 8ull << 30);
        double x = 0.0;
        fake::launches.clear();
        CHECK(procell_relaxed_jacobian(r, &x, &x, &x, nullptr) == PROCELL_OK);
        uint64_t segments = 0, walks = 0;
        for (const fake::Launch &l : fake::launches)
            if (l.kernel.find("walk_kernel") != std::string::npos) {
                segments += l.grid;
                ++walks;
            }
        CHECK(segments == n && walks == (n > 1000 ? 3 : 1));
        CHECK(procell_relaxed_destroy(r) == PROCELL_OK);
    }
}

int main(int argc, char **argv)
{
    const struct {
        const char *name;
        void (*f)();
    } checks[] = {{"stage", check_stage}, {"noalloc", check_noalloc}, {"reset", check_reset}, {"kernel", check_kernel}, {"window", check_window},
                  {"autotune", check_autotune},
                  {"stacks", check_stacks}};
    for (const auto &c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.f();
            printf("%s: %d failed\n", c.name, g_failures);
            return g_failures ? 1 : 0;
        }
    fprintf(stderr, "usage: host_paths <check>\n");
    return 2;
}
