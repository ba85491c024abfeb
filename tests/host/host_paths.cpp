// host_paths.cpp -- libprocell's host code over the stand-in HIP runtime
// (fake_hip.cpp): which device memory, streams and launches the entry points
// use, and which run their results come from.  usage: host_paths <check>; exit
// status 0 when it held.
#include <stdio.h>
#include <string.h>

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

int main(int argc, char **argv)
{
    const struct {
        const char *name;
        void (*f)();
    } checks[] = {{"stage", check_stage}, {"noalloc", check_noalloc}, {"reset", check_reset}};
    for (const auto &c : checks)
        if (argc == 2 && !strcmp(argv[1], c.name)) {
            c.f();
            printf("%s: %d failed\n", c.name, g_failures);
            return g_failures ? 1 : 0;
        }
    fprintf(stderr, "usage: host_paths <check>\n");
    return 2;
}
