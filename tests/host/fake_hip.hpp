// fake_hip.hpp -- switches and records of the CPU stand-in for the HIP runtime
// (fake_hip.cpp), for the programs that drive libprocell's host code with it.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <string>
#include <vector>

namespace fake {

struct Launch {
    std::string kernel;  // mangled name
    unsigned grid, block;
    size_t lds;
};

extern std::vector<Launch> launches;       // every kernel that ran, in order
extern uint64_t sim_runs;                  // simulation kernels so far; each leaves this number as its sets' division counts
extern int fail_event_record;              // > 0: that many calls of hipEventRecord from now on, the last one fails
extern uint64_t dead_stream_uses;          // calls that named a stream that does not exist
extern uint64_t foreign_stream_uses;       // calls that named a stream of take_stream()
extern uint64_t streams_alive, memory_alive, memory_bytes;  // memory_bytes: the largest allocation so far
extern float (*elapsed_ms)();              // what hipEventElapsedTime reports
extern std::vector<uint32_t> segment_cells;  // the cells [first, end) of the walk kernel's segments, last launch

void device_reset();                       // hipDeviceReset: streams and memory are gone, their handles and addresses free
void take_stream();                        // the host program makes a stream
void take_memory();                        // the host program allocates device memory of the smallest size

}  // namespace fake
