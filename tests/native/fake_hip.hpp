// A stand-in for the HIP runtime and the kernels, for tests of what the host
// code does with device memory, streams and graphs.  It runs on the CPU and
// computes no results: device memory is a set of address ranges (never given
// out twice), a launch only asks that the arrays it was given are allocated
// when it runs, and a stream under capture collects its work for a graph.
// Calls that HIP refuses during a capture (allocation, synchronous copies, in
// a mode that forbids them) fail here and end the capture in error.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace fake {
extern size_t memory;      // bytes of the device
extern size_t used;        // allocated now
extern int dead_accesses;  // launches and copies that met memory not allocated
extern int launches;       // kernels run, replays included
extern int graph_launches;
extern int allocations;
}  // namespace fake
