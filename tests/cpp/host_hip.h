// The part of the HIP runtime that the library's host code calls, on host memory
// (host_hip.cpp): device and pinned allocations are the heap's, copies are made at
// once, streams, events and graphs do nothing.  Kernel launch functions come from
// the program that links it, or do nothing (tests/host_build.py).
#pragma once
#include <cstddef>
#include <cstdint>

namespace host_hip {

extern int units;              // compute units of the device
extern bool no_pinned;         // hipHostMalloc fails
extern int64_t mallocs_left;   // device allocations until one fails, and all after it
extern int64_t device_bytes;   // allocated now
extern int64_t mallocs;        // device allocations so far

}  // namespace host_hip
