// mpmw_readback.hpp -- device fields to host arrays in the caller's layout.
//
// A caller's array interleaves the components of a vector or matrix and is
// FP64, the device holds one array per component in the kernel precision.  A
// kernel widens and interleaves them straight into pinned host memory, one
// launch for as many arrays as fit a chunk, while the host moves the chunk
// before it out to the caller.  With a copy per component into pageable
// memory, a widening loop and a strided loop, a pass that ends in the state
// of 173 thousand FP64 particles took 25 ms, now 22; of 131 thousand
// F-tracking particles 31, now 26; in the sums of 2.1 M nodes 174, now 156.
#pragma once

#include <hip/hip_runtime.h>

#include "mpmw_readback_plan.hpp"

namespace mpmw_internal {

// Fills every array that has a destination with its first n rows, after the
// work already on `stream`.  Returns an MPMW_* status.
int read_back(int device, hipStream_t stream, const std::vector<ReadArray> &arrays, int64_t n);

}  // namespace mpmw_internal
