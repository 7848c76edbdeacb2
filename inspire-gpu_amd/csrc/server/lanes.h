// The streams that pipelined answers run on: per device, kLaneSets sets of
// three (database passes, Horner chains, collapse or pack), shared by the
// device's servers and released with the last of them.
#pragma once
#include <hip/hip_runtime.h>

namespace inspire {

constexpr int kLaneSets = 4;
struct LaneStreams {
    hipStream_t pass = nullptr, horner = nullptr, side = nullptr;
};
// A server's sets, lane 0 first: the least-used set and the others after it.
// Throws std::runtime_error where the streams cannot be created.
int acquire_lanes(int device, LaneStreams (&out)[kLaneSets]);
void release_lanes(int device, int first);

}  // namespace inspire
