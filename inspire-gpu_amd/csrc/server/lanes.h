// The streams that pipelined answers run on: per device, kLaneSets sets of
// three (database passes, Horner chains, collapse or pack), shared by the
// device's servers and released with the last of them.
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

namespace inspire {

constexpr int kLaneSets = 4;
struct LaneStreams {
    hipStream_t pass = nullptr, horner = nullptr, side = nullptr;
};
// A server's sets, lane 0 first: the least-used set and the others after it.
// Throws std::runtime_error where the streams cannot be created.
int acquire_lanes(int device, LaneStreams (&out)[kLaneSets]);
void release_lanes(int device, int first);
// How many of a device's sets have streams that run side by side now (on an
// idle device).
int lanes_apart(int device);

// A thread's turn to put waits into a device's queues. Streams share a few
// hardware queues, and a stream's wait for an event holds up whatever was
// enqueued behind it in its hardware queue, other streams' kernels too. A
// streamed answer's pack and chains wait inside their kernels, for a bounded
// time, for kernels enqueued after their release: it enqueues all of them in
// one turn, so no other thread's wait (for a caller's busy stream, say) gets
// between. A thread may take a turn within its turn.
class QueueTurn {
public:
    explicit QueueTurn(int device) : lk_(mutex(device)) {}

private:
    static std::recursive_mutex& mutex(int device);
    std::lock_guard<std::recursive_mutex> lk_;
};

}  // namespace inspire
