// Streams of one set have to sit on different hardware queues: a process has
// 4, HIP maps streams to them by its own counts, and kernels of two streams
// on one queue run one after another, so that chains waiting beside their
// pass only start when it ends (16 GB, 32 queries: 5.5 ms per answer where
// the three are apart, 7.0 or 8.1 ms where two share a queue). The mapping
// cannot be asked for, so a set is put together from streams whose kernels
// are seen to run side by side.
#include "lanes.h"

#include <algorithm>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "kernels.h"
#include "trace.h"

namespace inspire {

namespace {

constexpr int kMaxDevices = 64;
// Polls of 128 clocks and a load, about 1 ms: far above the launch of a second
// kernel on an idle device. Beside other work that launch may take longer
// (four threads with 2 ms of kernels in flight each: sets of one to three
// streams apart were found), so where a set stays incomplete its remaining
// candidates are tried again with the longer wait, which only a kernel behind
// the waiting one on its own queue uses up.
constexpr uint32_t kProbePolls[] = {2000, 60000};
constexpr int kProbeStreams = 10;  // candidates tried for one set

// words: [0] the flag, [1] whether the waiting kernel saw it
__global__ void k_probe_wait(uint32_t* words, uint32_t polls) {
    uint32_t seen = 0;
    for (uint32_t i = 0; i < polls && !seen; i++) {
        seen = __hip_atomic_load(words, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_sleep(2);
    }
    __hip_atomic_store(words + 1, seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__global__ void k_probe_set(uint32_t* words) {
    __hip_atomic_store(words, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

void check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// Whether a kernel on b runs while one enqueued before it on a still runs.
bool side_by_side(hipStream_t a, hipStream_t b, uint32_t* d_words, uint32_t polls = kProbePolls[0]) {
    check(ipx::launch_fill_u32(d_words, 2, 0, a), "stream probe");
    check(hipStreamSynchronize(a), "stream probe");
    hipLaunchKernelGGL(k_probe_wait, dim3(1), dim3(1), 0, a, d_words, polls);
    hipLaunchKernelGGL(k_probe_set, dim3(1), dim3(1), 0, b, d_words);
    check(hipGetLastError(), "stream probe");
    check(hipStreamSynchronize(a), "stream probe");
    check(hipStreamSynchronize(b), "stream probe");
    uint32_t seen = 0;
    check(hipMemcpy(&seen, d_words + 1, 4, hipMemcpyDeviceToHost), "stream probe");
    return seen != 0;
}

struct DeviceLanes {
    int servers = 0;
    int users[kLaneSets] = {};
    LaneStreams set[kLaneSets];
};
std::mutex g_mu;
DeviceLanes g_lanes[kMaxDevices];

void destroy(DeviceLanes& d) {
    for (LaneStreams& s : d.set) {
        for (hipStream_t x : {s.pass, s.horner, s.side})
            if (x) (void)hipStreamDestroy(x);
        s = LaneStreams{};
    }
}

void create(DeviceLanes& d) {
    uint32_t* words = nullptr;
    std::vector<hipStream_t> spare;
    bool few = false;  // the longer waits did not complete a set either
    auto cleanup = [&] {
        for (hipStream_t x : spare) (void)hipStreamDestroy(x);
        if (words) (void)hipFree(words);
    };
    try {
        check(hipMalloc((void**)&words, 8), "stream probe");
        for (LaneStreams& s : d.set) {
            std::vector<hipStream_t> got;
            // Streams left over from earlier sets first, then new ones. The
            // rejected ones live until every set is complete: destroyed early,
            // their queue would be the next stream's again.
            for (const uint32_t polls : kProbePolls) {
                if (polls != kProbePolls[0] && few) break;
                for (int k = 0; k < kProbeStreams && got.size() < 3; k++) {
                    if ((size_t)k >= spare.size()) {
                        hipStream_t x = nullptr;
                        check(hipStreamCreate(&x), "hipStreamCreate");
                        spare.push_back(x);
                    }
                    const hipStream_t x = spare[k];
                    bool apart = std::find(got.begin(), got.end(), x) == got.end();
                    for (size_t i = 0; i < got.size() && apart; i++) apart = side_by_side(got[i], x, words, polls);
                    if (apart) got.push_back(x);
                }
            }
            few = few || got.size() < 3;
            while (got.size() < 3) {  // fewer queues than roles, or a very busy device: any will do
                hipStream_t x = nullptr;
                check(hipStreamCreate(&x), "hipStreamCreate");
                spare.push_back(x);
                got.push_back(x);
            }
            for (hipStream_t x : got)
                for (size_t i = 0; i < spare.size(); i++)
                    if (spare[i] == x) {
                        spare.erase(spare.begin() + i);
                        break;
                    }
            s.pass = got[0];
            s.horner = got[1];
            s.side = got[2];
            const int l = (int)(&s - d.set);
            static const char* names[kLaneSets][3] = {{"passes 0", "horner 0", "side 0"},
                                                      {"passes 1", "horner 1", "side 1"},
                                                      {"passes 2", "horner 2", "side 2"},
                                                      {"passes 3", "horner 3", "side 3"}};
            trace_name_stream(s.pass, names[l][0]);
            trace_name_stream(s.horner, names[l][1]);
            trace_name_stream(s.side, names[l][2]);
        }
    } catch (...) {
        cleanup();
        destroy(d);
        throw;
    }
    cleanup();
}

}  // namespace

int acquire_lanes(int device, LaneStreams (&out)[kLaneSets]) {
    if (device < 0 || device >= kMaxDevices) throw std::runtime_error("acquire_lanes: device out of range");
    std::lock_guard<std::mutex> lk(g_mu);
    DeviceLanes& d = g_lanes[device];
    if (d.servers == 0) create(d);
    d.servers++;
    int first = 0;
    for (int l = 1; l < kLaneSets; l++)
        if (d.users[l] < d.users[first]) first = l;
    d.users[first]++;
    for (int l = 0; l < kLaneSets; l++) out[l] = d.set[(first + l) % kLaneSets];
    return first;
}

std::recursive_mutex& QueueTurn::mutex(int device) {
    static std::recursive_mutex m[kMaxDevices];
    return m[device >= 0 && device < kMaxDevices ? device : 0];
}

int lanes_apart(int device) {
    if (device < 0 || device >= kMaxDevices) return 0;
    std::lock_guard<std::mutex> lk(g_mu);
    DeviceLanes& d = g_lanes[device];
    if (d.servers == 0) return 0;
    uint32_t* words = nullptr;
    check(hipMalloc((void**)&words, 8), "stream probe");
    int n = 0;
    try {
        for (const LaneStreams& s : d.set)
            n += side_by_side(s.pass, s.horner, words) && side_by_side(s.pass, s.side, words) &&
                 side_by_side(s.horner, s.side, words);
    } catch (...) {
        (void)hipFree(words);
        throw;
    }
    (void)hipFree(words);
    return n;
}

void release_lanes(int device, int first) {
    std::lock_guard<std::mutex> lk(g_mu);
    DeviceLanes& d = g_lanes[device];
    d.users[first]--;
    if (--d.servers == 0) destroy(d);
}

}  // namespace inspire
