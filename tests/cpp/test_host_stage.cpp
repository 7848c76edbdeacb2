// HostStage (inspire-gpu_amd/csrc/server/host_stage.h) on the CPU: with as
// many helper threads as the process can have (fewer than asked for, here by
// a limit on its address space), every item of a job is done once, and a
// failed one is reported once everything has been waited for.
#include <pthread.h>
#include <sys/resource.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <stdexcept>

#include "host_stage.h"

static void check(bool ok, const char* what) {
    if (ok) return;
    std::printf("failed: %s\n", what);
    std::exit(1);
}

static void run_jobs(size_t helpers) {
    constexpr size_t kItems = 64;
    inspire::HostStage st(helpers, kItems);
    for (size_t n : {(size_t)1, (size_t)7, kItems}) {
        for (int bad = 0; bad < 2; bad++) {
            std::atomic<int> times[kItems] = {};
            bool threw = false;
            st.begin(n, [&](size_t i) {
                times[i]++;
                if (bad && i == n / 2) throw std::runtime_error("item");
            }, n > 1);
            try {
                for (size_t k = 1; k <= n; k++) st.wait(k);
            } catch (const std::runtime_error&) {
                threw = true;
            }
            const bool ok = st.finish();
            for (size_t i = 0; i < kItems; i++) check(times[i] == (i < n ? 1 : 0), "every item once");
            check(!threw, "a failed item does not end the waits");
            check(ok == (bad == 0) && st.finish() == ok, "failures are reported at the end");
        }
    }
}

int main() {
    run_jobs(0);
    run_jobs(3);
    // 1 GiB of stack per thread, address space for one of three
    pthread_attr_t a;
    check(pthread_attr_init(&a) == 0 && pthread_attr_setstacksize(&a, (size_t)1 << 30) == 0 &&
              pthread_setattr_default_np(&a) == 0, "thread attributes");
    const rlimit lim{(rlim_t)2 << 30, (rlim_t)2 << 30};
    check(setrlimit(RLIMIT_AS, &lim) == 0, "address space limit");
    run_jobs(3);
    std::printf("host stage checks passed\n");
    return 0;
}
