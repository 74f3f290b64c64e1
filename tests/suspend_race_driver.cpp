// An application suspends and resumes its own queue while the local scheduler's rounds do the
// same (every round resumes the queues that its policy lets run). After each of the
// application's resumes the queue has to make progress again, whatever the rounds did in between.
// Built against the libraries and run by tests/test_suspend_race.py.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>

#include <unistd.h>

#include "xsched/hint.h"
#include "xsched/host/hal.h"
#include "xsched/xqueue.h"

#define CHECK_X(call) do { XResult r_ = (call); if (r_ != kXSchedSuccess) { \
    fprintf(stderr, "%s -> %d\n", #call, (int)r_); _exit(3); } } while (0)

static void WorkGroup(void *, uint32_t, uint32_t)
{
    for (int spin = 0; spin < 300; ++spin) asm volatile("" ::: "memory");
}

int main(int argc, char **argv)
{
    const int rounds = argc > 1 ? atoi(argv[1]) : 3000;
    CHECK_X(XHintSetScheduler(kSchedulerLocal, kPolicyHighestPriorityFirst));
    HwQueueHandle hwq = 0;
    XQueueHandle xq = 0;
    CHECK_X(HostQueueCreate(&hwq));
    CHECK_X(XQueueCreate(&xq, hwq, kPreemptLevelDeactivate, kQueueCreateFlagNone));
    CHECK_X(XQueueSetLaunchConfig(xq, 2, 1));
    CHECK_X(XHintPriority(xq, 1));

    std::atomic<bool> stop { false };
    std::atomic<long> bursts { 0 };
    std::thread submitter([&]() {
        while (!stop.load()) {
            for (int i = 0; i < 16; ++i) {
                HwCommandHandle cmd = 0;
                CHECK_X(HostKernelCommandCreate(&cmd, WorkGroup, nullptr, 16, 1));
                CHECK_X(XQueueSubmit(xq, cmd));
            }
            CHECK_X(XQueueWaitAll(xq));
            bursts.fetch_add(1);
        }
    });
    uint64_t lcg = 99;
    for (int i = 0; i < rounds; ++i) {
        lcg = lcg * 6364136223846793005ull + 1442695040888963407ull;
        std::this_thread::sleep_for(std::chrono::microseconds(20 + (lcg >> 33) % 200));
        CHECK_X(XQueueSuspend(xq, kQueueSuspendFlagSyncHwQueue));
        std::this_thread::sleep_for(std::chrono::microseconds(30));
        CHECK_X(XQueueResume(xq, kQueueResumeFlagNone));
        const long before = bursts.load();
        const auto give_up = std::chrono::steady_clock::now() + std::chrono::seconds(10);
        while (bursts.load() == before) {
            if (std::chrono::steady_clock::now() > give_up) {
                printf("stuck after resume %d\n", i);
                fflush(stdout);
                _exit(1);
            }
            std::this_thread::yield();
        }
    }
    stop.store(true);
    submitter.join();
    CHECK_X(XQueueDestroy(xq));
    CHECK_X(HwQueueDestroy(hwq));
    printf("%d suspensions, %ld bursts\n", rounds, bursts.load());
    return 0;
}
