// A foreground queue beside a background queue that its commands interrupt, on the host adapter
// and the local scheduler's highest-priority-first policy. Built against the libraries and run by
// tests/test_foreground_bursts.py.
//   burst_driver bursts N GAP   N bursts of 20 foreground commands of 30 us, each waited for, GAP us between
//                               them, over background commands of 2 ms in work-groups of 5 us that
//                               a deactivation flushes. Prints the background's replays per burst
//                               and the foreground's median latency.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <unistd.h>

#include "xsched/hint.h"
#include "xsched/host/hal.h"
#include "xsched/xqueue.h"

#define CHECK_X(call) do { XResult r_ = (call); if (r_ != kXSchedSuccess) { \
    fprintf(stderr, "%s -> %d\n", #call, (int)r_); _exit(3); } } while (0)

using Clock = std::chrono::steady_clock;

static double Micros(Clock::duration d) { return std::chrono::duration<double, std::micro>(d).count(); }

static void Busy(double us)
{
    const auto end = Clock::now() + std::chrono::nanoseconds((int64_t)(us * 1e3));
    while (Clock::now() < end) {}
}
static void WorkGroup5us(void *, uint32_t, uint32_t) { Busy(5); }

static void Make(HwQueueHandle *hwq, XQueueHandle *xq, XPreemptLevel level, int priority)
{
    CHECK_X(HostQueueCreate(hwq));
    CHECK_X(XQueueCreate(xq, *hwq, level, kQueueCreateFlagNone));
    CHECK_X(XQueueSetLaunchConfig(*xq, 8, 4));
    CHECK_X(XHintPriority(*xq, priority));
}

static void Submit(XQueueHandle xq, HostKernelFn fn, uint32_t work_groups, int guarded)
{
    HwCommandHandle cmd = 0;
    CHECK_X(HostKernelCommandCreate(&cmd, fn, nullptr, work_groups, guarded));
    CHECK_X(XQueueSubmit(xq, cmd));
}

static uint64_t Replays(HwQueueHandle hwq)
{
    uint64_t executed = 0, skipped = 0, replays = 0;
    CHECK_X(HostQueueGetStats(hwq, &executed, &skipped, &replays));
    return replays;
}

static void Bursts(int bursts, int gap_us)
{
    CHECK_X(XHintSetScheduler(kSchedulerLocal, kPolicyHighestPriorityFirst));
    HwQueueHandle bg_hw = 0, fg_hw = 0;
    XQueueHandle bg = 0, fg = 0;
    Make(&bg_hw, &bg, kPreemptLevelDeactivate, 0);
    Make(&fg_hw, &fg, kPreemptLevelDeactivate, 1);
    CHECK_X(XQueueSetLaunchConfig(bg, 2, 1));
    usleep(50000);   // the hints are folded in by the scheduler's own thread

    std::vector<double> latency;
    const uint64_t before = Replays(bg_hw);
    for (int b = 0; b < bursts; ++b) {
        Submit(bg, WorkGroup5us, 400, 1);
        Submit(bg, WorkGroup5us, 400, 1);
        Busy(300);
        for (int i = 0; i < 20; ++i) {
            const auto t = Clock::now();
            Submit(fg, WorkGroup5us, 6, 1);
            CHECK_X(XQueueWaitAll(fg));
            latency.push_back(Micros(Clock::now() - t));
            if (gap_us > 0) Busy(gap_us);
        }
        CHECK_X(XQueueWaitAll(bg));
    }
    std::sort(latency.begin(), latency.end());
    printf("%.2f replays per burst, %.1f us p50\n", (double)(Replays(bg_hw) - before) / bursts, latency[latency.size() / 2]);
    CHECK_X(XQueueDestroy(fg)); CHECK_X(XQueueDestroy(bg));
    CHECK_X(HwQueueDestroy(fg_hw)); CHECK_X(HwQueueDestroy(bg_hw));
}

int main(int argc, char **argv)
{
    if (argc < 4 || strcmp(argv[1], "bursts") != 0) return 2;
    Bursts(atoi(argv[2]), atoi(argv[3]));
    return 0;
}
