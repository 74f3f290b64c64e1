// A foreground queue beside a background queue that its commands interrupt, on the host adapter
// and the local scheduler's highest-priority-first policy. Built against the libraries and run by
// tests/test_foreground_bursts.py.
//   burst_driver bursts N GAP   N bursts of 20 foreground commands of 30 us, each waited for, GAP us between
//                               them, over background commands of 2 ms in work-groups of 5 us that
//                               a deactivation flushes. Prints the background's replays per burst
//                               and the foreground's median latency.
//   burst_driver waited N       a queue suspended by the application after its commands have
//   burst_driver stopped N      finished, or in its work; beside it N commands of 400 us of another
//                               queue, far apart. Prints the processor time that this
//                               queue's launcher uses per command.
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <filesystem>
#include <set>
#include <vector>

#include <time.h>
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
static void Sleep400us(void *, uint32_t, uint32_t) { usleep(400); }

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

static std::set<int> Threads()
{
    std::set<int> tids;
    for (const auto &e : std::filesystem::directory_iterator("/proc/self/task")) tids.insert(atoi(e.path().filename().c_str()));
    return tids;
}

/// Processor time that a thread of this process has used.
static double ThreadMicros(int tid)
{
    timespec t {};
    const clockid_t clock = ((~(clockid_t)tid) << 3) | 6;   // the kernel's number for the thread's processor-time clock
    if (clock_gettime(clock, &t) != 0) { perror("clock_gettime"); _exit(4); }
    return (double)t.tv_sec * 1e6 + (double)t.tv_nsec * 1e-3;
}

static void Beside(int commands, bool finished)
{
    CHECK_X(XHintSetScheduler(kSchedulerAppManaged, kPolicyUnknown));
    HwQueueHandle other_hw = 0, hw = 0;
    XQueueHandle other = 0, xq = 0;
    Make(&other_hw, &other, kPreemptLevelDeactivate, 0);
    CHECK_X(HostQueueCreate(&hw));
    const std::set<int> threads = Threads();
    CHECK_X(XQueueCreate(&xq, hw, kPreemptLevelDeactivate, kQueueCreateFlagNone));
    int launcher = -1;
    for (const int tid : Threads()) if (threads.count(tid) == 0) launcher = tid;
    Submit(other, WorkGroup5us, 400, 1);
    CHECK_X(XQueueSuspend(other, finished ? kQueueSuspendFlagWaitAll : kQueueSuspendFlagNone));

    const double before = ThreadMicros(launcher);
    for (int i = 0; i < commands; ++i) {
        XQueueState state = kQueueStateUnknown;
        CHECK_X(XQueueQuery(xq, &state));   // somebody follows the queue: the next command is launched by its submitter
        Submit(xq, Sleep400us, 1, 0);
        usleep(1000);
    }
    printf("%.1f us of the launcher per command\n", (ThreadMicros(launcher) - before) / commands);
    CHECK_X(XQueueResume(other, kQueueResumeFlagNone));
    CHECK_X(XQueueWaitAll(other)); CHECK_X(XQueueWaitAll(xq));
    CHECK_X(XQueueDestroy(xq)); CHECK_X(XQueueDestroy(other));
    CHECK_X(HwQueueDestroy(hw)); CHECK_X(HwQueueDestroy(other_hw));
}

int main(int argc, char **argv)
{
    if (argc < 3) return 2;
    const int count = atoi(argv[2]);
    if (strcmp(argv[1], "bursts") == 0) Bursts(count, argc > 3 ? atoi(argv[3]) : 0);
    else Beside(count, strcmp(argv[1], "waited") == 0);
    return 0;
}
