// Drives lucida_amd/csrc/side_stream.hpp against stand-ins for the four HIP calls
// it makes: streams are counters of queued work, an event the amount that it
// was recorded at. No device and no HIP library.
#include <cstdio>
#include <cstdlib>

#include "side_stream.hpp"

struct ihipStream_t {
    int queued = 0, after_other = 0;  // work queued; how much of the other stream's precedes what comes next
};
struct ihipEvent_t {
    int at = -1;
};

static int fail_records = 0, fail_waits = 0, synchronized = 0;

extern "C" hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (fail_records) return hipErrorUnknown;
    e->at = s->queued;
    return hipSuccess;
}
extern "C" hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    if (fail_waits) return hipErrorUnknown;
    s->after_other = e->at;
    return hipSuccess;
}
extern "C" hipError_t hipStreamSynchronize(hipStream_t s) {
    synchronized = s->queued;
    return hipSuccess;
}

static void expect(bool ok, const char* what) {
    if (ok) return;
    std::printf("failed: %s\n", what);
    std::exit(1);
}

static ihipStream_t first, second;
static ihipEvent_t ready, done;

// Three steps with work on both streams; `stop` is the step whose work on the
// first stream fails after the second's has been queued (3: none).
static bool steps(int stop, bool join) {
    first = second = ihipStream_t{};
    ready = done = ihipEvent_t{};
    synchronized = 0;
    lucida::SideStream side(&first, &second, &ready, &done);
    for (int k = 0; k < 3; ++k) {
        first.queued += 1;
        if (side.fork() != hipSuccess) return false;
        expect(second.after_other == k + 1, "the second stream waits for the first's work");
        second.queued += 1;
        if (k == stop) return false;
    }
    return !join || side.join() == hipSuccess;
}

int main() {
    expect(steps(3, true) && first.after_other == 3, "joined");
    for (int stop = 0; stop < 3; ++stop) {
        expect(!steps(stop, true), "an error is reported");
        expect(first.after_other == stop + 1, "a return on an error joins the second stream's work");
        expect(synchronized == 0, "without a wait on the host");
    }
    expect(steps(3, false) && first.after_other == 3, "the end of the scope joins");
    fail_waits = 1;
    expect(!steps(3, true) && first.after_other == 0 && synchronized == second.queued, "no join: the host waits");
    fail_waits = 0;
    fail_records = 1;
    expect(!steps(3, true), "a failed fork is reported");
    std::printf("ok\n");
    return 0;
}
