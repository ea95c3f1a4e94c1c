// Work on a second stream beside a first. fork() has the second wait for what
// the first has queued; join() has the first wait for all that the second has
// queued. A fork that was not joined is joined at the end of the scope: a return
// on an error leaves nothing on the second stream that later work on the first
// could overtake (and, say, overwrite its inputs).
#pragma once
#include <hip/hip_runtime_api.h>

namespace lucida {

class SideStream {
public:
    SideStream(hipStream_t first, hipStream_t second, hipEvent_t ready, hipEvent_t done)
        : first_(first), second_(second), ready_(ready), done_(done) {}
    SideStream(const SideStream&) = delete;
    SideStream& operator=(const SideStream&) = delete;
    ~SideStream() {
        if (open_) (void)join();
    }
    hipError_t fork() {
        open_ = true;
        const hipError_t e = hipEventRecord(ready_, first_);
        return e != hipSuccess ? e : hipStreamWaitEvent(second_, ready_, 0);
    }
    // Where the streams cannot be joined, the host waits for the second.
    hipError_t join() {
        open_ = false;
        hipError_t e = hipEventRecord(done_, second_);
        if (e == hipSuccess) e = hipStreamWaitEvent(first_, done_, 0);
        if (e != hipSuccess) (void)hipStreamSynchronize(second_);
        return e;
    }

private:
    hipStream_t first_, second_;
    hipEvent_t ready_, done_;
    bool open_ = false;
};

}  // namespace lucida
