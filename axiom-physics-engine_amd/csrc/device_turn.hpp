// Order between the steps of different worlds on one device.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <condition_variable>
#include <mutex>

#include "axiom/axm.h"

namespace axm {

// Kernels of a step (colouring, sorts, sweeps, scans) have workgroups that wait for others of
// their own grid, so a grid must become resident as a whole.  The sweeps take a CU's whole LDS per
// workgroup: two worlds' grids at once could each hold CUs that the other waits for, until the
// bounded waits give up.  So the steps of a device's worlds run one after the other: whoever
// enqueues holds the device's turn, and its stream first waits for what the stream that had the
// turn before may still run.  Turns go in the order they are asked for.  A world alone, or worlds
// stepped in turn, wait for nothing (a stream that its host has seen idle is not waited for).
class DeviceTurn {
public:
    static DeviceTurn& of(int32_t device);
    static constexpr int32_t DEVICES = 256;

    // Takes the turn for work on `stream`; `event` is that stream's own for this.
    hipError_t enter(hipStream_t stream, hipEvent_t event) {
        std::unique_lock<std::mutex> lk(mu_);
        const uint64_t mine = next_++;
        cv_.wait(lk, [&] { return serving_ == mine; });
        hipError_t e = hipSuccess;
        if (busy_ && busy_ != stream) {
            e = hipEventRecord(event, busy_);
            if (e == hipSuccess) e = hipStreamWaitEvent(stream, event, 0);
        }
        if (e == hipSuccess) busy_ = stream;
        return e;
    }
    void leave() {
        {
            std::lock_guard<std::mutex> lk(mu_);
            ++serving_;
        }
        cv_.notify_all();
    }
    // All work on the stream is done.
    void idle(hipStream_t stream) {
        std::lock_guard<std::mutex> lk(mu_);
        if (busy_ == stream) busy_ = nullptr;
    }

private:
    std::mutex mu_;
    std::condition_variable cv_;
    uint64_t next_ = 0, serving_ = 0;
    hipStream_t busy_ = nullptr;  // had the turn last, and may still run

    union Kept;  // one turn per device, never destroyed: threads may outlive the statics
};
union DeviceTurn::Kept {
    DeviceTurn turn[DEVICES];
    Kept() : turn() {}
    ~Kept() {}
};
inline DeviceTurn& DeviceTurn::of(int32_t device) {
    static Kept all;
    return all.turn[device];
}

// One turn, until the end of the scope.
class Turn {
public:
    Turn(int32_t device, hipStream_t stream, hipEvent_t event) : t_(DeviceTurn::of(device)) {
        ok_ = t_.enter(stream, event) == hipSuccess;
    }
    ~Turn() { t_.leave(); }
    Turn(const Turn&) = delete;
    Turn& operator=(const Turn&) = delete;
    axm_status status() const { return ok_ ? AXM_SUCCESS : AXM_GPU_OPERATION_FAILED; }

private:
    DeviceTurn& t_;
    bool ok_;
};

}  // namespace axm
