// Transfers between a caller's arrays and one block of device memory, through pinned memory.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstring>

#include "axiom/axm.h"

namespace axm {

// Large transfers go through the pinned block in two halves, one on the link while the host
// copies the other.  Pinned memory moves 57 GB/s here, pageable memory 17 GB/s down and 29 GB/s
// up (and a small copy takes 36 us instead of 13), so a transfer is bound by the host's own copy
// to or from the block.
constexpr size_t STAGE_PINNED = 8u << 20;

// One host array's place in the block.
struct StagePart {
    void* host;
    size_t off, bytes;
};

class Staging {
public:
    Staging() = default;
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    ~Staging() { release(); }

    uint8_t* dev() const { return dev_; }
    uint8_t* pinned() const { return pinned_; }

    // Room for `bytes` on the current device.
    axm_status ensure(size_t bytes) {
        if (cap_ < bytes) {
            if (dev_) (void)hipFree(dev_);
            dev_ = nullptr;
            cap_ = 0;
            if (hipMalloc((void**)&dev_, bytes) != hipSuccess) {
                dev_ = nullptr;
                return AXM_BUFFER_ALLOCATION_FAILED;
            }
            cap_ = bytes;
        }
        const size_t want = std::min(bytes, STAGE_PINNED);
        if (pinned_cap_ < want) {
            if (pinned_) (void)hipHostFree(pinned_);
            pinned_ = nullptr;
            pinned_cap_ = 0;
            if (hipHostMalloc((void**)&pinned_, want, hipHostMallocDefault) != hipSuccess) {
                pinned_ = nullptr;
                return AXM_BUFFER_ALLOCATION_FAILED;
            }
            pinned_cap_ = want;
        }
        for (hipEvent_t& e : ev_)
            if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return AXM_GPU_OPERATION_FAILED;
        return AXM_SUCCESS;
    }
    // Frees device memory above `bytes`.
    void trim(size_t bytes) {
        if (cap_ <= bytes) return;
        (void)hipFree(dev_);
        dev_ = nullptr;
        cap_ = 0;
    }
    void release() {
        if (dev_) (void)hipFree(dev_);
        if (pinned_) (void)hipHostFree(pinned_);
        for (hipEvent_t& e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        dev_ = pinned_ = nullptr;
        cap_ = pinned_cap_ = 0;
    }
    // The arrays to the block's bytes [0, total) on stream s; they are free on return.
    hipError_t up(const StagePart* part, int parts, size_t total, hipStream_t s) {
        const size_t piece = piece_of(total);
        for (size_t k = 0, lo = 0; lo < total; ++k, lo += piece) {
            const size_t hi = std::min(total, lo + piece);
            uint8_t* buf = pinned_ + (k & 1) * piece;
            hipError_t e = k >= 2 ? hipEventSynchronize(ev_[k & 1]) : hipSuccess;  // the piece before in this half
            if (e == hipSuccess) {
                copy(part, parts, lo, hi, buf, false);
                e = hipMemcpyAsync(dev_ + lo, buf, hi - lo, hipMemcpyHostToDevice, s);
            }
            if (e == hipSuccess) e = hipEventRecord(ev_[k & 1], s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    // The block's bytes [first, first + total) to the arrays (offsets from first), which are filled
    // on return.
    hipError_t down(const StagePart* part, int parts, size_t first, size_t total, hipStream_t s) {
        const size_t piece = piece_of(total), pieces = (total + piece - 1) / piece;
        for (size_t k = 0; k <= pieces; ++k) {
            hipError_t e = hipSuccess;
            if (k < pieces) {
                const size_t lo = k * piece, hi = std::min(total, lo + piece);
                e = hipMemcpyAsync(pinned_ + (k & 1) * piece, dev_ + first + lo, hi - lo, hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(ev_[k & 1], s);
            }
            if (e == hipSuccess && k > 0) {
                const size_t lo = (k - 1) * piece;
                e = hipEventSynchronize(ev_[(k - 1) & 1]);
                if (e == hipSuccess)
                    copy(part, parts, lo, std::min(total, lo + piece), pinned_ + ((k - 1) & 1) * piece, true);
            }
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }

private:
    size_t piece_of(size_t total) const { return total <= pinned_cap_ ? std::max<size_t>(total, 1) : pinned_cap_ / 2; }
    // Copies the part of the range [lo, hi) between the arrays and `buf`, which holds it.
    static void copy(const StagePart* part, int parts, size_t lo, size_t hi, uint8_t* buf, bool out) {
        for (int k = 0; k < parts; ++k) {
            const size_t a = std::max(lo, part[k].off), b = std::min(hi, part[k].off + part[k].bytes);
            if (a >= b) continue;
            uint8_t* h = static_cast<uint8_t*>(part[k].host) + (a - part[k].off);
            if (out) std::memcpy(h, buf + (a - lo), b - a);
            else std::memcpy(buf + (a - lo), h, b - a);
        }
    }

    uint8_t* dev_ = nullptr;
    size_t cap_ = 0;
    uint8_t* pinned_ = nullptr;
    size_t pinned_cap_ = 0;
    hipEvent_t ev_[2] = {nullptr, nullptr};
};

}  // namespace axm
