// Synchronous copies and fills beside other threads' stream captures.
#pragma once
#include <hip/hip_runtime.h>

#include <shared_mutex>

namespace axm {

// hipMemcpy and hipMemset use the null stream.  While any thread captures a stream, the runtime
// refuses them to every thread (hipErrorStreamCaptureImplicit) and gives up the capture too, also one
// begun in thread-local mode.  So captures hold this lock alone and these calls share it.
inline std::shared_mutex& capture_lock() {
    union Kept {  // never destroyed: threads may outlive the statics
        std::shared_mutex m;
        Kept() : m() {}
        ~Kept() {}
    };
    static Kept kept;
    return kept.m;
}
inline hipError_t copy_sync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
    std::shared_lock<std::shared_mutex> lk(capture_lock());
    return hipMemcpy(dst, src, bytes, kind);
}
inline hipError_t fill_sync(void* dst, int value, size_t bytes) {
    std::shared_lock<std::shared_mutex> lk(capture_lock());
    return hipMemset(dst, value, bytes);
}

}  // namespace axm
