// Device arrays to the caller's (pageable) host arrays.
#pragma once

#include <cstddef>
#include <mutex>

#include <hip/hip_runtime.h>

namespace ibt {

constexpr int HC_THREADS = 4;                   // host threads of a large copy
constexpr size_t HC_SLOT = (size_t)2 << 20;     // bytes of a pinned slot, two per thread
// bytes on the device from which copies are staged (six arrays, ms direct /
// staged: 300 x 300, 4.4 MB, 0.24 / 0.30; 512 x 384, 9.7 MB, 0.55 / 0.40)
constexpr size_t HC_STAGED = (size_t)8 << 20;

// The pinned slots of one context or ensemble (16 MB, allocated by its first
// large copy, freed with it); one copy at a time uses them.
struct HostCopy {
    std::mutex use;
    char *pin = nullptr;
    hipEvent_t ev[2 * HC_THREADS] = {};
};

// n numbers on the device to n doubles on the host; f32: floats, widened.
struct HostPart {
    double *dst;
    const void *src;
    size_t n;
    bool f32;
};

// Copies all parts behind the stream's work and waits for them; on return the
// host arrays hold the values.  Several threads may copy from one object at a
// time.  Errors leave a message and return its code; nothing is thrown.
int host_copy(int device, hipStream_t stream, HostCopy &h, const HostPart *parts, int nparts);
void host_copy_release(HostCopy &h);

}  // namespace ibt
