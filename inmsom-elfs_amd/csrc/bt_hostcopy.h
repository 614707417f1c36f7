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
// bytes that an object copies without slots before it makes them: the copy that
// does takes up to 2 ms longer (the host's page faults on 16 MB; little where the
// process had freed such memory before), which staging saves over 60 MB.  ms of
// a context's first read, direct / making the slots, first in the process and
// later: 512 x 384, 10 MB, 0.7 / 2.0, 2.0; 700 x 600, 20 MB, 1.4 / 2.7, 2.7; 1021 x
// 763, 37 MB, 2.4 / 3.1, 1.4; 1400 x 1200, 81 MB, 5.0 / 4.3, 2.5; 2048 x 1536,
// 151 MB, 9.2 / 6.4, 4.5.
constexpr size_t HC_FIRST = (size_t)32 << 20;

// The pinned slots of one context or ensemble (16 MB, made by the large copy
// that passes HC_FIRST, freed with it); one copy at a time uses them.
struct HostCopy {
    std::mutex use;
    size_t direct = 0;  // bytes of large copies made without slots
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
// time.  whole: bytes of the reads that this copy is one of (an ensemble's members
// are read one after the other), where they are more than its own.  Errors leave
// a message and return its code; nothing is thrown.
int host_copy(int device, hipStream_t stream, HostCopy &h, const HostPart *parts, int nparts, size_t whole = 0);
void host_copy_release(HostCopy &h);

}  // namespace ibt
