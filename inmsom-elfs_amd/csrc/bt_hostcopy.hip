// Copies of device arrays to pageable host arrays (bt_hostcopy.h).
//
// The runtime's own copy to pageable memory goes through one staging buffer on
// one thread, which then also takes the page faults of a new array: 10 to 17
// GB/s.  Here HC_THREADS host threads each move their chunks (chunk c to thread
// c % HC_THREADS) through two pinned slots: the next chunk is under way while
// the last one is copied out, or widened.  Measured on MI355X (six arrays, ms
// before / now): 1021 x 763 2.1 / 1.07, 2048 x 1536 8.7 / 3.9 (38 GB/s: the link;
// 2 or 8 threads the same, slots of 1 MB 4.9), FP32 widened 9.3 / 3.1; the copy
// that makes the slots takes up to 2 ms longer (HC_FIRST).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "bt_hostcopy.h"
#include "bt_internal.h"

namespace ibt {

namespace {

size_t elem(const HostPart &q) { return q.f32 ? sizeof(float) : sizeof(double); }

int hc_fail(hipError_t e)
{
    set_error(std::string("copy to the host: ") + hipGetErrorString(e));
    return INMSOM_BT_EDEVICE;
}

// without staging: small copies, and where pinned memory cannot be had
int copy_direct(hipStream_t stream, const HostPart *parts, int nparts)
{
    std::vector<float> t;
    for (int k = 0; k < nparts; ++k) {
        const HostPart &q = parts[k];
        if (q.f32 && t.size() < q.n) {
            try {
                t.resize(q.n);
            } catch (const std::bad_alloc &) {
                set_error("copy to the host: out of memory");
                return INMSOM_BT_ENOMEM;
            }
        }
        hipError_t e = hipMemcpyAsync(q.f32 ? (void *)t.data() : q.dst, q.src, q.n * elem(q), hipMemcpyDeviceToHost,
                                      stream);
        if (e == hipSuccess && (q.f32 || k == nparts - 1)) e = hipStreamSynchronize(stream);
        if (e != hipSuccess) return hc_fail(e);
        if (q.f32) std::copy(t.begin(), t.begin() + (ptrdiff_t)q.n, q.dst);
    }
    return INMSOM_BT_OK;
}

// Chunk c of the parts, each of which is cut into whole slots and a rest.
struct Chunk {
    const HostPart *part;
    size_t first, n;
};
size_t chunks_of(const HostPart &q)
{
    const size_t per = HC_SLOT / elem(q);
    return (q.n + per - 1) / per;
}
Chunk chunk_at(const HostPart *part, size_t c)
{
    for (; c >= chunks_of(*part); ++part) c -= chunks_of(*part);
    const size_t per = HC_SLOT / elem(*part);
    return Chunk{part, c * per, std::min(per, part->n - c * per)};
}

// chunks t, t + step, .. of `total` through two slots
void copy_chunks(int device, hipStream_t stream, HostCopy &h, const HostPart *parts, size_t total, int t, int step,
                 std::atomic<int> &err)
{
    auto failed = [&](hipError_t e) {
        if (e != hipSuccess) err.store((int)e);
        return e != hipSuccess || err.load() != 0;
    };
    if (failed(hipSetDevice(device))) return;
    auto issue = [&](size_t c, int slot) {
        const Chunk q = chunk_at(parts, c);
        const size_t es = elem(*q.part);
        const hipError_t e = hipMemcpyAsync(h.pin + (size_t)slot * HC_SLOT, (const char *)q.part->src + q.first * es,
                                            q.n * es, hipMemcpyDeviceToHost, stream);
        return e != hipSuccess ? e : hipEventRecord(h.ev[slot], stream);
    };
    int cur = 2 * t;
    if ((size_t)t < total && failed(issue((size_t)t, cur))) return;
    for (size_t c = (size_t)t; c < total; c += (size_t)step) {
        const int nxt = cur ^ 1;
        // the other slot was copied out in the round before
        if (c + (size_t)step < total && failed(issue(c + (size_t)step, nxt))) break;
        if (failed(hipEventSynchronize(h.ev[cur]))) break;
        const Chunk q = chunk_at(parts, c);
        const char *from = h.pin + (size_t)cur * HC_SLOT;
        double *to = q.part->dst + q.first;
        if (q.part->f32)
            std::copy((const float *)from, (const float *)from + q.n, to);
        else
            std::memcpy(to, from, q.n * sizeof(double));
        cur = nxt;
    }
}

// memory the runtime does not know: pageable (what it does know, pinned by the
// caller for instance, it copies to directly)
bool pageable(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

bool ensure_slots(HostCopy &h)
{
    if (h.pin) return true;
    for (hipEvent_t &e : h.ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            (void)hipGetLastError();
            return false;
        }
    void *p = nullptr;
    if (hipHostMalloc(&p, 2 * HC_THREADS * HC_SLOT, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    h.pin = static_cast<char *>(p);
    return true;
}

}  // namespace

int host_copy(int device, hipStream_t stream, HostCopy &h, const HostPart *parts, int nparts, size_t whole)
{
    size_t bytes = 0;
    for (int k = 0; k < nparts; ++k) bytes += parts[k].n * elem(parts[k]);
    bool staged = bytes >= HC_STAGED;
    for (int k = 0; k < nparts && staged; ++k) staged = pageable(parts[k].dst);
    if (!staged) return copy_direct(stream, parts, nparts);
    std::unique_lock<std::mutex> one_at_a_time(h.use);
    if (!h.pin && h.direct + std::max(bytes, whole) < HC_FIRST) {
        h.direct += bytes;
        one_at_a_time.unlock();
        return copy_direct(stream, parts, nparts);
    }
    if (!ensure_slots(h)) return copy_direct(stream, parts, nparts);
    size_t total = 0;
    for (int k = 0; k < nparts; ++k) total += chunks_of(parts[k]);
    std::atomic<int> err{0};
    // a thread that cannot be started leaves its chunks to this one
    std::thread th[HC_THREADS];
    bool mine[HC_THREADS] = {true};
    for (int t = 1; t < HC_THREADS; ++t) {
        try {
            th[t] = std::thread([&, t] { copy_chunks(device, stream, h, parts, total, t, HC_THREADS, err); });
        } catch (const std::exception &) {
            mine[t] = true;
        }
    }
    for (int t = 0; t < HC_THREADS; ++t)
        if (mine[t]) copy_chunks(device, stream, h, parts, total, t, HC_THREADS, err);
    for (std::thread &t : th)
        if (t.joinable()) t.join();
    // nothing of this copy may still be under way when the slots are used again
    const hipError_t e = hipStreamSynchronize(stream);
    if (err.load() != 0) return hc_fail((hipError_t)err.load());
    return e == hipSuccess ? INMSOM_BT_OK : hc_fail(e);
}

void host_copy_release(HostCopy &h)
{
    if (h.pin) (void)hipHostFree(h.pin);
    h.pin = nullptr;
    for (hipEvent_t &e : h.ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

}  // namespace ibt
