// host_copy.hip -- large copies between device memory and a caller's pageable
// host memory.
//
// The runtime moves them through one bounce buffer with one host thread, which
// on the way down also takes the page faults of a fresh destination: about
// 10 GB/s, a fifth of the link, and 28 GB/s on the way up.  Here HC_THREADS
// threads each own two pinned slots and take every HC_THREADS-th chunk, one
// slot on the link while the other is copied on the host.  Below HC_MIN bytes
// the threads cost more than they save and the runtime's copy is used.
// 185 MB of velocities: down 18.7 -> 5.7 ms (33 GB/s), up 6.6 -> 4.9 ms; 9.6
// and 8.9 ms with 512 KiB chunks and eight threads, which wait on the runtime's
// locks; 4 MiB or eight threads of 2 MiB gain nothing.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "cismgpu_internal.h"

namespace {

constexpr size_t HC_CHUNK = 2 << 20;
constexpr size_t HC_MIN = 6 << 20;
constexpr int HC_THREADS = 4;

struct HostSeg { void* host; void* dev; size_t n; };

// The pinned slots of one system (16 MiB), made by its first large copy.
struct HostPipe {
    char* mem = nullptr;
    hipEvent_t ev[2 * HC_THREADS] = {};

    int open() {
        if (mem) return CISMGPU_OK;
        for (auto& e : ev)
            if (!e) CG_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        CG_CHECK(hipHostMalloc(&mem, 2 * HC_THREADS * HC_CHUNK, hipHostMallocDefault));
        return CISMGPU_OK;
    }
    void close() {
        if (mem) hipHostFree(mem);
        for (auto& e : ev)
            if (e) hipEventDestroy(e);
        mem = nullptr;
    }
};

// Copies the segments down to host memory (or up from it), ordered on stream
// s; returns when they are complete.  Takes no memory from the heap, and does
// with the runtime's copy where there is no pinned memory and with fewer
// threads where one cannot be started, so it fails only if a copy does.
int host_copy(HostPipe& P, hipStream_t s, const HostSeg* segs, int nseg, bool down = true) {
    size_t total = 0, nchunk = 0;
    for (int g = 0; g < nseg; ++g) {
        total += segs[g].n;
        nchunk += (segs[g].n + HC_CHUNK - 1) / HC_CHUNK;
    }
    if (total < HC_MIN || P.open() != CISMGPU_OK) {
        (void)hipGetLastError();                  // the copy below is what counts
        for (int g = 0; g < nseg; ++g)
            CG_CHECK(down ? hipMemcpyAsync(segs[g].host, segs[g].dev, segs[g].n, hipMemcpyDeviceToHost, s)
                          : hipMemcpyAsync(segs[g].dev, segs[g].host, segs[g].n, hipMemcpyHostToDevice, s));
        CG_CHECK(hipStreamSynchronize(s));
        return CISMGPU_OK;
    }
    struct Chunk { char* host; char* dev; size_t n; };
    auto chunk = [&](size_t c) {                  // the c-th of all segments
        int g = 0;
        for (size_t m; c >= (m = (segs[g].n + HC_CHUNK - 1) / HC_CHUNK); ++g) c -= m;
        const size_t o = c * HC_CHUNK;
        return Chunk{(char*)segs[g].host + o, (char*)segs[g].dev + o, std::min(HC_CHUNK, segs[g].n - o)};
    };
    int dev = 0;
    CG_CHECK(hipGetDevice(&dev));
    std::atomic<int> err{hipSuccess};
    auto keep = [&](hipError_t e) {
        int ok = hipSuccess;
        if (e != hipSuccess) err.compare_exchange_strong(ok, (int)e);
        return e == hipSuccess;
    };
    auto work = [&](int t) {
        if (!keep(hipSetDevice(dev))) return;
        char* slot[2] = {P.mem + (2 * t) * HC_CHUNK, P.mem + (2 * t + 1) * HC_CHUNK};
        hipEvent_t* ev = P.ev + 2 * t;
        // the link's part of this thread's c-th chunk
        auto link = [&](size_t c, int b) {
            const Chunk k = chunk(c);
            return keep(down ? hipMemcpyAsync(slot[b], k.dev, k.n, hipMemcpyDeviceToHost, s)
                             : hipMemcpyAsync(k.dev, slot[b], k.n, hipMemcpyHostToDevice, s)) &&
                   keep(hipEventRecord(ev[b], s));
        };
        const size_t n = nchunk;
        int b = 0;
        if (!down) {
            for (size_t c = t, m = 0; c < n; c += HC_THREADS, b ^= 1, ++m) {
                if (m >= 2 && !keep(hipEventSynchronize(ev[b]))) return;
                const Chunk k = chunk(c);
                memcpy(slot[b], k.host, k.n);
                if (!link(c, b)) return;
            }
            return;
        }
        if ((size_t)t < n && !link(t, 0)) return;
        for (size_t c = t; c < n; c += HC_THREADS, b ^= 1) {
            if (c + HC_THREADS < n && !link(c + HC_THREADS, b ^ 1)) return;
            if (!keep(hipEventSynchronize(ev[b]))) return;
            const Chunk k = chunk(c);
            memcpy(k.host, slot[b], k.n);
        }
    };
    std::thread th[HC_THREADS];
    bool started[HC_THREADS] = {};
    for (int t = 1; t < HC_THREADS; ++t) {
        try {
            th[t] = std::thread(work, t);
            started[t] = true;
        } catch (...) {                           // no thread, or no memory for one: its share is done below
        }
    }
    work(0);
    for (int t = 1; t < HC_THREADS; ++t) {
        if (started[t]) th[t].join();
        else work(t);
    }
    CG_CHECK(hipStreamSynchronize(s));            // the slots are free again
    if (err.load() != hipSuccess) {
        cismgpu_set_error("host copy: %s", hipGetErrorString((hipError_t)err.load()));
        return CISMGPU_ERR_HIP;
    }
    return CISMGPU_OK;
}

}  // namespace
