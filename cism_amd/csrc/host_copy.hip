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
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

#include "cismgpu_internal.h"

namespace {

constexpr size_t HC_CHUNK = 2 << 20;
constexpr size_t HC_MIN = 6 << 20;
constexpr int HC_THREADS = 4;

struct HostSeg { void* host; const void* dev; size_t n; };   // dev is written to on the way up

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
// s; returns when they are complete.
int host_copy(HostPipe& P, hipStream_t s, const std::vector<HostSeg>& segs, bool down = true) {
    size_t total = 0;
    for (const HostSeg& g : segs) total += g.n;
    if (total < HC_MIN) {
        for (const HostSeg& g : segs)
            CG_CHECK(down ? hipMemcpyAsync(g.host, g.dev, g.n, hipMemcpyDeviceToHost, s)
                          : hipMemcpyAsync((void*)g.dev, g.host, g.n, hipMemcpyHostToDevice, s));
        CG_CHECK(hipStreamSynchronize(s));
        return CISMGPU_OK;
    }
    const int st = P.open();
    if (st) return st;
    struct Chunk { char* host; char* dev; size_t n; };
    std::vector<Chunk> chunks;
    for (const HostSeg& g : segs)
        for (size_t o = 0; o < g.n; o += HC_CHUNK)
            chunks.push_back({(char*)g.host + o, (char*)g.dev + o, std::min(HC_CHUNK, g.n - o)});
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
            const Chunk& k = chunks[c];
            return keep(down ? hipMemcpyAsync(slot[b], k.dev, k.n, hipMemcpyDeviceToHost, s)
                             : hipMemcpyAsync(k.dev, slot[b], k.n, hipMemcpyHostToDevice, s)) &&
                   keep(hipEventRecord(ev[b], s));
        };
        const size_t n = chunks.size();
        int b = 0;
        if (!down) {
            for (size_t c = t, m = 0; c < n; c += HC_THREADS, b ^= 1, ++m) {
                if (m >= 2 && !keep(hipEventSynchronize(ev[b]))) return;
                memcpy(slot[b], chunks[c].host, chunks[c].n);
                if (!link(c, b)) return;
            }
            return;
        }
        if ((size_t)t < n && !link(t, 0)) return;
        for (size_t c = t; c < n; c += HC_THREADS, b ^= 1) {
            if (c + HC_THREADS < n && !link(c + HC_THREADS, b ^ 1)) return;
            if (!keep(hipEventSynchronize(ev[b]))) return;
            memcpy(chunks[c].host, slot[b], chunks[c].n);
        }
    };
    std::thread th[HC_THREADS];
    bool started[HC_THREADS] = {};
    for (int t = 1; t < HC_THREADS; ++t) {
        try {
            th[t] = std::thread(work, t);
            started[t] = true;
        } catch (const std::system_error&) {      // no thread: its share is done below
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
