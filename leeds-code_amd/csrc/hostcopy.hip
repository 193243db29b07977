// Copies between a caller's arrays and the device through pinned chunks.
//
// The caller's arrays are pageable.  A plain copy of one pins its pages or
// moves them through the runtime's own staging with one thread, and a result
// array's pages are mapped by that thread as it first writes them, which
// bounds the copy at about 6-8 GB/s against the 55 GB/s of the link.  Here
// HC_THREADS threads (the caller's among them) each own two pinned chunks:
// while one chunk is on the link the other is copied to or from the caller's
// array, so the page mapping and the host copies of the threads run side by
// side with the transfers.  The chunks belong to one context or network and
// are freed with it.  Three components to the grid and back at L = M = 64,
// N = 64, 96 x 192 (69 MB), in new arrays: 4.2 -> 3.4 ms; one field to the grid
// in arrays that are kept (19 MB): 1.31 -> 0.82 ms.
#include <cstring>
#include <exception>
#include <thread>

#include "lsd_internal.h"

namespace lsd {

constexpr int HC_THREADS = 4;  // eight gain nothing: mapping the pages takes turns
constexpr size_t HC_CHUNK = size_t(1) << 20;
// From these sizes on the threads' start (about 50 us) is made up for, also for
// arrays that the caller keeps from call to call.  Results, 2.4 MB: 212 us
// directly, 189 through the chunks; new arrays 606 and 433.  Uploads find
// their pages mapped and gain later, analysis of one field and of three: 4.7 MB
// 253 us directly, 346 through the chunks; 18.9 MB 770 and 883 (new arrays
// 940, 920), 28.3 MB 1140-1380 and 1302 (1410, 1340), 56.6 MB 2595 and 2448:
// their callers say from where (HC_UPLOAD by default).
constexpr size_t HC_MIN = size_t(2) << 20;

bool HostStage::reserve() {
    if (buf) return true;
    for (hipEvent_t& e : ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) e = nullptr;
    for (const hipEvent_t& e : ev)
        if (!e) return false;
    if (hipHostMalloc((void**)&buf, 2 * HC_THREADS * HC_CHUNK, hipHostMallocDefault) != hipSuccess) buf = nullptr;
    return buf != nullptr;
}

void HostStage::release() {
    static_assert(sizeof(ev) / sizeof(ev[0]) == 2 * HC_THREADS, "two chunks a thread");
    if (buf) (void)hipHostFree(buf);
    buf = nullptr;
    for (hipEvent_t& e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

// Chunk q of the parts: host and device address and length.
struct HcChunk {
    char* host;
    char* dev;
    size_t n;
};
static HcChunk chunk_at(const HostPart* parts, int np, size_t q) {
    for (int k = 0; k < np; k++) {
        const size_t nq = (parts[k].bytes + HC_CHUNK - 1) / HC_CHUNK;
        if (q < nq) {
            const size_t at = q * HC_CHUNK;
            return {(char*)parts[k].host + at, (char*)parts[k].dev + at, std::min(HC_CHUNK, parts[k].bytes - at)};
        }
        q -= nq;
    }
    return {nullptr, nullptr, 0};
}

// The chunks t, t + HC_THREADS, ... of one thread.
static hipError_t copy_share(HostStage& st, int device, hipStream_t stream, const HostPart* parts, int np, size_t nq,
                             int t, bool to_host) {
    hipError_t e = hipSetDevice(device);
    if (e != hipSuccess) return e;
    HcChunk prev{nullptr, nullptr, 0};
    int slot = 2 * t;
    for (size_t q = t; q < nq; q += HC_THREADS, slot ^= 1) {
        const HcChunk c = chunk_at(parts, np, q);
        char* b = st.buf + slot * HC_CHUNK;
        if (to_host) {
            if ((e = hipMemcpyAsync(b, c.dev, c.n, hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
            if ((e = hipEventRecord(st.ev[slot], stream)) != hipSuccess) return e;
            if (prev.n) {
                if ((e = hipEventSynchronize(st.ev[slot ^ 1])) != hipSuccess) return e;
                memcpy(prev.host, st.buf + (slot ^ 1) * HC_CHUNK, prev.n);
            }
            prev = c;
        } else {
            // the chunk's last copy has left it (a new event counts as done)
            if ((e = hipEventSynchronize(st.ev[slot])) != hipSuccess) return e;
            memcpy(b, c.host, c.n);
            if ((e = hipMemcpyAsync(c.dev, b, c.n, hipMemcpyHostToDevice, stream)) != hipSuccess) return e;
            if ((e = hipEventRecord(st.ev[slot], stream)) != hipSuccess) return e;
        }
    }
    if (prev.n) {
        if ((e = hipEventSynchronize(st.ev[slot ^ 1])) != hipSuccess) return e;
        memcpy(prev.host, st.buf + (slot ^ 1) * HC_CHUNK, prev.n);
    }
    return hipSuccess;
}

// Memory the runtime does not know.  Pinned, managed or device memory in a
// caller's array goes straight to the link.
static bool pageable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

// Result arrays that share memory: the last part's data are to stay, so the
// parts go one after another.
static bool overlap(const HostPart* parts, int np) {
    for (int k = 0; k < np; k++)
        for (int q = 0; q < k; q++) {
            const uintptr_t a = (uintptr_t)parts[k].host, b = (uintptr_t)parts[q].host;
            if (a < b + parts[q].bytes && b < a + parts[k].bytes) return true;
        }
    return false;
}

// to_host: on return the host arrays hold the data.  Otherwise the copies are
// in the stream's order; they may still read the host arrays (pinned ones, of
// any size), and on an error copies either way may be under way.  The calling
// entry point waits for the stream before it returns (CopyGuard).
int host_copy(HostStage& st, hipStream_t stream, const HostPart* parts, int np, bool to_host, size_t upload_min) {
    size_t total = 0, nq = 0;
    for (int k = 0; k < np; k++) {
        if (!parts[k].host) {
            set_error("null host array");
            return LSD_E_HIP;
        }
        total += parts[k].bytes;
        nq += (parts[k].bytes + HC_CHUNK - 1) / HC_CHUNK;
    }
    bool chunks = total >= (to_host ? HC_MIN : upload_min);
    for (int k = 0; k < np && chunks; k++) chunks = pageable(parts[k].host);
    if (to_host && overlap(parts, np)) chunks = false;
    if (chunks && !st.reserve()) {
        // no pinned memory to be had: a plain copy needs none of it
        (void)hipGetLastError();
        chunks = false;
    }
    if (!chunks) {
        for (int k = 0; k < np; k++)
            LSD_HIP(hipMemcpyAsync(to_host ? parts[k].host : parts[k].dev, to_host ? parts[k].dev : parts[k].host,
                                   parts[k].bytes, to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, stream));
        if (to_host) LSD_HIP(hipStreamSynchronize(stream));
        return LSD_OK;
    }
    int device = 0;
    LSD_HIP(hipGetDevice(&device));
    hipError_t err[HC_THREADS];
    std::thread th[HC_THREADS];
    auto share = [&](int t) { err[t] = copy_share(st, device, stream, parts, np, nq, t, to_host); };
    for (int t = 1; t < HC_THREADS; t++) {
        try {
            th[t] = std::thread(share, t);
        } catch (const std::exception&) {
            // no thread to be had, or no memory for one: the caller's takes
            // the share below
        }
    }
    share(0);
    for (int t = 1; t < HC_THREADS; t++) {
        if (th[t].joinable()) th[t].join();
        else share(t);
    }
    for (int t = 0; t < HC_THREADS; t++) LSD_HIP(err[t]);
    return LSD_OK;
}

}  // namespace lsd
