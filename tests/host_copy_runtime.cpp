// A HIP runtime on the CPU for the host copies of leeds-code_amd/csrc/hostcopy.hip:
// copies from and to pinned memory are queued and run when their stream or a
// later event of it is waited for (as late as the runtime may), copies of
// pageable memory run at once, after all that is queued.  One stream.
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <new>
#include <thread>

#include "../leeds-code_amd/csrc/lsd_internal.h"

namespace {
struct Op {
    void* dst;
    const void* src;
    size_t n;
    hipEvent_t ev;  // a record, if set
};
std::mutex mu;
std::deque<Op> queue;
std::map<const char*, size_t> pinned;
std::thread::id caller;
thread_local bool in_runtime = false;
struct Lock {
    std::lock_guard<std::mutex> g{mu};
    Lock() { in_runtime = true; }
    ~Lock() { in_runtime = false; }
};
int caller_delay_ms = 0, copies_ok = -1, threads_fail = 0, no_pinned = 0;

bool is_pinned(const void* p) {
    auto it = pinned.upper_bound((const char*)p);
    if (it == pinned.begin()) return false;
    --it;
    return (const char*)p < it->first + it->second;
}
void run_until(hipEvent_t ev) {
    bool have = !ev;
    for (const Op& o : queue) have = have || o.ev == ev;
    while (have && !queue.empty()) {
        const Op o = queue.front();
        queue.pop_front();
        if (o.n) memmove(o.dst, o.src, o.n);
        if (ev && o.ev == ev) return;
    }
}
}  // namespace

extern "C" {
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
    Lock lock;
    if (copies_ok == 0) return hipErrorInvalidValue;
    if (copies_ok > 0) copies_ok--;
    queue.push_back({dst, src, n, nullptr});
    if (!is_pinned(kind == hipMemcpyHostToDevice ? src : dst)) run_until(nullptr);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    Lock lock;
    run_until(nullptr);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = (hipEvent_t)malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    free((void*)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    Lock lock;
    for (Op& o : queue)
        if (o.ev == e) o.ev = nullptr;
    queue.push_back({nullptr, nullptr, 0, e});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (caller_delay_ms && std::this_thread::get_id() == caller)
        std::this_thread::sleep_for(std::chrono::milliseconds(caller_delay_ms));
    Lock lock;
    run_until(e);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (no_pinned) return hipErrorOutOfMemory;
    *p = malloc(n);
    Lock lock;
    pinned[(const char*)*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    Lock lock;
    run_until(nullptr);  // as the runtime waits for the device
    pinned.erase((const char*)p);
    free(p);
    return hipSuccess;
}
#undef hipPointerGetAttributes
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    Lock lock;
    memset(a, 0, sizeof *a);
    a->type = is_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

// a thread's state is allocated by the thread that starts it
void* operator new(size_t n) {
    if (threads_fail && !in_runtime && std::this_thread::get_id() == caller) throw std::bad_alloc();
    if (void* p = malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

namespace lsd {
void set_error(const std::string&) {}
}  // namespace lsd

extern "C" {
// One host_copy of np parts.  pin: the host arrays are pinned.  delay_ms:
// the calling thread waits that long at every event.  ok: hipMemcpyAsync
// fails after so many calls (-1: never).  oom: no memory for threads.  nopin:
// no pinned memory.
int fake_host_copy(int np, void** host, void** dev, const size_t* bytes, int to_host, int pin, int delay_ms, int ok,
                   int oom, int nopin) {
    lsd::HostStage st;
    lsd::HostPart parts[8];
    caller = std::this_thread::get_id();
    caller_delay_ms = delay_ms;
    copies_ok = ok;
    for (int k = 0; k < np; k++) {
        parts[k] = {host[k], dev[k], bytes[k]};
        if (pin) pinned[(const char*)host[k]] = bytes[k];
    }
    threads_fail = oom;
    no_pinned = nopin;
    int rc;
    try {
        rc = lsd::host_copy(st, nullptr, parts, np, to_host != 0);
    } catch (const std::exception&) {
        rc = -99;  // through a C entry point this would end the program
    }
    threads_fail = no_pinned = 0;
    copies_ok = -1;
    caller_delay_ms = 0;
    st.release();
    if (pin)
        for (int k = 0; k < np; k++) pinned.erase((const char*)host[k]);
    return rc;
}
// copies still queued
int fake_pending() { return (int)queue.size(); }
void fake_run() { (void)hipStreamSynchronize(nullptr); }
}
