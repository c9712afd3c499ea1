// Host <-> device copies of whole states through pinned chunks.
//
// A copy between the device and the caller's (pageable) array runs at 4-10 GB/s when the array's
// pages are new and 17 GB/s when they are not; the same bytes cross the bus to pinned memory at
// 56 GB/s.  A state therefore goes through a few pinned chunks kept with the context: the copy
// engine fills one while host threads empty the others (their page faults in parallel).  671 MB
// to a fresh array: 180 ms as one hipMemcpy (64 ms with huge pages), 26-32 ms (17 ms) this way.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>
#include "internal.h"

namespace rkdg {

namespace {

constexpr size_t ONE_SHOT = (size_t)3 << 19;  // up to 1.5 MiB one copy and one memcpy are faster than threads
constexpr size_t CHUNK = (size_t)8 << 20;     // 2 MiB chunks measured 2-3 times slower, larger ones no faster

// the pinned memory a transfer of n bytes wants; false: none to be had
bool reserve(Transfer& t, size_t n) {
    const size_t want = n <= ONE_SHOT ? ONE_SHOT : Transfer::CHUNKS * CHUNK;
    if (t.bytes >= want) return true;
    if (t.pin) (void)hipHostFree(t.pin);
    t.pin = nullptr;
    t.bytes = 0;
    if (hipHostMalloc(&t.pin, want, hipHostMallocDefault) != hipSuccess) {
        t.pin = nullptr;
        (void)hipGetLastError();
        return false;
    }
    t.bytes = want;
    return true;
}

// Chunks handed between the calling thread (which drives the copy engine) and the workers: a
// chunk is worked on by every worker (one slice each) once it is open, and closed when the last
// one is done.
struct Ring {
    std::mutex m;
    std::condition_variable opened, closed;
    long long open = 0;            // chunks 0 .. open - 1 may be worked on
    std::vector<int> left;         // workers yet to finish a chunk
    bool stop = false;

    Ring(long long n, int workers) : left((size_t)n, workers) {}
    bool wait_open(long long c) {
        std::unique_lock<std::mutex> l(m);
        opened.wait(l, [&] { return stop || open > c; });
        return !stop;
    }
    void done(long long c) {
        std::lock_guard<std::mutex> l(m);
        if (--left[(size_t)c] == 0) closed.notify_one();
    }
    void set_open(long long n) {
        { std::lock_guard<std::mutex> l(m); open = n; }
        opened.notify_all();
    }
    void wait_closed(long long c) {
        std::unique_lock<std::mutex> l(m);
        closed.wait(l, [&] { return left[(size_t)c] == 0; });
    }
    void abort() {
        { std::lock_guard<std::mutex> l(m); stop = true; }
        opened.notify_all();
    }
};

int copy_ring(Transfer& t, hipStream_t s, char* host, char* dev, size_t n, bool to_host) {
    const int B = Transfer::CHUNKS;
    const long long nch = (long long)((n + CHUNK - 1) / CHUNK);
    const int workers = std::max(1, std::min(8, host_threads()));
    Ring r(nch, workers);
    std::vector<hipEvent_t> ev(B, nullptr);
    hipError_t rc = hipSuccess;
    for (auto& e : ev)
        if (rc == hipSuccess) rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
    std::vector<std::thread> th;
    auto work = [&](int w) {
        for (long long c = 0; c < nch; ++c) {
            if (!r.wait_open(c)) return;
            const size_t o = (size_t)c * CHUNK, len = std::min(CHUNK, n - o);
            const size_t a = len * w / workers / 64 * 64, b = w == workers - 1 ? len : len * (w + 1) / workers / 64 * 64;
            char* p = t.pin + (size_t)(c % B) * CHUNK;
            if (to_host) std::memcpy(host + o + a, p + a, b - a);
            else std::memcpy(p + a, host + o + a, b - a);
            r.done(c);
        }
    };
    try {
        th.reserve(workers);
        for (int w = 0; w < workers; ++w) th.emplace_back(work, w);
    } catch (...) {  // no threads to be had: the caller copies without them
        r.abort();
        for (auto& x : th) x.join();
        for (auto e : ev) if (e) (void)hipEventDestroy(e);
        return -1;
    }
    auto move = [&](long long c) {
        const size_t o = (size_t)c * CHUNK, len = std::min(CHUNK, n - o);
        char* p = t.pin + (size_t)(c % B) * CHUNK;
        rc = to_host ? hipMemcpyAsync(p, dev + o, len, hipMemcpyDeviceToHost, s)
                     : hipMemcpyAsync(dev + o, p, len, hipMemcpyHostToDevice, s);
        if (rc == hipSuccess) rc = hipEventRecord(ev[c % B], s);
    };
    if (to_host) {
        long long issued = 0;
        for (long long c = 0; c < nch && rc == hipSuccess; ++c) {
            for (; issued < nch && issued < c + B && rc == hipSuccess; ++issued) {
                if (issued >= B) r.wait_closed(issued - B);
                move(issued);
            }
            if (rc == hipSuccess) rc = hipEventSynchronize(ev[c % B]);
            if (rc == hipSuccess) r.set_open(c + 1);
        }
    } else {
        r.set_open(std::min<long long>(B, nch));
        for (long long c = 0; c < nch && rc == hipSuccess; ++c) {
            r.wait_closed(c);
            move(c);
            // the next chunk of this buffer may be filled once its copy is through; the one
            // before it has had the longest time
            if (rc == hipSuccess && c >= 1 && c - 1 + B < nch) {
                rc = hipEventSynchronize(ev[(c - 1) % B]);
                if (rc == hipSuccess) r.set_open(c + B);
            }
        }
    }
    if (rc != hipSuccess) r.abort();
    for (auto& x : th) x.join();
    const hipError_t done = hipStreamSynchronize(s);  // nothing of the copy outlives the call
    if (rc == hipSuccess) rc = done;
    for (auto e : ev) if (e) (void)hipEventDestroy(e);
    return (int)rc;
}

int copy(Transfer& t, void* stream, char* host, char* dev, size_t n, bool to_host) {
    hipStream_t s = (hipStream_t)stream;
    hipError_t rc;
    if (n > 0 && reserve(t, n)) {
        if (n > ONE_SHOT) {
            const int e = copy_ring(t, s, host, dev, n, to_host);
            if (e >= 0) return e;
        } else {
            if (!to_host) std::memcpy(t.pin, host, n);
            rc = to_host ? hipMemcpyAsync(t.pin, dev, n, hipMemcpyDeviceToHost, s)
                         : hipMemcpyAsync(dev, t.pin, n, hipMemcpyHostToDevice, s);
            const hipError_t done = hipStreamSynchronize(s);
            if (rc == hipSuccess) rc = done;
            if (rc == hipSuccess && to_host) std::memcpy(host, t.pin, n);
            return (int)rc;
        }
    }
    rc = to_host ? hipMemcpyAsync(host, dev, n, hipMemcpyDeviceToHost, s)
                 : hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, s);
    const hipError_t done = hipStreamSynchronize(s);
    return (int)(rc == hipSuccess ? done : rc);
}

}  // namespace

int copy_to_host(Transfer& t, void* stream, void* host, const void* dev, size_t n) {
    return copy(t, stream, (char*)host, (char*)const_cast<void*>(dev), n, true);
}

int copy_to_device(Transfer& t, void* stream, void* dev, const void* host, size_t n) {
    return copy(t, stream, (char*)const_cast<void*>(host), (char*)dev, n, false);
}

void transfer_free(Transfer& t) {
    if (t.pin) (void)hipHostFree(t.pin);
    t.pin = nullptr;
    t.bytes = 0;
}

}  // namespace rkdg
