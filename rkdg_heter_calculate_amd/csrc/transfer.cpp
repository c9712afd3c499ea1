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
#include <functional>
#include <mutex>
#include <thread>
#include <vector>
#include "internal.h"

namespace rkdg {

namespace {

constexpr size_t ONE_SHOT = (size_t)3 << 19;  // up to 1.5 MiB one copy and one memcpy are faster than threads
constexpr size_t CHUNK = (size_t)8 << 20;     // 2 MiB chunks measured 2-3 times slower, larger ones no faster
constexpr long long chunks_of(size_t n) { return (long long)((n + CHUNK - 1) / CHUNK); }

// the pinned memory a transfer of n bytes in nch chunks wants, no more than it can use (it is kept:
// many small contexts hold little); false: none to be had
bool reserve(Transfer& t, size_t n, long long nch) {
    const size_t want = n <= ONE_SHOT ? (n + 4095) / 4096 * 4096 : (size_t)std::min<long long>(Transfer::CHUNKS, nch) * CHUNK;
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

// A transfer: parts of n bytes each, one after the other on the host, all through the same device
// buffer; form puts a part into it (on the way to the host) or takes it out.
struct Parts {
    char* host;
    char* dev;
    size_t n;
    int parts;
    const std::function<int(int)>& form;
    bool to_host;
};

int copy_ring(Transfer& t, hipStream_t s, const Parts& x) {
    const int B = Transfer::CHUNKS;
    const bool to_host = x.to_host;
    const long long per = chunks_of(x.n), nch = x.parts * per;  // chunks of a part, of all
    auto chunk = [&](long long c, size_t& hoff, size_t& doff) {
        doff = (size_t)(c % per) * CHUNK;
        hoff = (size_t)(c / per) * x.n + doff;
        return std::min(CHUNK, x.n - doff);
    };
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
            size_t o, d;
            const size_t len = chunk(c, o, d);
            const size_t a = len * w / workers / 64 * 64, b = w == workers - 1 ? len : len * (w + 1) / workers / 64 * 64;
            char* p = t.pin + (size_t)(c % B) * CHUNK;
            if (to_host) std::memcpy(x.host + o + a, p + a, b - a);
            else std::memcpy(p + a, x.host + o + a, b - a);
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
        size_t o, d;
        const size_t len = chunk(c, o, d);
        char* p = t.pin + (size_t)(c % B) * CHUNK;
        // (in stream order: a part is formed after the copies of the one before it, and taken
        // out before the copies of the next)
        if (to_host && c % per == 0) rc = (hipError_t)x.form((int)(c / per));
        if (rc == hipSuccess)
            rc = to_host ? hipMemcpyAsync(p, x.dev + d, len, hipMemcpyDeviceToHost, s)
                         : hipMemcpyAsync(x.dev + d, p, len, hipMemcpyHostToDevice, s);
        if (rc == hipSuccess) rc = hipEventRecord(ev[c % B], s);
        if (rc == hipSuccess && !to_host && c % per == per - 1) rc = (hipError_t)x.form((int)(c / per));
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

int copy(Transfer& t, void* stream, const Parts& x) {
    hipStream_t s = (hipStream_t)stream;
    const size_t total = x.n * x.parts;
    char* pin = nullptr;
    if (total > 0 && reserve(t, total, x.parts * chunks_of(x.n))) {
        if (total > ONE_SHOT) {
            const int e = copy_ring(t, s, x);
            if (e >= 0) return e;
        } else {
            pin = t.pin;
        }
    }
    // part by part, through pinned memory if there is some
    char* const host = pin ? pin : x.host;
    hipError_t rc = hipSuccess;
    if (pin && !x.to_host) std::memcpy(pin, x.host, total);
    for (int p = 0; p < x.parts && rc == hipSuccess; ++p) {
        if (x.to_host) rc = (hipError_t)x.form(p);
        if (rc == hipSuccess)
            rc = x.to_host ? hipMemcpyAsync(host + p * x.n, x.dev, x.n, hipMemcpyDeviceToHost, s)
                           : hipMemcpyAsync(x.dev, host + p * x.n, x.n, hipMemcpyHostToDevice, s);
        if (rc == hipSuccess && !x.to_host) rc = (hipError_t)x.form(p);
    }
    const hipError_t done = hipStreamSynchronize(s);
    if (rc == hipSuccess) rc = done;
    if (rc == hipSuccess && pin && x.to_host) std::memcpy(x.host, pin, total);
    return (int)rc;
}

}  // namespace

int copy_to_host(Transfer& t, void* stream, void* host, const void* dev, size_t n, int parts,
                 const std::function<int(int)>& form) {
    return copy(t, stream, Parts{(char*)host, (char*)const_cast<void*>(dev), n, parts, form, true});
}

int copy_to_device(Transfer& t, void* stream, void* dev, const void* host, size_t n, int parts,
                   const std::function<int(int)>& use) {
    return copy(t, stream, Parts{(char*)const_cast<void*>(host), (char*)dev, n, parts, use, false});
}

void transfer_free(Transfer& t) {
    if (t.pin) (void)hipHostFree(t.pin);
    t.pin = nullptr;
    t.bytes = 0;
}

}  // namespace rkdg
