// The few HIP calls of csrc/transfer.cpp on the CPU: a stream is a thread that works off a queue,
// device memory is host memory, pinned memory is counted.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipHostMallocDefault = 0, hipEventDisableTiming = 2 };

struct StubStream {
    std::mutex m;
    std::condition_variable cv, idle;
    std::deque<std::function<void()>> q;
    bool busy = false, stop = false;
    std::thread t{[this] { run(); }};
    ~StubStream() {
        { std::lock_guard<std::mutex> l(m); stop = true; }
        cv.notify_all();
        t.join();
    }
    void run() {
        for (;;) {
            std::function<void()> f;
            {
                std::unique_lock<std::mutex> l(m);
                busy = false;
                idle.notify_all();
                cv.wait(l, [&] { return stop || !q.empty(); });
                if (q.empty()) return;
                f = std::move(q.front());
                q.pop_front();
                busy = true;
            }
            f();
        }
    }
    void push(std::function<void()> f) {
        { std::lock_guard<std::mutex> l(m); q.push_back(std::move(f)); }
        cv.notify_all();
    }
    void wait() {
        std::unique_lock<std::mutex> l(m);
        idle.wait(l, [&] { return q.empty() && !busy; });
    }
};
struct StubEvent {
    std::mutex m;
    std::condition_variable cv;
    int pending = 0;
};
typedef StubStream* hipStream_t;
typedef StubEvent* hipEvent_t;

inline std::atomic<size_t> stub_pinned{0}, stub_pin_limit{(size_t)1 << 40};
inline std::atomic<int> stub_fail_copy{-1};  // the copy that fails

template <typename T>
hipError_t hipHostMalloc(T** p, size_t n, int) {
    if (stub_pinned + n > stub_pin_limit) return hipErrorOutOfMemory;
    size_t* b = (size_t*)std::malloc(n + 64);
    *b = n;
    stub_pinned += n;
    *p = (T*)((char*)b + 64);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    size_t* b = (size_t*)((char*)p - 64);
    stub_pinned -= *b;
    std::free(b);
    return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = new StubEvent; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    { std::lock_guard<std::mutex> l(e->m); ++e->pending; }
    s->push([e] {
        std::lock_guard<std::mutex> l(e->m);
        --e->pending;
        e->cv.notify_all();
    });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    std::unique_lock<std::mutex> l(e->m);
    e->cv.wait(l, [&] { return e->pending == 0; });
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) { s->wait(); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t st) {
    if (stub_fail_copy >= 0 && stub_fail_copy-- == 0) return hipErrorInvalidValue;
    st->push([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
