// csrc/transfer.cpp against the CPU stand-in for HIP (stub_hip): every byte of transfers at the
// edges of the one-copy limit, the chunks and the ring, in one part and in four through one part's
// buffer, both ways; without pinned memory; with a copy that fails; and the pinned bytes held.
#include <cstdio>
#include <vector>
#include "internal.h"
#include <hip/hip_runtime.h>

namespace rkdg {
int host_threads() { return 5; }
}  // namespace rkdg
using namespace rkdg;

static unsigned char val(size_t i) { return (unsigned char)((i * 2654435761u) >> 13); }
static int bad = 0;
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); ++bad; } } while (0)

static void round_trip(size_t n, int parts, int want_ok) {
    StubStream st;
    Transfer t;
    std::vector<unsigned char> dev(n), state(n * parts), host(n * parts, 0);
    for (size_t i = 0; i < state.size(); ++i) state[i] = val(i);
    int next = 0;
    auto out = [&](int p) {
        CHECK(p == next++);
        st.push([&, p] { std::memcpy(dev.data(), state.data() + p * n, n); });
        return 0;
    };
    const int rc = copy_to_host(t, &st, host.data(), dev.data(), n, parts, out);
    CHECK((rc == 0) == (want_ok != 0));
    if (want_ok) { CHECK(next == parts); CHECK(host == state); }
    std::vector<unsigned char> back(n * parts, 0);
    next = 0;
    auto in = [&](int p) {
        CHECK(p == next++);
        st.push([&, p] { std::memcpy(back.data() + p * n, dev.data(), n); });
        return 0;
    };
    if (want_ok) {
        CHECK(copy_to_device(t, &st, dev.data(), host.data(), n, parts, in) == 0);
        st.wait();
        CHECK(next == parts);
        CHECK(back == state);
    }
    // what is held: the bytes themselves or the transfer's chunks, 32 MiB at most
    const size_t total = n * parts, chunk = (size_t)8 << 20, chunks = parts * ((n + chunk - 1) / chunk) * chunk;
    CHECK(stub_pinned <= (2 * total <= 3u << 20 ? total + 4095 : std::min((size_t)32 << 20, chunks)));
    transfer_free(t);
    CHECK(stub_pinned == 0);
}

int main() {
    const size_t M = 1 << 20, edges[] = {1, 4099, 3 * M / 2, 3 * M / 2 + 1, 8 * M - 1, 8 * M, 8 * M + 8, 32 * M, 32 * M + 1, 75 * M + 3};
    for (size_t n : edges)
        for (int parts : {1, 4}) {
            std::printf("%zu bytes in %d parts\n", n, parts);
            round_trip(n, parts, 1);
        }
    stub_pin_limit = 0;  // no pinned memory
    round_trip(5 * M, 4, 1);
    round_trip(1000, 1, 1);
    stub_pin_limit = (size_t)1 << 40;
    for (int f : {0, 3, 9}) {
        stub_fail_copy = f;
        round_trip(20 * M, 4, 0);
        stub_fail_copy = -1;
    }
    std::printf("%d failures\n", bad);
    return bad != 0;
}
