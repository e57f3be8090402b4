// Transfers of upf_stage.h on the host (hip/hip_runtime.h here stands in for the
// runtime): whole and ragged sizes, and with threads, pinned memory or events
// refused.  Prints the case that fails and ends with 1.
#include <cstdint>
#include <cstdio>
#include <new>
#include <vector>

#include "upf_stage.h"

static std::atomic<int> allocations_left{-1};  // below zero: no limit
void* operator new(size_t n) {
    if (allocations_left >= 0 && allocations_left.fetch_sub(1) <= 0) {
        allocations_left = 0;
        throw std::bad_alloc();
    }
    void* p = std::malloc(n);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static bool transfers(upf::Stage& stage, size_t a, size_t b, int allocations = -1) {
    std::vector<char> x(a), y(b), dev(a + b), x2(a), y2(b);
    for (size_t i = 0; i < a; ++i) x[i] = (char)(i * 7 + i / 251);
    for (size_t i = 0; i < b; ++i) y[i] = (char)(i * 11 + i / 253);
    const upf::StagePart up[2] = {{x.data(), 0, a}, {y.data(), a, b}}, down[2] = {{x2.data(), 0, a}, {y2.data(), a, b}};
    allocations_left = allocations;
    const bool ok = stage.to_device(dev.data(), a + b, up, 2, nullptr) && stage.to_host(dev.data(), a + b, down, 2, nullptr);
    std::atomic<long> sum{0};
    upf::Stage::split(1000, 10, [&](int, size_t beg, size_t end) { sum += (long)(end - beg); });
    allocations_left = -1;
    return ok && last_error == hipSuccess && sum == 1000 && x == x2 && y == y2;
}

int main() {
    const size_t sizes[][2] = {{1, 0}, {1000, 17}, {1u << 20, 1}, {3000001, 70001}, {9u << 20, 9u << 20}, {40000003, 5}};
    for (int mode = 0; mode < 4; ++mode) {
        upf::Stage stage;
        for (auto& s : sizes) {
            no_pinned = mode == 2;
            no_events = mode == 3;
            pinned_copies = plain_copies = 0;
            std::printf("mode %d, %zu + %zu bytes\n", mode, s[0], s[1]);
            std::fflush(stdout);
            if (!transfers(stage, s[0], s[1], mode == 1 ? 3 : -1)) return 1;  // 1: three threads start, no more
            if ((mode < 2 ? plain_copies : pinned_copies) != 0) return 1;
        }
        // what was refused is there again
        no_pinned = no_events = false;
        if (!transfers(stage, 5000000, 3)) return 1;
        if (pinned_copies == 0) return 1;
    }
    return 0;
}
