// upf_stage.h -- large transfers between a caller's ordinary memory and the device.
//
// A copy to or from pageable memory runs at the speed of one host thread: the
// runtime's staging copy, and a page fault per page of a buffer that the
// caller has just allocated (81 MB of state: 23 ms, most of it this).  Here
// several threads move one contiguous device range in slices, each through a
// pinned slice of its own, so that host copies, page faults and DMA overlap.
#ifndef UPF_STAGE_H_
#define UPF_STAGE_H_

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <thread>

namespace upf {

// One caller array of a transfer: bytes host[0 .. bytes) at device offset off.
struct StagePart {
    char* host;
    size_t off, bytes;
};

class Stage {
  public:
    // largest: bytes of the largest transfer to come, which sizes the pinned
    // memory (its first use allocates it, at most THREADS slices)
    explicit Stage(size_t largest = 0) : largest_(largest) {}
    Stage(const Stage&) = delete;
    Stage& operator=(const Stage&) = delete;
    void expect(size_t largest) { largest_ = largest; }

    static constexpr size_t SLICE = 1u << 20;  // 1 MiB: about 20 us of DMA (512 KiB: 5 % slower)
    static constexpr int THREADS = 8;
    static constexpr size_t PER_THREAD = 2u << 20;  // a further thread's start pays from here on

    ~Stage() {
        for (auto& e : ev_)
            if (e) (void)hipEventDestroy(e);
        if (pin_) (void)hipHostFree(pin_);
    }
    // device range -> the parts / the parts -> device range (total bytes, the
    // parts in ascending order of off); returns when the transfer is complete
    bool to_host(const char* dev, size_t total, const StagePart* parts, int n, hipStream_t st) {
        return run<false>(const_cast<char*>(dev), total, parts, n, st);
    }
    bool to_device(char* dev, size_t total, const StagePart* parts, int n, hipStream_t st) {
        return run<true>(dev, total, parts, n, st);
    }
    // f(k, begin, end) over [0, n) in up to THREADS contiguous pieces k of at least `grain`
    template <class F>
    static void split(size_t n, size_t grain, F f) {
        const int t = (int)std::min<size_t>(THREADS, std::max<size_t>(1, n / grain));
        std::atomic<int> next{0};
        parallel(t, [&](int) {
            for (int k; (k = next.fetch_add(1)) < t;) f(k, n * k / t, n * (k + 1) / t);
        });
    }

  private:
    size_t largest_;
    char* pin_ = nullptr;
    size_t cap_ = 0;  // bytes of pin_
    hipEvent_t ev_[THREADS] = {};

    // work(k) on the caller (k = 0) and on up to t - 1 further threads; work
    // must take its items from a shared counter, since fewer threads may start
    template <class F>
    static void parallel(int t, F work) {
        std::thread pool[THREADS];
        int started = 1;
        try {
            for (; started < t; ++started) pool[started] = std::thread(work, started);
        } catch (...) {  // no thread, or no memory for one
        }
        work(0);
        for (int k = 1; k < started; ++k) pool[k].join();
    }

    static int threads(size_t total) {
        return (int)std::min<size_t>(THREADS, (total + PER_THREAD - 1) / PER_THREAD);
    }
    bool reserve(size_t total) {
        total = std::max(total, largest_);
        const int t = threads(total);
        // any thread may take any chunk: whole slices, unless there is one chunk
        const size_t bytes = total <= SLICE ? total : (size_t)t * SLICE;
        for (int k = 0; k < t; ++k)
            if (!ev_[k] && hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming) != hipSuccess) return false;
        if (bytes <= cap_) return true;
        if (pin_) (void)hipHostFree(pin_);
        pin_ = nullptr;
        cap_ = 0;
        if (hipHostMalloc((void**)&pin_, bytes, hipHostMallocDefault) != hipSuccess) return false;
        cap_ = bytes;
        return true;
    }

    // without pinned memory
    template <bool UP>
    static bool copy_parts(char* dev, const StagePart* parts, int n, hipStream_t st) {
        bool ok = true;
        for (int p = 0; p < n && ok; ++p) {
            char *d = dev + parts[p].off, *h = parts[p].host;
            if (parts[p].bytes)
                ok = hipMemcpyAsync(UP ? d : h, UP ? h : d, parts[p].bytes,
                                    UP ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st) == hipSuccess;
        }
        return hipStreamSynchronize(st) == hipSuccess && ok;
    }

    template <bool UP>
    bool run(char* dev, size_t total, const StagePart* parts, int n, hipStream_t st) {
        if (total == 0) return hipStreamSynchronize(st) == hipSuccess;
        const size_t chunks = (total + SLICE - 1) / SLICE;
        const int t = threads(total);
        int device = 0;
        if (!reserve(total)) {
            (void)hipGetLastError();  // else a launch's check would find it
            return copy_parts<UP>(dev, parts, n, st);
        }
        if (hipGetDevice(&device) != hipSuccess) return false;
        std::atomic<size_t> next{0};
        std::atomic<bool> ok{true};
        parallel(t, [&](int k) {
            if (k && hipSetDevice(device) != hipSuccess) ok = false;
            char* slice = pin_ + (size_t)k * SLICE;
            bool busy = false;
            for (size_t c; ok && (c = next.fetch_add(1)) < chunks;) {
                const size_t beg = c * SLICE, end = std::min(beg + SLICE, total);
                // the transfer that used the slice last
                if (busy && hipEventSynchronize(ev_[k]) != hipSuccess) ok = false;
                auto copy = [&] {
                    for (int p = 0; p < n; ++p) {
                        const size_t b = std::max(beg, parts[p].off), e = std::min(end, parts[p].off + parts[p].bytes);
                        if (b >= e) continue;
                        char* h = parts[p].host + (b - parts[p].off);
                        if (UP) std::memcpy(slice + (b - beg), h, e - b);
                        else std::memcpy(h, slice + (b - beg), e - b);
                    }
                };
                if (UP) copy();
                if (hipMemcpyAsync(UP ? dev + beg : slice, UP ? slice : dev + beg, end - beg,
                                   UP ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, st) != hipSuccess ||
                    hipEventRecord(ev_[k], st) != hipSuccess)
                    ok = false;
                busy = UP;
                if (!UP) {
                    if (hipEventSynchronize(ev_[k]) != hipSuccess) ok = false;
                    if (ok) copy();
                }
            }
        });
        return hipStreamSynchronize(st) == hipSuccess && ok;
    }
};

}  // namespace upf

#endif
