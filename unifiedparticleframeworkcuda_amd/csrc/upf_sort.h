// upf_sort.h -- device radix sort entry points.
#ifndef UPF_SORT_H_
#define UPF_SORT_H_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace upf {

// Smallest tiles of the multi-block passes: 512 threads x 4 keys.
constexpr int RS_THREADS = 512;
constexpr int RS_IPT_MIN = 4;
constexpr int RS_MAX_DIGITS = 1024;  // 10-bit digits

// Working memory of a sort of n keys: digit counts of every tile, digit
// totals, one ping-pong buffer of keys and values.
constexpr size_t radix_sort_temp_bytes(int n) {
    const size_t tile = (size_t)RS_THREADS * RS_IPT_MIN;
    const size_t ntiles = ((size_t)n + tile - 1) / tile;
    return (RS_MAX_DIGITS * (ntiles + 1) + 2 * (size_t)n) * sizeof(uint32_t);
}

hipError_t radix_sort(const uint32_t* keys, const uint32_t* vals, uint32_t* keys_out, uint32_t* vals_out, int n,
                      int bits, void* temp, hipStream_t st);

}  // namespace upf

#endif
