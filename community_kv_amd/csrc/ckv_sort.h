// Stable radix sort of (uint32 key, uint32 value) pairs for the graph kernels.
#pragma once

#include <string.h>

#include <hip/hip_runtime.h>
#include <rocprim/rocprim.hpp>

#include <stddef.h>
#include <stdint.h>

namespace ckv {

// rocPRIM sorts up to MergeSortLimit items by merging (two launches per
// doubling of the sorted runs) and more by one-sweep radix passes.  Its limit
// of 1,048,576 items costs the graphs of short prompts dozens of launches
// (62 for the half million edge entries of a 2,000-token layer): above 16,384
// items the three passes of a 19-bit key are fewer launches and less traffic.
constexpr size_t SORT_MERGE_LIMIT = 16384;
using PairSortConfig = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                                  rocprim::default_config, SORT_MERGE_LIMIT>;

inline size_t sort_pairs_bytes(size_t n) {
  size_t bytes = 0;
  if (n > 0)
    (void)rocprim::radix_sort_pairs<PairSortConfig>(nullptr, bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr,
                                                    (const uint32_t*)nullptr, (uint32_t*)nullptr, n, 0, 32,
                                                    (hipStream_t)0);
  return bytes;
}

inline hipError_t sort_pairs(void* temp, size_t temp_bytes, const uint32_t* keys_in, uint32_t* keys_out,
                             const uint32_t* values_in, uint32_t* values_out, size_t n, int bits, hipStream_t st) {
  return rocprim::radix_sort_pairs<PairSortConfig>(temp, temp_bytes, keys_in, keys_out, values_in, values_out, n, 0,
                                                   (unsigned)bits, st);
}

inline size_t scan_bytes(size_t n) {
  size_t bytes = 0;
  (void)rocprim::exclusive_scan(nullptr, bytes, (const int32_t*)nullptr, (int32_t*)nullptr, (int32_t)0, n,
                                rocprim::plus<int32_t>(), (hipStream_t)0);
  return bytes;
}

inline hipError_t exclusive_scan_i32(void* temp, size_t temp_bytes, const int32_t* in, int32_t* out, size_t n,
                                     hipStream_t st) {
  return rocprim::exclusive_scan(temp, temp_bytes, in, out, (int32_t)0, n, rocprim::plus<int32_t>(), st);
}

// Bits needed to hold the values 0..x.
inline int bits_for(uint64_t x) {
  int b = 1;
  while (b < 63 && (x >> b) != 0) ++b;
  return b;
}
inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace ckv
