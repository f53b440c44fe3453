// Wave helpers and the LDS hash table of the graph kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace ckv {

__device__ inline int lane() { return (int)__lane_id(); }

__device__ inline double wave_sum_f64(double x) {
  for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

// Orders the wave's LDS accesses (all lanes' writes before, reads after).
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr uint32_t EMPTY = 0xffffffffu;  // a free slot

__device__ inline uint32_t hash_id(uint32_t x) { return (x * 0x9E3779B1u) >> 8; }

// Slots (a power of two, at most cap) for `most` ids: at least twice as many
// where cap allows.
__device__ inline uint32_t table_size(uint64_t most, uint32_t cap) {
  uint32_t size = 64;
  while (size < 2 * most && size < cap) size <<= 1;
  return size;
}

// Adds w to id u of an open-addressing LDS table (size slots, a power of two),
// counting new ids in *added (may be null); false when every slot holds another id.
__device__ inline bool insert(uint32_t* tk, double* ts, uint32_t size, uint32_t u, float w, int* added) {
  uint32_t h = hash_id(u) & (size - 1);
  for (uint32_t probe = 0; probe < size; ++probe) {
    const uint32_t cur = __hip_atomic_load(tk + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    bool mine = cur == u;
    if (cur == EMPTY) {
      const uint32_t prev = atomicCAS(tk + h, EMPTY, u);
      mine = prev == EMPTY || prev == u;
      if (prev == EMPTY && added) atomicAdd(added, 1);
    }
    if (mine) {
      unsafeAtomicAdd(ts + h, (double)w);
      return true;
    }
    h = (h + 1) & (size - 1);
  }
  return false;
}

// The same while *added, the new ids so far, is below `most`: false for a new
// id afterwards (threads that look at once may add one each past it).
__device__ inline bool insert_few(uint32_t* tk, double* ts, uint32_t size, uint32_t u, float w, int* added, int most) {
  uint32_t h = hash_id(u) & (size - 1);
  for (uint32_t probe = 0; probe < size; ++probe) {
    const uint32_t cur = __hip_atomic_load(tk + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    bool mine = cur == u;
    if (cur == EMPTY) {
      if (__hip_atomic_load(added, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >= most) return false;
      const uint32_t prev = atomicCAS(tk + h, EMPTY, u);
      mine = prev == EMPTY || prev == u;
      if (prev == EMPTY) atomicAdd(added, 1);
    }
    if (mine) {
      unsafeAtomicAdd(ts + h, (double)w);
      return true;
    }
    h = (h + 1) & (size - 1);
  }
  return false;
}

}  // namespace ckv
