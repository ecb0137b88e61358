// Shared device/host helpers of libnemo (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

namespace nemo {

typedef _Float16 half_t;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Largest number of requests one execution plan carries (ragged tables are
// passed by value as kernel arguments).
constexpr int kMaxBatch = 64;

// Prefix offsets of a ragged token layout: request b owns packed rows
// [start[b], start[b + 1]).
struct Ragged {
  int count;
  int start[kMaxBatch + 1];
};

__device__ __forceinline__ float h2f(uint16_t bits) { return (float)__builtin_bit_cast(half_t, bits); }
__device__ __forceinline__ uint16_t f2h(float v) { return __builtin_bit_cast(uint16_t, (half_t)v); }

// Request index owning packed row t (t < r.start[r.count], the same for the
// whole wave, every lane active): lane l compares the end of request l, one
// load instead of a chain of up to 64.
static_assert(kMaxBatch <= 64, "one lane per request");
__device__ __forceinline__ int ragged_find(const Ragged& r, int t) {
  const int l = (int)(threadIdx.x & 63);
  const bool past = l + 1 < r.count && t >= r.start[l + 1];
  return (int)__popcll(__builtin_amdgcn_ballot_w64(past));
}

// s_waitcnt immediate waiting for at most `n` outstanding vector memory
// operations (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt and lgkmcnt
// left at their maxima).
constexpr int vmcnt_imm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

// Lets `Kernel` be launched with up to `bytes` of dynamic LDS on the current
// device: one attribute call per kernel and device, from any thread. (The
// kernel is the template's argument, not its type: kernels of one signature
// have one type, and would share a flag.)
template <auto Kernel>
inline void allow_lds(int bytes) {
  static std::atomic<uint64_t> done{0};  // bit d: device d
  int device = 0;
  (void)hipGetDevice(&device);
  const uint64_t bit = 1ull << (device & 63);
  if (done.load(std::memory_order_acquire) & bit) return;
  (void)hipFuncSetAttribute((const void*)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  done.fetch_or(bit, std::memory_order_release);
}

}  // namespace nemo
