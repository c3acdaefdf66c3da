// How the tiled attention kernels hand their output rows to memory.
#pragma once

#include "common.hpp"

namespace esp {

// A wavefront's 32 output rows of RB bytes on their way through LDS: written by row (lane % 32), stored 1 KB of consecutive rows at a
// time. The 16-byte parts of a row are turned by its number, which spreads both sides over the banks.
template <int RB>
struct RowsOut {
  static constexpr int P = RB / 16, RPI = 64 / P;  // parts of a row; rows one store instruction takes
  static __device__ __forceinline__ char* at(char* ob, int r, int p) { return ob + r * RB + (p ^ (r & (P < 16 ? P - 1 : 15))) * 16; }
  // dst: where this lane's row (lane % 32) goes, 0 where there is none
  static __device__ __forceinline__ void store(char* ob, uint64_t dst, int lane) {
    using out16 = uint32_t __attribute__((ext_vector_type(4), aligned(8)));  // a row of O starts at any multiple of 8 bytes
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");  // the rows are written: one wavefront's LDS accesses keep their order
    const int lo = int(uint32_t(dst)), hi = int(uint32_t(dst >> 32));
    constexpr int N = 32 / RPI, B = N < 8 ? N : 8;
#pragma unroll
    for (int j0 = 0; j0 < N; j0 += B) {
      u32x4 v[B];
      uint64_t d[B];
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int r = (j0 + j) * RPI + lane / P;
        v[j] = *reinterpret_cast<const u32x4*>(at(ob, r, lane % P));
        d[j] = uint64_t(uint32_t(__shfl(lo, r))) | uint64_t(uint32_t(__shfl(hi, r))) << 32;
      }
#pragma unroll
      for (int j = 0; j < B; ++j)
        if (d[j]) *(__attribute__((address_space(1))) out16*)(d[j] + uint64_t(lane % P) * 16) = v[j];
    }
  }
  // The same where rows are `ld` bytes apart from dst on, the first n of them to be stored: an address and a stride instead of two lane exchanges
  // a store. With the rows' facts no longer reduced over the tile where nothing but their numbers counts: 122 fresh rows, 32 heads of 128,
  // 9.8 us -> 9.1; six prompts of 40 .. 900 rows 38.0 -> 36.3.
  static __device__ __forceinline__ void store_even(char* ob, void* dst, uint32_t ld, int n, int lane) {
    using out16 = uint32_t __attribute__((ext_vector_type(4), aligned(8)));
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
    constexpr int N = 32 / RPI;
    char* to = static_cast<char*>(dst);
    uint32_t off = uint32_t(lane / P) * ld + uint32_t(lane % P) * 16;
    const uint32_t step = uint32_t(RPI) * ld;
    u32x4 v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = *reinterpret_cast<const u32x4*>(at(ob, j * RPI + lane / P, lane % P));
#pragma unroll
    for (int j = 0; j < N; ++j, off += step)
      if (j * RPI + lane / P < n) *(__attribute__((address_space(1))) out16*)(to + off) = v[j];
  }
};

}  // namespace esp
