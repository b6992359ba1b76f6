// Device helpers shared by the sparse-product kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace nmg {

constexpr int kXcd = 8;  // accelerator complex dies (XCDs) of an MI355X

// Kernel flags of the sparse products: bit 0 XCD-contiguous workgroup order,
// bit 1 non-temporal (streaming) loads of the matrix values and indices.
// Workgroup b of a launch runs on XCD b % 8 (round-robin dispatch).  With
// bit 0 set the logical block index gives each XCD one contiguous range,
// so neighbouring node rows -- which gather the same x entries -- share one
// XCD's L2 instead of being spread over eight.  A bijection of [0, grid).
__device__ __forceinline__ int64_t xcd_block(int flags) {
  const int64_t b = blockIdx.x;
  if (!(flags & 1)) return b;
  const int64_t n = gridDim.x, q = n / kXcd, r = n % kXcd;
  const int64_t x = b % kXcd, i = b / kXcd;
  return x < r ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}
// position of value q of BSR3 entry k (planes, or tiles of 64 entries)
__device__ __forceinline__ int64_t bidx(int64_t k, int q, int64_t nbnz, int flags) {
  return (flags & 4) ? ((k >> 6) * 576 + (int64_t)q * 64 + (k & 63)) : ((int64_t)q * nbnz + k);
}

// lane permutation by DPP: within groups of four (quad_perm), or mirrored in
// rows of 8 (0x141) or 16 (0x140) lanes
template <int CTRL>
__device__ __forceinline__ int quad(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double quad(double v) {
  const int lo = quad<CTRL>((int)__double2loint(v)), hi = quad<CTRL>((int)__double2hiint(v));
  return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ __forceinline__ float quad(float v) {
  return __int_as_float(quad<CTRL>(__float_as_int(v)));
}

}  // namespace nmg
