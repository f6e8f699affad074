// s2dw_dev.h -- helpers shared by the device sources of the contractions.
#pragma once

#include <hip/hip_runtime.h>

namespace s2dw {

constexpr int kMaxSc = 32;
constexpr int kMaxCol = 32;
constexpr int kChunk = 8;  // columns per contraction launch
// Buffer descriptor word 3 for raw (untyped) loads on gfx9-family GPUs, and
// an offset past the end of any buffer used with it: range-checked buffer
// loads at that offset return 0, so a kernel can issue a load for every
// lane unconditionally (buffers used this way stay below 2^31 bytes).
constexpr int kBufWord3 = 0x00020000;
constexpr unsigned kBufOut = 0x80000000u;
constexpr long long kBufMaxBytes = 0x7fffffffLL;

__host__ __device__ __forceinline__ long long tri0(long long l) { return l * (l + 1) / 2; }

// Read-only tables indexed by wave-uniform values are read through the
// constant address space so that the loads become scalar (s_load) and the
// values feed v_fma_f64 as SGPR operands.
typedef const double __attribute__((address_space(4))) *cdptr;
__device__ __forceinline__ cdptr as_const(const double *p) { return (cdptr)(p); }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
typedef const int __attribute__((address_space(4))) *ciptr;
__device__ __forceinline__ ciptr as_const(const int *p) { return (ciptr)(p); }
// analysis/thin row (m', l), m' <= l < L
__host__ __device__ __forceinline__ long long rowA(long long mp, long long l, long long L) {
  return mp * L - mp * (mp - 1) / 2 + (l - mp);
}

// start value of the l-chain of (m', m) at l0 = max(m', m)
__device__ __forceinline__ double lchain_start(const double *__restrict__ S0, int mp, int m) {
  if (mp >= m) {
    const double v = S0[tri0(mp) + m];
    return ((mp - m) & 1) ? -v : v;
  }
  return S0[tri0(m) + mp];
}

}  // namespace s2dw
