// Fr29 over the lanes of a wave: conversions, shuffles and the small LDS tables of
// libpoly.so's scans and folds.  "plain" and "up" are the two forms of fr29.hpp:
// up * up is up, plain * up is plain, an up factor is the second operand.
#pragma once
#include <hip/hip_runtime.h>

#include "../field/fr29.hpp"

namespace zkp {
namespace poly {

__device__ __forceinline__ Fr29 plain(const Fr& x) { return Fr29::from_words<0>(x.v); }
__device__ __forceinline__ Fr29 up(const Fr& x) { return Fr29::from_words<5>(x.v); }
__device__ __forceinline__ Fr29 one_up() { return up(Fr::one()); }

// Words of x below 1.0002 r (either form), and the canonical element of a plain x.
__device__ __forceinline__ Fr words(const Fr29& x) {
  Fr y;
  x.reduce().to_words(y.v);
  return y;
}
__device__ __forceinline__ Fr canonical(const Fr29& x) { return Fr::reduce_once(words(x)); }

// Keeps a value that is the same on all lanes on the vector unit: the scalar unit
// has no 64-bit multiply-add and takes several instructions for each.
__device__ __forceinline__ void vary(Fr29& x) {
#pragma unroll
  for (int i = 0; i < 9; i++) asm("" : "+v"(x.l[i]));
}

__device__ __forceinline__ Fr29 lanes_up(const Fr29& x, uint32_t off) {  // lane t gets lane t - off
  Fr29 y;
#pragma unroll
  for (int i = 0; i < 9; i++) y.l[i] = __shfl_up(x.l[i], off);
  return y;
}

// The product of the wave's 64 up values, on every lane.
__device__ __forceinline__ Fr29 lanes_product(Fr29 x) {
#pragma unroll 1
  for (int off = 1; off < 64; off <<= 1) {
    Fr29 y;
#pragma unroll
    for (int i = 0; i < 9; i++) y.l[i] = __shfl_xor(x.l[i], off);
    x = Fr29::mul(x, y);
  }
  return x;
}

__device__ __forceinline__ Fr29 limbs_of(const uint4& a, const uint4& b, int32_t c) {
  return Fr29{{(int32_t)a.x, (int32_t)a.y, (int32_t)a.z, (int32_t)a.w, (int32_t)b.x, (int32_t)b.y, (int32_t)b.z,
               (int32_t)b.w, c}};
}

// One value per wave of a workgroup (and one more).
struct WaveLds {
  int32_t l[5][12];
  __device__ __forceinline__ Fr29 get(uint32_t w) const {
    Fr29 x;
#pragma unroll
    for (int i = 0; i < 9; i++) x.l[i] = l[w][i];
    return x;
  }
  __device__ __forceinline__ void put(uint32_t w, const Fr29& x) {
#pragma unroll
    for (int i = 0; i < 9; i++) l[w][i] = x.l[i];
  }
};

// LDS written by a lane is read by others of its wave behind this.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace poly
}  // namespace zkp
