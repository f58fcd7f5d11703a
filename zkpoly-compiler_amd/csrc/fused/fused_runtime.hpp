// Device helpers included by generated fused kernels (see codegen.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../common/poly_ptr.hpp"
#include "../field/bn254.hpp"
#include "../field/fr29.hpp"

namespace zkp {
namespace fused {

// PolyPtr -> index map (iter.cuh:309-327: a rotation becomes offset = len - rotate).
template <class P>
__device__ __forceinline__ PolyView view(const P& p) {
  PolyView v;
  v.ptr = const_cast<uint32_t*>(p.ptr);
  v.len = p.len;
  v.whole_len = p.whole_len ? p.whole_len : p.len;
  v.offset = p.rotate ? p.len - p.rotate : p.offset;
  return v;
}

// grid-stride launches: at most `cap` workgroups
inline unsigned grid_capped(uint64_t n, unsigned threads, unsigned cap) {
  const uint64_t g = (n + threads - 1) / threads;
  return (unsigned)(g < cap ? (g ? g : 1) : cap);
}

// Spill slots of generated kernels: slot s of a thread is two 16-byte planes and, in
// limbs, behind those of all slots, one of 4 bytes, each lane-contiguous over the
// `threads` threads of the kernel's capped grid, so a wave's spill or reload is
// coalesced.
// `me` is the thread's global index.  A plane's start is the same on all lanes and
// stays on the scalar unit, hidden from the compiler, which otherwise forms every
// plane's lane address before the loop and keeps them all in scratch.
template <class T>
__device__ __forceinline__ T& spill_at(char* spill, uint64_t plane_bytes, uint32_t me) {
  asm volatile("" : "+s"(plane_bytes));
  return *reinterpret_cast<T*>(spill + plane_bytes + me * (uint32_t)sizeof(T));
}
__device__ __forceinline__ void spill_store(char* spill, uint32_t me, uint64_t s, uint64_t slots, uint64_t threads, const Fr29& x) {
  spill_at<uint4>(spill, 32 * s * threads, me) = make_uint4((u32)x.l[0], (u32)x.l[1], (u32)x.l[2], (u32)x.l[3]);
  spill_at<uint4>(spill, (32 * s + 16) * threads, me) = make_uint4((u32)x.l[4], (u32)x.l[5], (u32)x.l[6], (u32)x.l[7]);
  spill_at<int32_t>(spill, (32 * slots + 4 * s) * threads, me) = x.l[8];
}
// In words the planes' addresses are left to the compiler.
__device__ __forceinline__ void spill_store(char* spill, uint32_t me, uint64_t s, uint64_t, uint64_t threads, const Fr& x) {
  uint4* p = reinterpret_cast<uint4*>(spill) + me;
  p[2 * s * threads] = make_uint4(x.v[0], x.v[1], x.v[2], x.v[3]);
  p[(2 * s + 1) * threads] = make_uint4(x.v[4], x.v[5], x.v[6], x.v[7]);
}
template <class T>
__device__ __forceinline__ T spill_load(char* spill, uint32_t me, uint64_t s, uint64_t slots, uint64_t threads) {
  if constexpr (std::is_same<T, Fr>::value) {
    const uint4* p = reinterpret_cast<const uint4*>(spill) + me;
    const uint4 a = p[2 * s * threads], b = p[(2 * s + 1) * threads];
    return Fr{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w}};
  } else {
    const uint4 a = spill_at<uint4>(spill, 32 * s * threads, me), b = spill_at<uint4>(spill, (32 * s + 16) * threads, me);
    return Fr29{{(int32_t)a.x, (int32_t)a.y, (int32_t)a.z, (int32_t)a.w, (int32_t)b.x, (int32_t)b.y, (int32_t)b.z,
                 (int32_t)b.w, spill_at<int32_t>(spill, (32 * slots + 4 * s) * threads, me)}};
  }
}

// ---------------------------------------------------------------- kernels in 29-bit limbs
//
// Values are up: 32 x 2^256 mod r (fr29.hpp); the generator keeps their ranges.

__device__ __forceinline__ Fr29 load_up(const uint32_t* p) { return Fr29::from_words<5>(Fr::load(p).v); }

// Element idx of a view.  The address is taken as a distance from a kernel argument
// (any), hidden from the compiler: a pointer read from memory is accessed as a flat
// one, and an address that is used again is otherwise kept in registers, or in
// scratch, from the first use to the last.
__device__ __forceinline__ uint32_t* element(const PolyView& v, uint64_t idx, const void* anchor) {
  int64_t d = reinterpret_cast<char*>(v.elem(idx)) - reinterpret_cast<const char*>(anchor);
  asm volatile("" : "+v"(d));
  return reinterpret_cast<uint32_t*>(const_cast<char*>(reinterpret_cast<const char*>(anchor)) + d);
}
__device__ __forceinline__ Fr29 load_up(const PolyView& v, uint64_t idx, const void* anchor) {
  asm volatile("" : "+v"(idx));
  return load_up(element(v, idx, anchor));
}

// x as a product's second operand: hides from the compiler that carried limbs are
// not negative, or it multiplies them as unsigned by the other operand's signed
// limbs, in four instructions for one.
__device__ __forceinline__ Fr29 factor(Fr29 x) {
#pragma unroll
  for (int i = 0; i < 9; i++) asm("" : "+v"(x.l[i]));
  return x;
}

// A computed value, formed where the source forms it.  Left alone the compiler puts
// sums off until they are used and holds their operands instead: a kernel of 24
// columns, 71 products and a running sum kept 1 380 bytes of scratch and took 395 us
// over 2^18 elements, with this none and 176 (in words 222).
__device__ __forceinline__ Fr29 pinned(Fr29 x) {
  asm volatile(""
               : "+v"(x.l[0]), "+v"(x.l[1]), "+v"(x.l[2]), "+v"(x.l[3]), "+v"(x.l[4]), "+v"(x.l[5]), "+v"(x.l[6]),
                 "+v"(x.l[7]), "+v"(x.l[8]));
  return x;
}

// A scalar that every lane computes with: kept on the vector unit, the scalar unit
// has no 64-bit multiply-add.
__device__ __forceinline__ Fr29 scalar_in(const uint32_t* p) { return factor(load_up(p)); }

__device__ __forceinline__ Fr29 neg(const Fr29& x) {
  Fr29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = -x.l[i];
  return r;
}
__device__ __forceinline__ Fr29 pick(bool c, const Fr29& a, const Fr29& b) {
  Fr29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = c ? a.l[i] : b.l[i];
  return r;
}
// x^e, x normalised and within 33 r
__device__ __forceinline__ Fr29 pow(Fr29 x, uint64_t e) {
  if (e == 0) return Fr29::from_words<5>(Fr::one().v);
  Fr29 r = x;
  bool started = false;
  for (;; e >>= 1) {
    if (e & 1) {
      r = started ? Fr29::mul(r, factor(x)) : x;
      started = true;
    }
    if (e == 1) return r;
    x = Fr29::mul(x, factor(x));
  }
}

// The canonical element of an up value: (x + c r) / 32 with c = -q + k, q as in
// reduce() and 0 <= k < 32 making the sum divisible (r = 1 mod 2^28), which is
// below (1.0002 + 31) r / 32; then one conditional subtraction.
__device__ __forceinline__ Fr down(const Fr29& x) {
  const int32_t top = x.l[8] + (x.l[7] >> 29);
  const int32_t q = (int32_t)floorf((float)top * (1.0f / 3171406.449f) - 0x1p-13f);
  const int32_t c = ((q - x.l[0]) & 31) - q;
  Fr29 t;
  int64_t acc = 0;
#pragma unroll
  for (int i = 0; i < 9; i++) {
    acc += (int64_t)-c * Fr29::NEG_R[i] + x.l[i];
    t.l[i] = i < 8 ? (int32_t)((u32)acc & (u32)Fr29::MASK) : (int32_t)acc;
    acc >>= 29;
  }
#pragma unroll
  for (int i = 0; i < 9; i++)
    t.l[i] = (int32_t)((u32)t.l[i] >> 5 | (i < 8 ? ((u32)t.l[i + 1] & 31) << 24 : 0));
  Fr y;
  t.to_words(y.v);
  return Fr::reduce_once(y);
}

__device__ __forceinline__ void store_down(const Fr29& x, const PolyView& v, uint64_t idx, bool live,
                                           const void* anchor) {
  const Fr y = down(x);
  asm volatile("" : "+v"(idx));
  if (live) y.store(element(v, idx, anchor));
}

// Entry of the scalar table: nine limbs in 12 words, as computed (put_raw).
__device__ __forceinline__ void put_raw(uint32_t* p, const Fr29& x) {
#pragma unroll
  for (int i = 0; i < 9; i++) p[i] = (u32)x.l[i];
}
__device__ __forceinline__ Fr29 entry(const uint32_t* p) {
  Fr29 x;
#pragma unroll
  for (int i = 0; i < 9; i++) x.l[i] = (int32_t)p[i];
  return x;
}

// The table's entries below 1.0002 r, by one workgroup that has written them.
__device__ __forceinline__ void reduce_entries(uint32_t* table, unsigned count) {
  __threadfence();
  __syncthreads();
  for (unsigned t = threadIdx.x; t < count; t += blockDim.x) put_raw(table + 12 * t, entry(table + 12 * t).reduce());
}

// largest k < n with prefix[k] <= g (prefix has n + 1 non-decreasing entries)
__device__ __forceinline__ unsigned instance_of(const unsigned long long* prefix, unsigned n, uint64_t g) {
  unsigned lo = 0, hi = n;  // invariant: prefix[lo] <= g < prefix[hi]
  while (hi - lo > 1) {
    const unsigned mid = (lo + hi) >> 1;
    if (prefix[mid] <= g)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

}  // namespace fused
}  // namespace zkp
