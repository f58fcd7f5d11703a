// libpoly.so -- BN254 Fr polynomial kernels for gfx950.
//
// C ABI of the reference's libpoly.so (core/src/poly/src/poly.h:4-28;
// cudaError_t -> hipError_t, cudaStream_t -> hipStream_t), bound by the
// closures of core/src/poly.rs.  Semantics:
//  * poly_add / poly_sub / poly_mul: element i < min(|a|, |b|) is a op b; the
//    rest of the longer operand is copied (for a - b with |a| < |b|: negated)
//    up to max(|a|, |b|) (poly_basic.cu:4-54, poly_basic.cuh:4-52);
//  * poly_zero / poly_one_coef / poly_one_lagrange: 0..0 / 1,0..0 / 1..1;
//  * inv_scalar (zero stays zero) / scalar_pow on one device element
//    (poly_basic.cu:65-73);
//  * scan_mul: in-place inclusive prefix product (scan_mul.cuh:7-27);
//  * batched_invert: x_i^-1 for x_i != 0, zero stays zero
//    (batched_invert.cuh:49-91), by Montgomery's trick within tiles;
//  * poly_eval: sum_i a_i x^i into a device element (poly_eval.cuh:8-71);
//  * kate_division: q_i = sum_{j>i} p_j b^(j-i-1), i.e. the quotient of
//    (p(X) - p(b)) / (X - b), with q_{n-1} = 0 (kate_division.cuh:55-83).
// Field arithmetic is exact, so any association order gives the reference's
// bytes; the work is organised for the GPU rather than after cub.
//
// Scans and folds take two launches: every workgroup folds its share of the
// elements to one value; then every workgroup derives its carry from the values
// of the shares before it and scans its share.  (A single workgroup between the
// two that scans the values costs a launch and a chain of its own; from at most
// 1 024 shares a carry takes four products and a wave scan.)  poly_eval is a fold
// and its total.  All arithmetic is in signed 29-bit limbs (Fr29).
//
// Temporary buffers follow the reference's protocol: with temp_buf == NULL
// the size is written to *temp_buf_size and nothing runs.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <utility>

#include "fr_lanes.hpp"
#include "scan.hpp"

namespace zkp {
namespace poly {

// ---------------------------------------------------------------- elementwise

// op: 0 add, 1 sub, 2 mul.  a is the longer operand; `neg` (sub with |a| < |b|
// swapped) means the result is b - a on the common part and -a on the tail.
__global__ void __launch_bounds__(TH)
    k_binary(PolyView r, PolyView a, PolyView b, uint64_t len, uint64_t upper, int op, bool neg) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < upper; i += stride) {
    const Fr x = ld(a, i);
    Fr y;
    if (i >= len) {
      y = (op == 1 && neg) ? x.neg() : x;
    } else {
      const Fr z = ld(b, i);
      y = op == 0 ? x + z : op == 2 ? x * z : (neg ? z - x : x - z);
    }
    st(r, i, y);
  }
}

// mode: 0 all zero, 1 one then zeros, 2 all one
__global__ void __launch_bounds__(TH) k_fill(PolyView r, int mode) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < r.len; i += stride)
    st(r, i, (mode == 2 || (mode == 1 && i == 0)) ? Fr::one() : Fr::zero());
}

__global__ void __launch_bounds__(64) k_inv_scalar(uint32_t* x) {  // one wave
  Fr29 a = plain(Fr::load(x)).reduce();
  vary(a);
  const Fr y = canonical(Fr29Inverse::inverse(a, Fr29Inverse::INV_PLAIN));
  if (threadIdx.x == 0) y.store(x);
}

__global__ void k_pow_scalar(uint32_t* x, uint64_t e) {
  if (threadIdx.x == 0 && blockIdx.x == 0) Fr::load(x).pow(e).store(x);
}

// ---------------------------------------------------------------- prefix products

// A workgroup's share of a scan or fold is `len` consecutive elements, len a
// multiple of TH * PER.
//
// Products commute, so the fold takes its elements in lane order.  2^20 elements:
// 19 us, and the scan below 41, where 32-bit products, tiles of 2 048 and a
// workgroup between the two for the carries took 26 + 26 + 40.
__global__ void __launch_bounds__(TH)
    k_prod_fold(PolyView v, uint64_t n, uint64_t len, uint32_t* __restrict__ partial) {
  __shared__ WaveLds L;
  uint64_t k = (uint64_t)blockIdx.x * len + threadIdx.x;
  Fr a[4];
  auto fetch = [&](uint64_t k) {
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = k + j * TH < n ? ld(v, k + j * TH) : Fr::one();
  };
  fetch(k);
  Fr29 t = one_up();
#pragma unroll 1
  for (uint64_t done = 0; done < len; done += 4 * TH) {
    const Fr29 x0 = up(a[0]), x1 = up(a[1]), x2 = up(a[2]), x3 = up(a[3]);
    k += 4 * TH;
    if (done + 4 * TH < len) fetch(k);
    t = done ? Fr29::mul(t, x0) : x0;
    t = Fr29::mul(t, x1);
    t = Fr29::mul(t, x2);
    t = Fr29::mul(t, x3);
  }
  t = lanes_product(t);
  const uint32_t wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) L.put(wave, t);
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < TH / 64; w++) t = Fr29::mul(t, L.get(w));
    words(t).store(partial + (uint64_t)blockIdx.x * 8);
  }
}

// The prefix products of the workgroup's share: the fold of the shares before
// it (at most SHARES, PARTIALS a thread), then per TH * PER elements the threads'
// own products, a scan over them, and the elements again from the thread's
// carry-in.  The running product stays up and the element it meets is plain, so
// every product is an output at once.
template <int PER>
__global__ void __launch_bounds__(TH)
    k_prod_scan(PolyView v, uint64_t n, uint64_t len, const uint32_t* __restrict__ partial) {
  __shared__ WaveLds L, C;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  Fr29 carry = one_up();
  if (blockIdx.x) {
    Fr29 t = one_up();
    for (uint32_t j = threadIdx.x; j < blockIdx.x; j += TH) t = Fr29::mul(t, plain(Fr::load(partial + (uint64_t)j * 8)));
    t = lanes_product(t);
    if (lane == 0) C.put(wave, t);
    __syncthreads();
    carry = C.get(0);
    vary(carry);
    for (uint32_t w = 1; w < TH / 64; w++) carry = Fr29::mul(carry, C.get(w));
  }
#pragma unroll 1
  for (uint64_t done = 0; done < len; done += TH * PER) {
    const uint64_t k0 = (uint64_t)blockIdx.x * len + done + (uint64_t)threadIdx.x * PER;
    if (done && k0 - (uint64_t)threadIdx.x * PER >= n) break;  // the same for the whole workgroup
    Fr a[4];
    auto fetch = [&](uint64_t k) {
#pragma unroll
      for (int j = 0; j < 4; j++) a[j] = k + j < n ? ld(v, k + j) : Fr::one();
    };
    fetch(k0);
    Fr29 t;
#pragma unroll 1
    for (int at = 0; at < PER; at += 4) {
      const Fr29 x0 = up(a[0]), x1 = up(a[1]), x2 = up(a[2]), x3 = up(a[3]);
      if (at + 4 < PER) fetch(k0 + at + 4);
      t = at ? Fr29::mul(t, x0) : x0;
      t = Fr29::mul(t, x1);
      t = Fr29::mul(t, x2);
      t = Fr29::mul(t, x3);
    }
#pragma unroll 1
    for (uint32_t off = 1; off < 64; off <<= 1) {
      const Fr29 y = Fr29::mul(t, lanes_up(t, off));
      if (lane >= off) t = y;
    }
    if (lane == 63) L.put(wave, t);
    __syncthreads();
    Fr29 acc = carry;
    for (uint32_t w = 0; w < wave; w++) acc = Fr29::mul(acc, L.get(w));
    if (done + TH * PER < len)
      for (uint32_t w = 0; w < TH / 64; w++) carry = Fr29::mul(carry, L.get(w));
    const Fr29 before = Fr29::mul(acc, lanes_up(t, 1));
    if (lane) acc = before;
    fetch(k0);
#pragma unroll 1
    for (int at = 0; at < PER; at += 4) {
      Fr29 x[4];
#pragma unroll
      for (int j = 0; j < 4; j++) x[j] = plain(a[j]);
      if (at + 4 < PER) fetch(k0 + at + 4);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const Fr y = canonical(Fr29::mul(acc, x[j]));
        if (k0 + at + j < n) st(v, k0 + at + j, y);
        acc = up(y);
      }
    }
    __syncthreads();  // L is written again
  }
}

// ---------------------------------------------------------------- Horner folds and scans
//
// Elements are taken from the top: position k is index npad - 1 - k, npad the
// shares' total, indices from n on reading as zero.  Thread t's PER positions
// fold to s_t = sum p b^(what is below in the run), the state below them is
// (state above) b^PER + s_t.  All runs are whole, so the powers are the same on
// every lane and the scan carries no pairs: the level that adds M s_(t - off)
// squares M on lane 0, which has nothing to add.  Bound by products: at 2^21 an
// element costs one in the fold (34 us) and two in the quotient's scan (73 us) with
// 20 to 30 more per thread, against 62 + 34 + 107 us for scans over pairs of 32-bit
// products, eight elements a thread.

// s_t = sum over u <= t of m^(t - u) s_u within the wave; m becomes m^64.
// With POWER, *pw becomes m^lane.  s: limbs below 2 2^29, plain; m: up.
template <bool POWER>
__device__ __forceinline__ void horner_lanes(Fr29& s, Fr29& m, Fr29* pw) {
  const uint32_t lane = threadIdx.x & 63;
  if (POWER) *pw = one_up();
#pragma unroll 1
  for (uint32_t l = 0; l < 6; l++) {
    const uint32_t off = 1u << l;
    Fr29 x = lanes_up(s, off);
#pragma unroll
    for (int i = 0; i < 9; i++) x.l[i] = lane == 0 ? m.l[i] : x.l[i];
    const Fr29 p = Fr29::mul(x, m);
    if (POWER) {
      const Fr29 y = Fr29::mul(*pw, m);
      if ((lane >> l) & 1) *pw = y;
    }
#pragma unroll
    for (int i = 0; i < 9; i++) {
      s.l[i] += lane >= off ? p.l[i] : 0;
      m.l[i] = __builtin_amdgcn_readlane(p.l[i], 0);
    }
    s = s.norm();
  }
}

__device__ __forceinline__ Fr29 power_of_two(Fr29 m, uint32_t e) {  // m^e, e a power of two
  vary(m);
  for (; e > 1; e >>= 1) m = Fr29::mul(m, m);
  return m;
}

// Four elements from index `top` down; those from n on are zero.
__device__ __forceinline__ void fetch_down(const PolyView& v, uint64_t n, uint64_t top, Fr (&a)[4]) {
#pragma unroll
  for (int j = 0; j < 4; j++) a[j] = top - j < n ? ld(v, top - j) : Fr::zero();
}

// PER elements from index `top` down
template <int PER>
__device__ __forceinline__ Fr29 horner_run(const PolyView& v, uint64_t n, uint64_t top, const Fr29& b) {
  Fr a[4];
  fetch_down(v, n, top, a);
  Fr29 s = plain(a[0]);
#pragma unroll 1
  for (int done = 0; done < PER; done += 4) {
    const Fr29 x0 = plain(a[0]), x1 = plain(a[1]), x2 = plain(a[2]), x3 = plain(a[3]);
    if (done + 4 < PER) fetch_down(v, n, top - done - 4, a);
    if (done) s = Fr29::mul(s, b) + x0;
    s = Fr29::mul(s, b) + x1;
    s = Fr29::mul(s, b) + x2;
    s = Fr29::mul(s, b) + x3;
  }
  return s;
}

// ((t_0 m + t_1) m + ...) over the wave totals before wave `end`, from s
__device__ __forceinline__ Fr29 horner_waves(const WaveLds& L, Fr29 s, const Fr29& m, uint32_t end) {
  vary(s);
  for (uint32_t w = 0; w < end; w++) s = (Fr29::mul(s, m) + L.get(w)).norm();
  return s;
}

// total[b] = the fold of share b, of `rounds` (a power of two) times TH * PER
// positions; *power = x^len.  Without last_total the last share's total, which
// nobody reads, is not written and its place may be *power's.  With res (a single
// share) the fold is the result and goes there.
template <int PER>
__global__ void __launch_bounds__(TH)
    k_horner_fold(PolyView v, const uint32_t* x, uint64_t n, uint64_t npad, uint32_t rounds,
                  uint32_t* __restrict__ total, uint32_t* __restrict__ power, bool last_total, uint32_t* res) {
  __shared__ WaveLds L;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  Fr29 b = up(Fr::load(x));
  vary(b);
  Fr29 m = power_of_two(b, PER);
  uint64_t top = npad - 1 - ((uint64_t)blockIdx.x * rounds * TH + threadIdx.x) * PER;
  Fr29 s = horner_run<PER>(v, n, top, b);
  if (rounds > 1) {
    const Fr29 step = power_of_two(m, TH);
#pragma unroll 1
    for (uint32_t r = 1; r < rounds; r++) {
      top -= TH * PER;
      s = Fr29::mul(s, step) + horner_run<PER>(v, n, top, b);
      s = s.norm();
    }
  }
  horner_lanes<false>(s, m, nullptr);
  if (lane == 63) L.put(wave, s);
  __syncthreads();
  const bool last = blockIdx.x + 1 == gridDim.x;
  if (threadIdx.x == 0) {
    Fr29 acc = L.get(0);
    vary(acc);
    for (uint32_t w = 1; w < TH / 64; w++) acc = (Fr29::mul(acc, m) + L.get(w)).norm();
    if (res)
      canonical(acc).store(res);
    else if (!last || last_total)
      words(acc).store(total + (uint64_t)blockIdx.x * 8);
  }
  if (threadIdx.x == 64 && last && power) words(power_of_two(m, TH / 64 * rounds)).store(power);
}

// The state below `count` shares (their totals in order, each share scaled by m):
// every thread takes per of them, zeros standing before the first.
__device__ __forceinline__ Fr29 horner_shares(WaveLds& L, const uint32_t* __restrict__ total, uint32_t count, Fr29 m) {
  uint32_t per = 1;
  while (per * TH < count) per <<= 1;
  const int64_t at = (int64_t)count - (int64_t)per * TH + (int64_t)threadIdx.x * per;
  Fr29 s = at >= 0 ? plain(Fr::load(total + at * 8)) : plain(Fr::zero());
  vary(m);
  for (uint32_t j = 1; j < per; j++) {
    s = Fr29::mul(s, m);
    if (at + j >= 0) s = s + plain(Fr::load(total + (at + j) * 8));
  }
  m = power_of_two(m, per);
  horner_lanes<false>(s, m, nullptr);
  if ((threadIdx.x & 63) == 63) L.put(threadIdx.x >> 6, s);
  __syncthreads();
  Fr29 t = L.get(0);
  vary(t);
  for (uint32_t w = 1; w < TH / 64; w++) t = (Fr29::mul(t, m) + L.get(w)).norm();
  return t;
}

__global__ void __launch_bounds__(TH)
    k_horner_total(const uint32_t* __restrict__ total, uint32_t count, const uint32_t* __restrict__ power,
                   uint32_t* __restrict__ res) {
  __shared__ WaveLds L;
  const Fr29 t = horner_shares(L, total, count, plain(Fr::load(power)));
  if (threadIdx.x == 0) canonical(t).store(res);
}

// Kate's quotient of a share: q at index i is the state above it, q_{i-1} = p_i +
// b q_i.  p and q may be one array: a thread reads an index before it writes it.
template <int PER>
__global__ void __launch_bounds__(TH)
    k_kate(PolyView p, PolyView q, const uint32_t* b, uint64_t n, uint64_t npad, uint32_t rounds,
           const uint32_t* __restrict__ total, const uint32_t* __restrict__ power) {
  __shared__ WaveLds L, C;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  Fr29 bb = up(Fr::load(b));
  vary(bb);
  Fr29 carry = plain(Fr::zero());
  if (blockIdx.x) carry = horner_shares(C, total, blockIdx.x, plain(Fr::load(power)));
  const Fr29 run = power_of_two(bb, PER);
  Fr29 weight;
  uint64_t top = npad - 1 - ((uint64_t)blockIdx.x * rounds * TH + threadIdx.x) * PER;
#pragma unroll 1
  for (uint32_t r = 0; r < rounds; r++, top -= TH * PER) {
    Fr29 s = horner_run<PER>(p, n, top, bb), m = run;
    if (r == 0)
      horner_lanes<true>(s, m, &weight);
    else
      horner_lanes<false>(s, m, nullptr);
    if (lane == 63) L.put(wave, s);
    __syncthreads();
    const Fr29 above = horner_waves(L, carry, m, wave);
    if (r + 1 < rounds) carry = horner_waves(L, carry, m, TH / 64);
    const Fr29 before = lanes_up(s, 1);
    s = Fr29::mul(above, weight);
#pragma unroll
    for (int i = 0; i < 9; i++) s.l[i] += lane ? before.l[i] : 0;
    Fr a[4];
    fetch_down(p, n, top, a);
#pragma unroll 1
    for (int done = 0; done < PER; done += 4) {
      Fr29 x[4];
#pragma unroll
      for (int j = 0; j < 4; j++) x[j] = plain(a[j]);
      const uint64_t i = top - done;
      if (done + 4 < PER) fetch_down(p, n, i - 4, a);
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if (i - j < n) st(q, i - j, canonical(s));
        s = Fr29::mul(s, bb) + x[j];
      }
    }
    __syncthreads();  // L is written again
  }
}

// ---------------------------------------------------------------- batched inversion
//
// Montgomery's trick by tile, zeros read as one, each tile with an inversion of
// its own: one launch, and no tile waits for another.  One of the four waves inverts
// the tile's product while the others form, per thread, the product of all other
// threads' elements; which one goes by the tile, so that tiles on one CU use
// different SIMDs.  The tables of 55 KB leave two workgroups to a CU, two waves to a
// SIMD.  (A fifth wave for the inversion measured 92 to 119 us: one workgroup to a CU.)
// 2^20 elements: 60 us, bound by products (three an element, 15 a thread, and the
// inversion with every wave of the chip waiting for it), where a fold, one workgroup
// with one inversion on one lane and a rescan took 216.
constexpr int INV_PER = 8;
constexpr int INV_TILE = TH * INV_PER;

// f(0), ..., f(N - 1) with constant arguments (a loop over products is past what
// the compiler unrolls, and would index registers)
template <class F, int... I>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each(F&& f) {
  each_of(f, std::make_integer_sequence<int, N>{});
}

struct InvertLds {
  uint4 p0[6][TH], p1[6][TH];  // products of 2^l lanes, limbs 0-3, 4-7 and 8
  int32_t p2[6][TH];
  WaveLds wave;  // the waves' products, then (slot 4) the inverse of all

  __device__ __forceinline__ Fr29 get(uint32_t l, uint32_t i) const { return limbs_of(p0[l][i], p1[l][i], p2[l][i]); }
  __device__ __forceinline__ void put(uint32_t l, uint32_t i, const Fr29& x) {
    p0[l][i] = make_uint4((u32)x.l[0], (u32)x.l[1], (u32)x.l[2], (u32)x.l[3]);
    p1[l][i] = make_uint4((u32)x.l[4], (u32)x.l[5], (u32)x.l[6], (u32)x.l[7]);
    p2[l][i] = x.l[8];
  }
};

__global__ void __launch_bounds__(TH) k_invert(PolyView v, uint64_t n) {
  __shared__ InvertLds L;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const uint64_t k0 = (uint64_t)blockIdx.x * INV_TILE + (uint64_t)threadIdx.x * INV_PER;
  auto element = [&](int j) { return k0 + j < n ? ld(v, k0 + j) : Fr::one(); };
  Fr29 before[INV_PER];  // the product of the thread's elements 0 .. j - 1
  Fr29 t;
  {
    Fr x[INV_PER];
#pragma unroll
    for (int j = 0; j < INV_PER; j++) x[j] = element(j);
    each<INV_PER>([&](auto j) {
      const Fr29 y = up(x[j].is_zero() ? Fr::one() : x[j]);
      before[j] = t;
      t = j ? Fr29::mul(t, y) : y;
    });
  }
#pragma unroll 1
  for (uint32_t l = 0; l < 6; l++) {
    L.put(l, threadIdx.x, t);
    wave_sync();
    t = Fr29::mul(t, L.get(l, threadIdx.x ^ (1u << l)));
  }
  if (lane == 0) L.wave.put(wave, t);
  __syncthreads();
  if (wave == (blockIdx.x & (TH / 64 - 1))) {
    vary(t);
    for (uint32_t w = 1; w < TH / 64; w++) t = Fr29::mul(t, L.wave.get((wave + w) % (TH / 64)));
    t = Fr29Inverse::inverse(t.reduce(), Fr29Inverse::INV_UP);
    if (lane == 0) L.wave.put(TH / 64, t);
  }
  Fr29 others = L.get(0, threadIdx.x ^ 1);
#pragma unroll 1
  for (uint32_t l = 1; l < 6; l++) others = Fr29::mul(others, L.get(l, threadIdx.x ^ (1u << l)));
  for (uint32_t w = 1; w < TH / 64; w++) others = Fr29::mul(others, L.wave.get((wave + w) % (TH / 64)));
  __syncthreads();
  // read again, an element ahead, instead of held in 64 registers from the first time
  Fr x = element(INV_PER - 1);
  Fr29 inv = Fr29::mul(L.wave.get(TH / 64), others);  // of the thread's own product
  each<INV_PER>([&](auto i) {
    constexpr int j = INV_PER - 1 - i;
    const bool zero = x.is_zero();
    const Fr29 xj = up(zero ? Fr::one() : x);
    if (j) x = element(j - 1);
    const Fr y = canonical(j ? Fr29::mul(inv, before[j]) : inv);
    if (k0 + j < n) st(v, k0 + j, zero ? Fr::zero() : y);
    if (j) inv = Fr29::mul(inv, xj);
  });
}



}  // namespace poly
}  // namespace zkp

using namespace zkp;
using namespace zkp::poly;

// ---------------------------------------------------------------- C ABI

static hipError_t binary(PolyPtr r, ConstPolyPtr a, ConstPolyPtr b, hipStream_t stream, int op) {
  PolyView vr, va, vb;
  if (!make_view(r, &vr) || !make_view(a, &va) || !make_view(b, &vb)) return hipErrorInvalidValue;
  bool neg = false;
  if (va.len < vb.len) {
    const PolyView t = va;
    va = vb;
    vb = t;
    neg = true;  // only sub uses it
  }
  const uint64_t len = vb.len, upper = va.len;
  if (upper == 0) return hipSuccess;
  if (vr.len < upper || vr.ptr == nullptr || va.ptr == nullptr || (len && vb.ptr == nullptr))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_binary, dim3(grid_for(upper)), dim3(TH), 0, stream, vr, va, vb, len, upper, op,
                     op == 1 && neg);
  return hipGetLastError();
}

static hipError_t fill(PolyPtr r, hipStream_t stream, int mode) {
  PolyView v;
  if (!make_view(r, &v)) return hipErrorInvalidValue;
  if (v.len == 0) return hipSuccess;
  if (v.ptr == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_fill, dim3(grid_for(v.len)), dim3(TH), 0, stream, v, mode);
  return hipGetLastError();
}

// Shares of a scan or fold of n > 0 elements: 4 to max_per elements a thread, the
// fewest that leave at most 256 workgroups -- one wave per SIMD, which already
// keeps a SIMD busy with products, so longer runs mean less of the fixed work of
// a workgroup (scan levels, carries) and shorter ones a quicker small call --
// then rounds over as many workgroups as a carry is computed from (SHARES).
constexpr uint64_t SHARES = 1024;
struct Shares {
  uint64_t len;
  uint32_t count, rounds;
  int per;
};
static Shares shares_of(uint64_t n, int max_per) {
  Shares s{0, 0, 1, 4};
  while (s.per < max_per && n > (uint64_t)TH * s.per * 256) s.per *= 2;
  while (n > (uint64_t)TH * s.per * s.rounds * SHARES) s.rounds *= 2;
  s.len = (uint64_t)TH * s.per * s.rounds;
  s.count = (uint32_t)((n + s.len - 1) / s.len);
  return s;
}

static void launch_horner_fold(const Shares& s, const PolyView& v, const uint32_t* x, uint32_t* total, uint32_t* power,
                               bool last_total, uint32_t* res, hipStream_t stream) {
  const uint64_t npad = s.len * s.count;
  auto* k = s.per == 4 ? k_horner_fold<4> : s.per == 8 ? k_horner_fold<8> : s.per == 16 ? k_horner_fold<16>
                                                                                        : k_horner_fold<32>;
  hipLaunchKernelGGL(k, dim3(s.count), dim3(TH), 0, stream, v, x, v.len, npad, s.rounds, total, power, last_total, res);
}

// ---------------------------------------------------------------- batched inversion launch

static size_t invert_part_bytes(uint64_t n) { return align256(tiles_of(n ? n : 1) * sizeof(Fr)); }

// What batched_invert asks its caller for: three products a tile and one element.
// Its kernel keeps them in LDS and reads none of it; the size stays what callers' plans
// and the runtime's checks hold.
static size_t invert_temp_bytes(uint64_t n) { return 3 * invert_part_bytes(n) + align256(sizeof(Fr)); }

static hipError_t invert_launch(const PolyView& v, hipStream_t stream) {
  const uint64_t n = v.len;
  if (n == 0) return hipSuccess;
  if (v.ptr == nullptr) return hipErrorInvalidValue;
  const uint64_t nb = (n + INV_TILE - 1) / INV_TILE;
  if (nb > 0x7fffffffull) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_invert, dim3((unsigned)nb), dim3(TH), 0, stream, v, n);
  return hipGetLastError();
}

// The longest polynomial zkp_batched_invert_noalloc takes: what its interface has
// always refused stays refused, though no scratch array sets the limit any more.
#define ZKP_INVERT_NOALLOC_MAX_LEN (1ull << 26)

extern "C" {

// r = a + b (poly.h:4)
hipError_t poly_add(PolyPtr r, ConstPolyPtr a, ConstPolyPtr b, hipStream_t stream) { return binary(r, a, b, stream, 0); }

// r = a - b (poly.h:6)
hipError_t poly_sub(PolyPtr r, ConstPolyPtr a, ConstPolyPtr b, hipStream_t stream) { return binary(r, a, b, stream, 1); }

// r = a * b elementwise (poly.h:8)
hipError_t poly_mul(PolyPtr r, ConstPolyPtr a, ConstPolyPtr b, hipStream_t stream) { return binary(r, a, b, stream, 2); }

// every element one (poly.h:10)
hipError_t poly_one_lagrange(PolyPtr target, hipStream_t stream) { return fill(target, stream, 2); }

// 1, 0, ..., 0 (poly.h:12)
hipError_t poly_one_coef(PolyPtr target, hipStream_t stream) { return fill(target, stream, 1); }

// every element zero (poly.h:14)
hipError_t poly_zero(PolyPtr target, hipStream_t stream) { return fill(target, stream, 0); }

// *res = sum_i poly_i x^i; res and x are device elements (poly.h:16)
hipError_t poly_eval(void* temp_buf, unsigned long* temp_buf_size, ConstPolyPtr poly, unsigned int* res,
                     const unsigned int* x, hipStream_t stream) {
  PolyView v;
  if (!make_view(poly, &v)) return hipErrorInvalidValue;
  const size_t part = align256(tiles_of(v.len ? v.len : 1) * 2 * sizeof(Fr));
  if (temp_buf == nullptr) {
    if (temp_buf_size == nullptr) return hipErrorInvalidValue;
    *temp_buf_size = part + align256(2 * sizeof(Fr));
    return hipSuccess;
  }
  if (res == nullptr || x == nullptr) return hipErrorInvalidValue;
  if (v.len == 0) {
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(TH), 0, stream, PolyView{res, 1, 0, 1}, 0);
    return hipGetLastError();
  }
  if (v.ptr == nullptr) return hipErrorInvalidValue;
  const Shares s = shares_of(v.len, 32);  // at most two totals to a tile of `part`
  auto* total = reinterpret_cast<uint32_t*>(temp_buf);
  if (s.count == 1) {
    launch_horner_fold(s, v, x, total, nullptr, true, res, stream);
    return hipGetLastError();
  }
  auto* power = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(temp_buf) + part);
  launch_horner_fold(s, v, x, total, power, true, nullptr, stream);
  hipLaunchKernelGGL(k_horner_total, dim3(1), dim3(TH), 0, stream, total, s.count, power, res);
  return hipGetLastError();
}

// q = (p(X) - p(b)) / (X - b) for p of 2^log_p coefficients, q_{n-1} = 0
// (poly.h:18)
hipError_t kate_division(void* temp_buf, unsigned long* temp_buf_size, unsigned int log_p, ConstPolyPtr p,
                         const unsigned int* b, PolyPtr q, hipStream_t stream) {
  if (log_p > 40) return hipErrorInvalidValue;
  const uint64_t n = 1ull << log_p;
  const size_t part = align256(tiles_of(n) * 2 * sizeof(Fr));
  if (temp_buf == nullptr) {
    if (temp_buf_size == nullptr) return hipErrorInvalidValue;
    *temp_buf_size = 2 * part;
    return hipSuccess;
  }
  PolyView vp, vq;
  if (!make_view(p, &vp) || !make_view(q, &vq) || vp.len != n || vq.len != n) return hipErrorInvalidValue;
  if (vp.ptr == nullptr || vq.ptr == nullptr || b == nullptr) return hipErrorInvalidValue;
  if (tiles_of(n) > 0x7fffffffull) return hipErrorInvalidValue;
  const Shares s = shares_of(n, 32);
  auto* total = reinterpret_cast<uint32_t*>(temp_buf);
  uint32_t* power = total + (uint64_t)(s.count - 1) * 8;  // no share follows the last one
  if (s.count > 1) launch_horner_fold(s, vp, b, total, power, false, nullptr, stream);
  auto* k = s.per == 4 ? k_kate<4> : s.per == 8 ? k_kate<8> : s.per == 16 ? k_kate<16> : k_kate<32>;
  hipLaunchKernelGGL(k, dim3(s.count), dim3(TH), 0, stream, vp, vq, b, n, s.len * s.count, s.rounds, total, power);
  return hipGetLastError();
}

// target_i = target_0 * ... * target_i in place (poly.h:20)
hipError_t scan_mul(void* temp_buffer, unsigned long* buffer_size, PolyPtr target, hipStream_t stream) {
  PolyView v;
  if (!make_view(target, &v)) return hipErrorInvalidValue;
  const uint64_t nb = tiles_of(v.len ? v.len : 1);
  const size_t part = align256(nb * sizeof(Fr));
  if (temp_buffer == nullptr) {
    if (buffer_size == nullptr) return hipErrorInvalidValue;
    *buffer_size = 2 * part;
    return hipSuccess;
  }
  if (v.len == 0) return hipSuccess;
  if (v.ptr == nullptr) return hipErrorInvalidValue;
  if (nb > 0x7fffffffull) return hipErrorInvalidValue;
  auto* partial = reinterpret_cast<uint32_t*>(temp_buffer);
  const Shares s = shares_of(v.len, 16);  // at most two partials to a tile
  if (s.count > 1)
    hipLaunchKernelGGL(k_prod_fold, dim3(s.count), dim3(TH), 0, stream, v, v.len, s.len, partial);
  auto* k = s.per == 4 ? k_prod_scan<4> : s.per == 8 ? k_prod_scan<8> : k_prod_scan<16>;
  hipLaunchKernelGGL(k, dim3(s.count), dim3(TH), 0, stream, v, v.len, s.len, partial);
  return hipGetLastError();
}

// poly_i = poly_i^-1 in place, zeros kept (poly.h:22)
hipError_t batched_invert(void* temp_buffer, unsigned long* buffer_size, PolyPtr poly, hipStream_t stream) {
  PolyView v;
  if (!make_view(poly, &v)) return hipErrorInvalidValue;
  if (temp_buffer == nullptr) {
    if (buffer_size == nullptr) return hipErrorInvalidValue;
    *buffer_size = invert_temp_bytes(v.len);
    return hipSuccess;
  }
  return invert_launch(v, stream);
}

// batched_invert without a temporary buffer; up to ZKP_INVERT_NOALLOC_MAX_LEN.
hipError_t zkp_batched_invert_noalloc(PolyPtr poly, hipStream_t stream) {
  PolyView v;
  if (!make_view(poly, &v)) return hipErrorInvalidValue;
  if (v.len > ZKP_INVERT_NOALLOC_MAX_LEN) return hipErrorInvalidValue;
  return invert_launch(v, stream);
}

// *target = *target^-1, zero stays zero (poly.h:24)
hipError_t inv_scalar(unsigned int* target, hipStream_t stream) {
  if (target == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_inv_scalar, dim3(1), dim3(64), 0, stream, target);
  return hipGetLastError();
}

// *target = *target^exp (poly.h:26)
hipError_t scalar_pow(unsigned int* target, unsigned long long exp, hipStream_t stream) {
  if (target == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pow_scalar, dim3(1), dim3(1), 0, stream, target, (uint64_t)exp);
  return hipGetLastError();
}

}  // extern "C"
