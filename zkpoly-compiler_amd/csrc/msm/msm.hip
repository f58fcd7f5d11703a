// libzkp_msm.so -- Pippenger MSM over BN254 G1 (kernels + host orchestration).
//
// The reference's per-configuration libraries libmsm_bn254_<w>_<t>_<dbg>.so
// (core/src/msm.rs:100-111) are thin wrappers (msm_abi.cpp) that bind its C
// ABI -- msm / msm_precompute of core/src/msm/src/msm.h:4-11, cudaError_t ->
// hipError_t -- to zkp_msm_host / zkp_msm_precompute_host below with their
// compiled-in MsmConfig.  The zkp_msm_* entry points take the window at run
// time.
//
// Algorithm (result sum_i k_i P_i, affine; identity (0, 0)):
//  1. digits: scalar -> canonical integer -> ceil(254/s) signed s-bit digits in
//     [-2^(s-1), 2^(s-1)) (the reference's signed_digit, msm_impl.cuh:22-33);
//     logical window w uses point table w / n_windows and physical window
//     w % n_windows (precomputed tables 2^(j*n_windows*s) P, msm_impl.cuh:358-371).
//  2. sort of the (window, |digit|) keys with values (point index | sign << 31):
//     a two-level partition sort in LDS (coarse bins, then the low bucket
//     bits), no device atomics; windows above 20 bits use a device-atomic
//     counting sort instead.
//  3. bucket accumulation, load balanced: every thread owns a chunk of
//     consecutive sorted entries and adds each run of equal keys into an XYZZ
//     sum (mixed additions); a run cut by chunk edges leaves pieces that one
//     thread (or quad of lanes) per run adds up, and a run of many pieces (a
//     bucket holding a large share of the points, e.g. the scalar-1 bucket) goes
//     to a tree over all pieces instead, so it costs log steps, not a serial walk.
//     Buckets and partials are G1X29 (xyzz29.hpp): Fq in nine 29-bit limbs,
//     radix 2^261, lazily reduced -- one instruction per limb product.
//  4. bucket reduction per window, S_w = sum_b b * B_b, by halving levels
//     (X, Y) -> (2 (X_2i + X_2i+1), X_2i+1 + Y_2i + Y_2i+1): X' and Y' run on
//     different threads, two point operations deep per level, since a chain of
//     point additions is latency bound; the last 128 items of a window are
//     halved inside one workgroup (LDS), all levels in one launch, and the
//     window sums leave in G1XYZZ's form (8 x 32-bit limbs, radix 2^256).
//  5. host: Horner over the window sums (s doublings each) and one inversion
//     to affine -- the serial tail runs where a modular product is ~30x lower
//     latency than one GPU wave (measured 738 ns per dependent product).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <chrono>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#include "../curve/g1.hpp"
#include "../curve/xyzz29.hpp"

namespace zkp {
namespace msm {

constexpr int THREADS = 256;
constexpr uint32_t RED_TAIL = 128;  // items per window finished inside one workgroup
constexpr uint32_t SCALAR_BITS = 254;
constexpr int MAX_LEVELS = 24;

// How up to `entries` sorted entries are shared out for the accumulation: `ch`
// consecutive entries (a multiple of 4, read as 16-byte words) per thread, or
// per quad of lanes.  65 536 lanes are one wave on each of the 1 024 SIMDs.  An
// addition takes 4.5 us of a lone wave, 2.3 us of a quad; every chunk edge leaves
// a piece of a run that costs a general addition (1.4 times the products) later.
//  * Up to 800 K entries the chain of one chunk's additions sets the time, so
//    quads take it, sixteen entries each, fewer where a bucket holds only a few.
//  * Up to 4 M: two waves per SIMD, which fill the VALU nearly, in chunks of 16
//    to 32, so that a bucket of the usual 32 entries has few pieces.
//  * Above: all threads resident at once, four waves per SIMD, so that no last
//    round of workgroups runs nearly empty; up to 128 entries.
struct Share {
  uint32_t ch;
  bool quads;
};
static inline Share share_for(uint64_t entries) {
  const bool quads = entries <= 800000;
  uint64_t c;
  if (quads) {
    c = entries / 8192;
    if (c > 16) c = 16;
    if (c < 4) c = 4;
  } else {
    const uint64_t all = (entries + 262143) / 262144, two = (entries + 131071) / 131072;
    c = two < 16 ? 16 : two < 32 ? two : 32;
    if (all > c) c = all;
    if (c > 128) c = 128;
  }
  return Share{(uint32_t)((c + 3) & ~3ull), quads};
}

#define ZKP_CHECK(x)                          \
  do {                                        \
    hipError_t e_ = (x);                      \
    if (e_ != hipSuccess) return e_;          \
  } while (0)

struct Config {
  uint32_t s;               // window bits
  uint32_t actual_windows;  // ceil(254 / s)
  uint32_t n_windows;       // physical windows per table
  uint32_t n_precompute;    // point tables
  uint32_t buckets;         // 2^(s-1)
  uint32_t top_log;         // the top window's buckets come in 2^top_log copies each
  uint32_t bias[8];         // sum of 2^(s-1) 2^(s w) over the windows below the top one
};

static inline uint32_t div_ceil32(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// MsmConfig semantics of core/src/msm/src/msm.cuh:51-70 / common/src/msm_config.rs:14-24.
// Top s-bit window of r - 1 (the largest canonical scalar) starting at bit `bit`.
static uint32_t top_window_of_r_minus_1(uint32_t bit, uint32_t s) {
  uint32_t v[8];
  for (int i = 0; i < 8; i++) v[i] = FrParams::P[i];
  v[0] -= 1;  // r is odd
  const uint32_t limb = bit >> 5, off = bit & 31;
  uint64_t two = limb < 8 ? v[limb] : 0;
  if (limb + 1 < 8) two |= (uint64_t)v[limb + 1] << 32;
  return (uint32_t)((two >> off) & ((1ull << s) - 1));
}

static bool make_config(uint32_t s, uint32_t target, Config* c) {
  if (s < 2 || s > 24 || target == 0) return false;
  c->s = s;
  const uint32_t ref_windows = div_ceil32(SCALAR_BITS, s);  // the reference's count
  const uint32_t ref_n_windows = ref_windows < target ? ref_windows : target;
  const uint32_t ref_precompute = div_ceil32(ref_windows, ref_n_windows);
  c->actual_windows = ref_windows;
  // the signed recoding must not carry out of the top window: top digit + 1 <
  // 2^(s-1); where it can (s = 2, 3) one more window is needed
  if (top_window_of_r_minus_1((c->actual_windows - 1) * s, s) + 1 >= (1u << (s - 1))) c->actual_windows += 1;
  c->n_windows = c->actual_windows < target ? c->actual_windows : target;
  // a target covering the reference's windows covers the extra one too, so the
  // caller's table count (the reference's MsmConfig) stays right
  if (target >= ref_windows) c->n_windows = c->actual_windows;
  c->n_precompute = div_ceil32(c->actual_windows, c->n_windows);
  if (c->n_precompute != ref_precompute) return false;  // would need a table the caller does not have
  c->buckets = 1u << (s - 1);
  // The top window has 254 - s (windows - 1) bits, one to seven for most s, so
  // its digits would put n points into a handful of buckets.  Where no other
  // window shares its buckets (one table) digit d goes to bucket
  // (d - 1) 2^top_log + (point index mod 2^top_log) instead, and the bucket
  // reduction folds the copies in its first top_log levels: the same number of
  // additions, and no run of thousands of pieces (2^14 points, s = 10, 4 bits:
  // the long-run kernels took 125 us and now return at once).
  c->top_log = 0;
  if (c->n_precompute == 1 && c->n_windows == c->actual_windows) {
    const uint32_t top = top_window_of_r_minus_1((c->actual_windows - 1) * s, s) + 1;  // largest digit
    while ((top << (c->top_log + 1)) <= c->buckets) c->top_log++;
  }
  for (int i = 0; i < 8; i++) c->bias[i] = 0;
  for (uint32_t w = 0; w + 1 < c->actual_windows; w++) {
    const uint32_t bit = s * w + s - 1;
    c->bias[bit >> 5] |= 1u << (bit & 31);
  }
  return true;
}

// ---------------------------------------------------------------- digits

// The signed s-bit digits of a scalar, lowest window first.  With 2^(s-1) added
// at every window but the top one, window w's digit is its s bits minus
// 2^(s-1): no carry runs from digit to digit, and the value moves down s bits
// per window in registers (an index by bit position would put it in scratch).
struct Digits {
  uint32_t v[8];

  __device__ __forceinline__ Digits(const uint32_t* scalar, const Config& cfg) {
    const Fr c = Fr::load(scalar).to_canonical();
    uint32_t carry = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = adc(c.v[i], cfg.bias[i], carry);  // below 2^255
  }
  // an entry of no digits but zeros: all windows give 0
  __device__ __forceinline__ explicit Digits(const Config& cfg) {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = cfg.bias[i];
  }
  __device__ __forceinline__ int next(const Config& cfg, uint32_t w) {
    const uint32_t d = v[0] & ((1u << cfg.s) - 1);
#pragma unroll
    for (int i = 0; i < 7; i++) v[i] = __builtin_amdgcn_alignbit(v[i + 1], v[i], cfg.s);
    v[7] >>= cfg.s;
    return w + 1 < cfg.actual_windows ? (int)d - (int)(1u << (cfg.s - 1)) : (int)d;
  }
};

// Key of a nonzero digit d of window w: its bucket over all physical windows.
__device__ __forceinline__ uint32_t bucket_key(const Config& cfg, uint32_t w, int d, uint64_t i) {
  uint32_t b = (uint32_t)(d < 0 ? -d : d) - 1;
  if (w + 1 == cfg.actual_windows) b = (b << cfg.top_log) | ((uint32_t)i & ((1u << cfg.top_log) - 1));
  return (w % cfg.n_windows) * cfg.buckets + b;
}

// Wave-aggregated atomic increment of counter[bin] for the active lanes;
// returns each lane's previous value plus its rank among lanes with the same
// bin.  Up to 4 rounds serve the bin of the lowest active lane with a single
// atomic for all lanes sharing it; what is left (all-distinct bins) falls back
// to one atomic per lane.  This removes the serialisation on the few bins of a
// narrow top window (e.g. bits 252..253 for s = 12, 14, 18) and on a bucket that
// receives a fixed share of all scalars.  Must be called by the whole wave.
__device__ __forceinline__ uint32_t aggregated_increment(uint32_t* counter, uint32_t bin, bool active) {
  const uint32_t lane = __lane_id();
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  uint32_t result = 0;
  for (int round = 0; round < 4; round++) {
    const uint64_t act = __ballot(active);
    if (act == 0) return result;
    const int leader = __ffsll((long long)act) - 1;
    const uint32_t lbin = __shfl(bin, leader);
    const uint64_t same = __ballot(active && bin == lbin);
    if (round > 0 && __popcll(same) < 2) break;
    uint32_t start = 0;
    if ((int)lane == leader) start = atomicAdd(&counter[lbin], (uint32_t)__popcll(same));
    start = __shfl(start, leader);
    if (active && bin == lbin) {
      result = start + (uint32_t)__popcll(same & below);
      active = false;
    }
  }
  if (active) result = atomicAdd(&counter[bin], 1u);
  return result;
}

// All lanes of a wave run the same number of iterations (inactive tails keep
// participating in the wave-wide ballots).
__global__ void __launch_bounds__(THREADS)
    k_histogram(const uint32_t* __restrict__ scalars, uint64_t n, Config cfg, uint32_t* __restrict__ hist) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t rounds = (n + stride - 1) / stride;
  for (uint64_t r = 0; r < rounds; r++) {
    const uint64_t i = r * stride + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    Digits digits = valid ? Digits(scalars + i * 8, cfg) : Digits(cfg);
    for (uint32_t w = 0; w < cfg.actual_windows; w++) {
      const int d = digits.next(cfg, w);
      aggregated_increment(hist, bucket_key(cfg, w, d, i), d != 0);
    }
  }
}

__global__ void __launch_bounds__(THREADS)
    k_scatter(const uint32_t* __restrict__ scalars, uint64_t n, Config cfg, uint32_t* __restrict__ cursor,
              uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t rounds = (n + stride - 1) / stride;
  for (uint64_t r = 0; r < rounds; r++) {
    const uint64_t i = r * stride + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    Digits digits = valid ? Digits(scalars + i * 8, cfg) : Digits(cfg);
    for (uint32_t w = 0; w < cfg.actual_windows; w++) {
      const int d = digits.next(cfg, w);
      const uint32_t table = w / cfg.n_windows;
      const uint32_t key = bucket_key(cfg, w, d, i);
      const bool active = d != 0;
      const uint32_t pos = aggregated_increment(cursor, key, active);
      if (active) {
        keys[pos] = key;
        vals[pos] = (uint32_t)(table * n + i) | (d < 0 ? 0x80000000u : 0u);
      }
    }
  }
}

// ---------------------------------------------------------------- scan (exclusive, in place)

constexpr int SCAN_BLOCK = 1024;  // elements per block: 256 threads x 4

template <int NT = THREADS>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* sh, uint32_t* total) {
  // inclusive scan inside each wave by shuffles, then the waves' totals through LDS
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, 64);
    if (lane >= (uint32_t)off) x += y;
  }
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < NT / 64; w++) {
    const uint32_t t = sh[w];
    before += w < wave ? t : 0u;
    all += t;
  }
  *total = all;
  __syncthreads();  // sh is free again for the caller
  return before + x - v;
}

__global__ void __launch_bounds__(THREADS) k_scan_blocks(uint32_t* data, uint32_t n, uint32_t* block_sums) {
  __shared__ uint32_t sh[THREADS];
  const uint32_t base = blockIdx.x * SCAN_BLOCK + threadIdx.x * 4;
  uint32_t v[4];
  for (int k = 0; k < 4; k++) v[k] = base + k < n ? data[base + k] : 0;
  const uint32_t local = v[0] + v[1] + v[2] + v[3];
  uint32_t total;
  uint32_t pre = block_exclusive_scan(local, sh, &total);
  for (int k = 0; k < 4; k++) {
    if (base + k < n) data[base + k] = pre;
    pre += v[k];
  }
  if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

// single block: exclusive scan of up to 256 * 16 block sums
__global__ void __launch_bounds__(THREADS) k_scan_sums(uint32_t* sums, uint32_t nb) {
  __shared__ uint32_t sh[THREADS];
  const uint32_t per = (nb + THREADS - 1) / THREADS;
  const uint32_t base = threadIdx.x * per;
  uint32_t local = 0;
  for (uint32_t k = 0; k < per; k++)
    if (base + k < nb) local += sums[base + k];
  uint32_t total;
  uint32_t pre = block_exclusive_scan(local, sh, &total);
  for (uint32_t k = 0; k < per; k++) {
    if (base + k < nb) {
      const uint32_t x = sums[base + k];
      sums[base + k] = pre;
      pre += x;
    }
  }
}

__global__ void __launch_bounds__(THREADS) k_scan_add(uint32_t* data, uint32_t n, const uint32_t* block_sums,
                                                      uint32_t* cursor) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const uint32_t v = data[i] + block_sums[i / SCAN_BLOCK];
    data[i] = v;
    if (cursor) cursor[i] = v;
  }
}

// ---------------------------------------------------------------- partition sort
//
// Sorts the (key, value) entries by key without device atomics, in two levels.
// A key is pw * buckets + |d| - 1; its coarse bin is key >> low_bits (the
// physical window and the top bits of the bucket).
//  1. k_part_count: every tile of `tp` points counts its entries per coarse
//     bin in LDS and writes the counts to matrix[bin * tiles + tile]; an
//     exclusive scan of the matrix gives every (bin, tile) run its place.
//  2. k_part_scatter: every tile ranks its entries within their bins in LDS,
//     stages them in bin order and writes each run contiguously.
//  3. k_seg_*: every coarse bin's segment is sorted by the low bits in slices
//     (LDS counting, one device atomic per nonzero bucket per slice of a
//     multi-slice segment).  The order inside a bucket is not kept; bucket
//     sums do not depend on it.

struct SortPlan {
  uint32_t low_bits;  // bits of the bucket sorted by the second level (<= 12)
  uint32_t nc;        // coarse bins: n_windows << (s - 1 - low_bits)
  uint32_t tp;        // points per tile
  uint32_t tiles;
  uint32_t lds_part;  // dynamic LDS of k_part_scatter (bytes)
};

// Counts the tile's nonzero digits per coarse bin into cnt (LDS, zeroed by the caller).
__device__ __forceinline__ void part_count_tile(const uint32_t* __restrict__ scalars, uint64_t n, const Config& cfg,
                                                uint32_t low_bits, uint64_t first, uint32_t tp, uint32_t* cnt) {
  for (uint32_t p = threadIdx.x; p < tp; p += THREADS) {
    const uint64_t i = first + p;
    if (i >= n) break;
    Digits digits(scalars + i * 8, cfg);
    for (uint32_t w = 0; w < cfg.actual_windows; w++) {
      const int d = digits.next(cfg, w);
      if (d != 0) atomicAdd(&cnt[bucket_key(cfg, w, d, i) >> low_bits], 1u);
    }
  }
}

// Also clears what the later kernels add into: the matrix's last entry and the
// H bucket counts of k_seg_hist.
__global__ void __launch_bounds__(THREADS)
    k_part_count(const uint32_t* __restrict__ scalars, uint64_t n, Config cfg, SortPlan sp,
                 uint32_t* __restrict__ matrix, uint32_t* __restrict__ ghist) {
  extern __shared__ uint32_t dyn[];
  uint32_t* cnt = dyn;  // nc
  for (uint32_t b = threadIdx.x; b < sp.nc; b += THREADS) cnt[b] = 0;
  __syncthreads();
  part_count_tile(scalars, n, cfg, sp.low_bits, (uint64_t)blockIdx.x * sp.tp, sp.tp, cnt);
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < sp.nc; b += THREADS) matrix[(uint64_t)b * sp.tiles + blockIdx.x] = cnt[b];
  if (blockIdx.x == 0 && threadIdx.x == 0) matrix[(uint64_t)sp.nc * sp.tiles] = 0;
  const uint32_t H = cfg.n_windows * cfg.buckets;
  for (uint32_t b = blockIdx.x * THREADS + threadIdx.x; b < H; b += gridDim.x * THREADS) ghist[b] = 0;
}

// Exclusive scan of a[0..m) in LDS by the whole block; sh is NT / 64 words of scratch.
template <int NT = THREADS>
__device__ __forceinline__ void lds_exclusive_scan(uint32_t* a, uint32_t m, uint32_t* sh) {
  const uint32_t per = (m + NT - 1) / NT;
  const uint32_t base = threadIdx.x * per;
  uint32_t local = 0;
  for (uint32_t k = 0; k < per; k++)
    if (base + k < m) local += a[base + k];
  uint32_t total;
  uint32_t pre = block_exclusive_scan<NT>(local, sh, &total);
  for (uint32_t k = 0; k < per; k++) {
    if (base + k < m) {
      const uint32_t x = a[base + k];
      a[base + k] = pre;
      pre += x;
    }
  }
  __syncthreads();
}

// Points per thread and windows per point whose entries k_part_scatter keeps
// in registers, with each entry's rank in its bin from the counting atomic:
// one digit pass over the tile instead of a counting pass and a placing pass.
// Other tile shapes take the two passes.
constexpr uint32_t PART_PPT = 2, PART_WMAX = 22;

__global__ void __launch_bounds__(THREADS)
    k_part_scatter(const uint32_t* __restrict__ scalars, uint64_t n, Config cfg, SortPlan sp,
                   const uint32_t* __restrict__ offsets, uint32_t* __restrict__ keys_out,
                   uint32_t* __restrict__ vals_out) {
  extern __shared__ uint32_t dyn[];
  __shared__ uint32_t sh[THREADS];
  uint32_t* base = dyn;               // nc: entries of each bin, then its first staging slot
  uint32_t* cur = dyn + sp.nc;        // nc: entries of each bin / staging cursor
  uint32_t* skey = dyn + 2 * sp.nc;   // tp * actual_windows
  uint32_t* sval = skey + (size_t)sp.tp * cfg.actual_windows;
  const uint64_t first = (uint64_t)blockIdx.x * sp.tp;
  for (uint32_t b = threadIdx.x; b < sp.nc; b += THREADS) base[b] = 0;
  __syncthreads();
  const bool regs = sp.tp == PART_PPT * THREADS && cfg.actual_windows <= PART_WMAX;  // uniform
  uint32_t ek[PART_PPT][PART_WMAX], er[PART_PPT][PART_WMAX];  // key | sign << 31 (~0: none), rank
  if (regs) {
#pragma unroll
    for (uint32_t p = 0; p < PART_PPT; p++) {
      const uint64_t i = first + p * THREADS + threadIdx.x;
      const bool valid = i < n;
      Digits digits = valid ? Digits(scalars + i * 8, cfg) : Digits(cfg);
#pragma unroll
      for (uint32_t w = 0; w < PART_WMAX; w++) {
        ek[p][w] = ~0u;
        er[p][w] = 0;
        if (w < cfg.actual_windows) {
          const int d = digits.next(cfg, w);
          if (d != 0) {
            const uint32_t key = bucket_key(cfg, w, d, i);
            ek[p][w] = key | (d < 0 ? 0x80000000u : 0u);
            er[p][w] = atomicAdd(&base[key >> sp.low_bits], 1u);
          }
        }
      }
    }
  } else {
    part_count_tile(scalars, n, cfg, sp.low_bits, first, sp.tp, base);
  }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < sp.nc; b += THREADS) cur[b] = base[b];
  lds_exclusive_scan(base, sp.nc, sh);
  uint32_t staged;
  if (regs) {
#pragma unroll
    for (uint32_t p = 0; p < PART_PPT; p++) {
      const uint32_t i = (uint32_t)(first + p * THREADS + threadIdx.x);
#pragma unroll
      for (uint32_t w = 0; w < PART_WMAX; w++) {
        if (ek[p][w] == ~0u) continue;
        const uint32_t key = ek[p][w] & 0x7fffffffu;
        const uint32_t slot = base[key >> sp.low_bits] + er[p][w];
        skey[slot] = key;
        sval[slot] = (uint32_t)((w / cfg.n_windows) * n + i) | (ek[p][w] & 0x80000000u);
      }
    }
    staged = base[sp.nc - 1] + cur[sp.nc - 1];
  } else {
    for (uint32_t b = threadIdx.x; b < sp.nc; b += THREADS) cur[b] = base[b];
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < sp.tp; p += THREADS) {
      const uint64_t i = first + p;
      if (i >= n) break;
      Digits digits(scalars + i * 8, cfg);
      for (uint32_t w = 0; w < cfg.actual_windows; w++) {
        const int d = digits.next(cfg, w);
        if (d == 0) continue;
        const uint32_t key = bucket_key(cfg, w, d, i);
        const uint32_t slot = atomicAdd(&cur[key >> sp.low_bits], 1u);
        skey[slot] = key;
        sval[slot] = (uint32_t)((w / cfg.n_windows) * n + i) | (d < 0 ? 0x80000000u : 0u);
      }
    }
    __syncthreads();
    staged = cur[sp.nc - 1];  // the last bin's cursor ends at the tile's entry count
  }
  __syncthreads();
  for (uint32_t slot = threadIdx.x; slot < staged; slot += THREADS) {
    const uint32_t key = skey[slot];
    const uint32_t b = key >> sp.low_bits;
    const uint32_t dst = offsets[(uint64_t)b * sp.tiles + blockIdx.x] + (slot - base[b]);
    keys_out[dst] = key;
    vals_out[dst] = sval[slot];
  }
}

// Second level: every coarse bin's segment is sorted by the low bits in slices
// of at most SEG_SLICE entries, so a segment holding most entries of a narrow
// window (s = 12, 13, 14, 18 and the small windows) is spread over many
// workgroups.  A segment of one slice is counted and placed by that slice's
// workgroup alone; the bucket counts of a longer one are added up first, with
// one device atomic per nonzero bucket per slice (k_seg_hist, k_seg_scan).
constexpr uint32_t SEG_SLICE = 8192;  // entries per workgroup, staged in LDS at once (64 KB)
constexpr uint32_t SEG_PER_THREAD = SEG_SLICE / THREADS;

// largest k < n with prefix[k] <= g (prefix: n + 1 non-decreasing entries)
__device__ __forceinline__ uint32_t find_segment(const uint32_t* prefix, uint32_t n, uint32_t g) {
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (prefix[mid] <= g)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

__device__ __forceinline__ uint32_t seg_begin(const uint32_t* offsets, const SortPlan& sp, uint32_t cb) {
  return offsets[(uint64_t)cb * sp.tiles];
}

// slice_prefix[cb] = slices of the segments before cb (nc + 1 entries, cnt: LDS
// of as many words), and the entry count; one workgroup of NT threads.
template <int NT>
__device__ __forceinline__ void seg_plan(const uint32_t* offsets, const SortPlan& sp, uint32_t* slice_prefix,
                                         uint32_t* counts, uint32_t* cnt, uint32_t* sh) {
  for (uint32_t cb = threadIdx.x; cb <= sp.nc; cb += NT) {
    uint32_t k = 0;
    if (cb < sp.nc) {
      const uint32_t size = seg_begin(offsets, sp, cb + 1) - seg_begin(offsets, sp, cb);
      k = (size + SEG_SLICE - 1) / SEG_SLICE;
    }
    cnt[cb] = k;
  }
  if (threadIdx.x == 0) counts[0] = seg_begin(offsets, sp, sp.nc);
  __syncthreads();
  lds_exclusive_scan<NT>(cnt, sp.nc + 1, sh);
  for (uint32_t cb = threadIdx.x; cb <= sp.nc; cb += NT) slice_prefix[cb] = cnt[cb];
}

__global__ void __launch_bounds__(THREADS)
    k_seg_plan(const uint32_t* __restrict__ offsets, SortPlan sp, uint32_t* __restrict__ slice_prefix,
               uint32_t* __restrict__ counts) {
  __shared__ uint32_t sh[THREADS];
  extern __shared__ uint32_t cnt[];  // nc + 1
  seg_plan<THREADS>(offsets, sp, slice_prefix, counts, cnt, sh);
}

// The scan of a small matrix (m entries) and the slice plan in one launch of
// one workgroup: 1 024 threads take 4 096 entries a step.  Up to
// SCAN_SMALL_MAX entries its steps (1 us each) take less than the four launches
// of the tiled scan and k_seg_plan (18 us).
constexpr int SCAN_SMALL_THREADS = 1024;
constexpr uint32_t SCAN_SMALL_MAX = 32768;
__global__ void __launch_bounds__(SCAN_SMALL_THREADS)
    k_scan_small(uint32_t* matrix, uint32_t m, SortPlan sp, uint32_t* __restrict__ slice_prefix,
                 uint32_t* __restrict__ counts) {
  __shared__ uint32_t sh[SCAN_SMALL_THREADS / 64];
  extern __shared__ uint32_t cnt[];  // nc + 1
  uint32_t carry = 0;
  for (uint32_t at = 0; at < m; at += 4 * SCAN_SMALL_THREADS) {
    const uint32_t base = at + threadIdx.x * 4;
    uint32_t v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = base + k < m ? matrix[base + k] : 0;
    uint32_t total;
    uint32_t pre = carry + block_exclusive_scan<SCAN_SMALL_THREADS>(v[0] + v[1] + v[2] + v[3], sh, &total);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (base + k < m) matrix[base + k] = pre;
      pre += v[k];
    }
    carry += total;
  }
  __syncthreads();
  seg_plan<SCAN_SMALL_THREADS>(matrix, sp, slice_prefix, counts, cnt, sh);
}

struct SegSlice {
  uint32_t cb, lo, hi;  // segment and entry range [lo, hi)
  bool single;          // the segment is one slice
};

__device__ __forceinline__ bool seg_slice(const uint32_t* offsets, const uint32_t* slice_prefix, const SortPlan& sp,
                                          SegSlice* out) {
  const uint32_t b = blockIdx.x;
  if (b >= slice_prefix[sp.nc]) return false;
  const uint32_t cb = find_segment(slice_prefix, sp.nc, b);
  const uint32_t start = seg_begin(offsets, sp, cb), end = seg_begin(offsets, sp, cb + 1);
  const uint32_t j = b - slice_prefix[cb];
  out->cb = cb;
  out->lo = start + j * SEG_SLICE;
  out->hi = out->lo + SEG_SLICE < end ? out->lo + SEG_SLICE : end;
  out->single = slice_prefix[cb + 1] - slice_prefix[cb] == 1;
  return true;
}

// ghist[cb * nb + bin] (zeroed beforehand) = entries of the segment in each
// bucket, for the segments of several slices.
__global__ void __launch_bounds__(THREADS)
    k_seg_hist(const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ offsets,
               const uint32_t* __restrict__ slice_prefix, SortPlan sp, uint32_t* __restrict__ ghist) {
  extern __shared__ uint32_t h[];  // nb
  SegSlice sl;
  if (!seg_slice(offsets, slice_prefix, sp, &sl) || sl.single) return;  // uniform per block
  const uint32_t nb = 1u << sp.low_bits, mask = nb - 1;
  for (uint32_t b = threadIdx.x; b < nb; b += THREADS) h[b] = 0;
  __syncthreads();
  for (uint32_t e = sl.lo + threadIdx.x; e < sl.hi; e += THREADS) atomicAdd(&h[keys_in[e] & mask], 1u);
  __syncthreads();
  uint32_t* g = ghist + (uint64_t)sl.cb * nb;
  for (uint32_t b = threadIdx.x; b < nb; b += THREADS) {
    const uint32_t c = h[b];
    if (c) atomicAdd(&g[b], c);
  }
}

// Per segment of several slices: ghist becomes the scatter cursor, the first
// entry of each bucket.
__global__ void __launch_bounds__(THREADS)
    k_seg_scan(const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ slice_prefix, SortPlan sp,
               uint32_t* __restrict__ ghist) {
  extern __shared__ uint32_t h[];  // nb
  __shared__ uint32_t sh[THREADS];
  const uint32_t nb = 1u << sp.low_bits;
  const uint32_t cb = blockIdx.x;
  if (slice_prefix[cb + 1] - slice_prefix[cb] <= 1) return;  // uniform per block
  const uint32_t start = seg_begin(offsets, sp, cb);
  uint32_t* g = ghist + (uint64_t)cb * nb;
  for (uint32_t b = threadIdx.x; b < nb; b += THREADS) h[b] = g[b];
  __syncthreads();
  lds_exclusive_scan(h, nb, sh);
  for (uint32_t b = threadIdx.x; b < nb; b += THREADS) g[b] = start + h[b];
}

// Every slice takes its run of each bucket from the cursor (one atomic per
// nonzero bucket; a one-slice segment owns the whole bucket) and moves its
// entries in one round: each thread holds its entries in registers with their
// rank inside their bucket (the value the counting atomic returned), stages
// them in bucket order in LDS, and the slice is written out so that each
// bucket's entries land as one contiguous run (coalesced stores instead of one
// scattered store per entry).  The order inside a bucket is not kept.
__global__ void __launch_bounds__(THREADS)
    k_seg_scatter(const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
                  const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ slice_prefix, SortPlan sp,
                  uint32_t* __restrict__ cursor, uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
  extern __shared__ uint32_t h[];  // cnt, lbase, gcur (nb each), then the staged keys and values
  __shared__ uint32_t sh[THREADS];
  SegSlice sl;
  if (!seg_slice(offsets, slice_prefix, sp, &sl)) return;  // uniform per block
  const uint32_t nb = 1u << sp.low_bits, mask = nb - 1;
  uint32_t* cnt = h;
  uint32_t* lbase = h + nb;
  uint32_t* gcur = h + 2 * nb;
  uint32_t* skey = h + 3 * nb;
  uint32_t* sval = skey + SEG_SLICE;
  for (uint32_t b = threadIdx.x; b < nb; b += THREADS) cnt[b] = 0;
  __syncthreads();
  uint32_t key[SEG_PER_THREAD], val[SEG_PER_THREAD], rank[SEG_PER_THREAD];
#pragma unroll
  for (uint32_t k = 0; k < SEG_PER_THREAD; k++) {
    const uint32_t e = sl.lo + k * THREADS + threadIdx.x;
    if (e < sl.hi) {
      key[k] = keys_in[e];
      val[k] = vals_in[e];
      rank[k] = atomicAdd(&cnt[key[k] & mask], 1u);
    }
  }
  __syncthreads();
  uint32_t* cur = cursor + (uint64_t)sl.cb * nb;
  for (uint32_t b = threadIdx.x; b < nb; b += THREADS) {
    const uint32_t c = cnt[b];
    if (!sl.single) gcur[b] = c ? atomicAdd(&cur[b], c) : 0u;
    lbase[b] = c;
  }
  __syncthreads();
  lds_exclusive_scan(lbase, nb, sh);
  if (sl.single)
    for (uint32_t b = threadIdx.x; b < nb; b += THREADS) gcur[b] = sl.lo + lbase[b];
#pragma unroll
  for (uint32_t k = 0; k < SEG_PER_THREAD; k++) {
    const uint32_t e = sl.lo + k * THREADS + threadIdx.x;
    if (e < sl.hi) {
      const uint32_t slot = lbase[key[k] & mask] + rank[k];
      skey[slot] = key[k];
      sval[slot] = val[k];
    }
  }
  __syncthreads();
  const uint32_t n = sl.hi - sl.lo;
  for (uint32_t slot = threadIdx.x; slot < n; slot += THREADS) {
    const uint32_t k = skey[slot];
    const uint32_t b = k & mask;
    const uint32_t dst = gcur[b] + (slot - lbase[b]);
    keys_out[dst] = k;
    vals_out[dst] = sval[slot];
  }
}

// Dynamic LDS of k_seg_scatter for 2^low_bits buckets per segment.
static inline uint32_t seg_scatter_lds(uint32_t low_bits) { return (3u * (1u << low_bits) + 2u * SEG_SLICE) * 4u; }

// ---------------------------------------------------------------- accumulation

// Closes a bucket: every bucket is completed exactly once (by one chunk, by
// its run's thread or by the piece tree), and the set it goes to was filled
// with the identity, so the sum is stored; an identity sum needs no store.
__device__ __forceinline__ void quad_close(u32* buckets, uint32_t key, const Quad29& sum, uint32_t q) {
  if (!sum.is_identity()) sum.store(buckets + (size_t)key * 32, q);
}

__device__ __forceinline__ Affine29 fetch_point(const u32* __restrict__ points, uint32_t v) {
  return Affine29::load(points + (size_t)(v & 0x7fffffffu) * 16, (v & 0x80000000u) != 0);
}

__device__ __forceinline__ uint32_t chunks_of(uint32_t entries, uint32_t ch) {
  return entries / ch + (entries % ch != 0);
}

// Thread t owns sorted entries [t * ch, ...) (key, point index | sign << 31) and
// sums each run of equal keys, one entry per loop step in every lane (a wave
// takes ch steps whatever the run lengths).  A run closed on both sides goes to
// its bucket; a run that continues from the previous chunk leaves its sum in
// piece slot 2t, another one that continues into the next chunk in slot 2t + 1.
// Nothing else is written: which slots hold a piece follows from the keys at
// the chunk edges.
// 109 VGPRs let four waves share a SIMD, which covers the dependent loads of an
// entry (key, point index, point): 2^20 points at window 16 take 1.27 ms, 88 %
// VALUBusy; with the doubling inlined a second time (three waves) it was 8 % more.
template <bool QUAD>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(3)))
    k_accumulate(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals,
                 const u32* __restrict__ points, uint32_t* counts, uint32_t ch, u32* buckets,
                 u32* __restrict__ pieces) {
  const uint32_t N = counts[0];
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t t = QUAD ? gid >> 2 : gid, q = gid & 3;
  if (gid == 0) counts[1] = 0;  // k_close_runs raises it
  if (t >= chunks_of(N, ch)) return;
  const uint32_t start = t * ch;
  const uint32_t end = N - start > ch ? start + ch : N;
  const bool open_left = start > 0 && keys[start - 1] == keys[start];
  const bool open_right = end < N && keys[end] == keys[end - 1];
  typename std::conditional<QUAD, Quad29, G1X29>::type acc;
  acc = acc.identity();
  auto put = [&](u32* p) {
    if constexpr (QUAD)
      acc.store(p, q);
    else
      acc.store(p);
  };
  bool first = true;  // still in the chunk's first run
  uint4 k4, v4;  // the next entries: a 16-byte load of each array per four steps
  uint32_t next_key = keys[start];
  for (uint32_t i = start; i < end; i++) {
    if (((i - start) & 3) == 0) {  // the arrays end on a 16-byte word
      k4 = *reinterpret_cast<const uint4*>(keys + i);
      v4 = *reinterpret_cast<const uint4*>(vals + i);
    }
    const uint32_t key = next_key, val = v4.x;
    v4 = make_uint4(v4.y, v4.z, v4.w, 0);
    k4 = make_uint4(k4.y, k4.z, k4.w, 0);
    const bool last = i + 1 == end;
    next_key = last ? ~key : ((i - start) & 3) == 3 ? keys[i + 1] : k4.x;
    if constexpr (QUAD) {
      u32 w[8];
      Fq29::load_words(points + (size_t)(val & 0x7fffffffu) * 16 + 8 * (q & 1), w);
      u32 any = 0;
#pragma unroll
      for (int j = 0; j < 8; j++) any |= w[j];
      any |= quad_perm<1, 0, 3, 2>(any);  // (0, 0) is the identity
      Fq29 xy = Fq29::from_words<5>(w);
      xy = lane_pick((q & 1) != 0 && (val & 0x80000000u) != 0, Fq29::zero().sub<32>(xy), xy);
      acc = acc.add_affine(xy, any == 0, q);
    } else {
      acc = acc.add_affine(fetch_point(points, val));
    }
    if (next_key != key) {
      if (first && open_left)
        put(pieces + (size_t)(2 * t) * 32);
      else if (last && open_right)
        put(pieces + (size_t)(2 * t + 1) * 32);
      else if (!acc.is_identity())
        put(buckets + (size_t)key * 32);
      acc = acc.identity();
      first = false;
    }
  }
}

// A run cut by chunk edges has pieces 2t + 1 (it starts in chunk t), 2(t + 1),
// 2(t + 2), ...  One thread (QUAD: one quad of lanes) per chunk edge
// adds the pieces of the run that starts left of it and closes the bucket.
// With scalars spread over the buckets nearly every edge starts a run of two
// to a few pieces, so the lanes of a wave stay busy.  A run of more than
// RUN_MAX pieces after its first is left to k_long_tiles, and counts[1] says so.
constexpr uint32_t RUN_MAX = 16;

template <bool QUAD>
__global__ void __launch_bounds__(THREADS)
    k_close_runs(const uint32_t* __restrict__ keys, const u32* __restrict__ pieces, uint32_t* counts, uint32_t ch,
                 u32* buckets) {
  const uint32_t N = counts[0];
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t t = QUAD ? gid >> 2 : gid, q = gid & 3;
  const uint32_t nchunks = chunks_of(N, ch);
  if (t + 1 >= nchunks) return;
  const uint32_t key = keys[t * ch + ch - 1];
  if (keys[(t + 1) * ch] != key) return;                                   // no run crosses this edge
  if (t > 0 && keys[t * ch] == key && keys[t * ch - 1] == key) return;  // it started further left
  if (t + 1 + RUN_MAX < nchunks && keys[(t + 1 + RUN_MAX) * ch] == key) {
    counts[1] = 1;
    return;
  }
  // pieces after the first: 1 .. RUN_MAX, the chunks from t + 1 on that start with the key
  uint32_t n = 1, above = RUN_MAX + 1;
  if (t + 2 >= nchunks || keys[(t + 2) * ch] != key) above = 2;
  while (above - n > 1) {
    const uint32_t mid = (n + above) >> 1;
    if (t + mid < nchunks && keys[(t + mid) * ch] == key)
      n = mid;
    else
      above = mid;
  }
  const u32* base = pieces + (size_t)(2 * t + 1) * 32;  // piece k > 0 is k * 64 - 32 words on
  if constexpr (QUAD) {
    Quad29 acc = Quad29::load(base, q), p = Quad29::load(base + 32, q);
    for (uint32_t k = 1;; k++) {
      // the next piece crosses from memory during this addition
      const Quad29 next = k < n ? Quad29::load(base + 32 + (size_t)k * 64, q) : p;
      acc = acc.add(p, q);
      if (k >= n) break;
      p = next;
    }
    quad_close(buckets, key, acc, q);
  } else {
    G1X29 acc = G1X29::load(base), p = G1X29::load(base + 32);
    for (uint32_t k = 1;; k++) {
      const G1X29 next = k < n ? G1X29::load(base + 32 + (size_t)k * 64) : p;
      acc = acc.add(p);
      if (k >= n) break;
      p = next;
    }
    if (!acc.is_identity()) acc.store(buckets + (size_t)key * 32);
  }
}

// ---- the pieces of long runs: a segmented sum over all pieces in order ----
//
// A segment of the piece sequence is its first run's key and sum, and, when it
// holds several runs, its last run's key and sum; the runs between are complete
// and closed.  Every quad of lanes walks a share of the pieces, the 64 quads of
// a workgroup join their segments in LDS as a tree, k_long_tiles leaves one
// segment per workgroup and k_long_join joins those.  So a run of any length
// costs (its pieces / 64 / LONG_TILES) + about 30 additions in sequence.
// Up to LONG_TILES workgroups, one chunk a quad where that takes fewer.
constexpr uint32_t LONG_QUADS = THREADS / 4;
constexpr uint32_t LONG_TILES = 512;
static inline uint32_t long_tiles_for(uint32_t chunks) {
  const uint32_t t = (chunks + LONG_QUADS - 1) / LONG_QUADS;
  return t < LONG_TILES ? t : LONG_TILES;
}

enum : uint32_t { SEG_EMPTY = 0, SEG_ONE = 1, SEG_SEVERAL = 2 };  // runs in a segment: none, one, more

struct SegmentLds {
  Quad29 first[LONG_QUADS][4], last[LONG_QUADS][4];  // [quad][lane]
  uint32_t key_first[LONG_QUADS], key_last[LONG_QUADS], runs[LONG_QUADS];
};

// The walk of one quad: pieces in order, each joined to the run before it.
struct SegmentWalk {
  uint32_t key_first = 0, key = 0, runs = SEG_EMPTY;
  Quad29 sum;

  __device__ __forceinline__ void piece(SegmentLds& S, uint32_t quad, uint32_t q, u32* buckets, uint32_t k,
                                        const Quad29& p) {
    if (runs != SEG_EMPTY && k == key) {
      sum = sum.add(p, q);
      return;
    }
    if (runs == SEG_EMPTY) {
      key_first = k;
      runs = SEG_ONE;
    } else {
      if (runs == SEG_ONE)
        S.first[quad][q] = sum;
      else
        quad_close(buckets, key, sum, q);
      runs = SEG_SEVERAL;
    }
    key = k;
    sum = p;
  }
  __device__ __forceinline__ void finish(SegmentLds& S, uint32_t quad, uint32_t q) const {
    if (runs == SEG_ONE) S.first[quad][q] = sum;
    if (runs == SEG_SEVERAL) S.last[quad][q] = sum;
    if (q != 0) return;
    S.runs[quad] = runs;
    S.key_first[quad] = key_first;
    S.key_last[quad] = key;
  }
};

// Joins the quads' segments into quad 0's (whole workgroup).  Every value a
// quad reads before it writes is its own or that of the quad it takes in.
__device__ __forceinline__ void join_segments(SegmentLds& S, uint32_t quad, uint32_t q, u32* buckets) {
  for (uint32_t step = 1; step < LONG_QUADS; step <<= 1) {
    __syncthreads();
    if (quad & (2 * step - 1)) continue;
    const uint32_t r = quad + step;
    const uint32_t lruns = S.runs[quad], rruns = S.runs[r];
    if (rruns == SEG_EMPTY) continue;
    const uint32_t lkey = S.key_last[quad], rkey = S.key_first[r];
    const Quad29 f = S.first[r][q];
    uint32_t runs = SEG_SEVERAL;
    if (lruns == SEG_EMPTY) {
      S.first[quad][q] = f;
      runs = rruns;
      if (q == 0) S.key_first[quad] = rkey;
    } else {
      const Quad29 l = lruns == SEG_ONE ? S.first[quad][q] : S.last[quad][q];
      if (lkey == rkey) {
        const Quad29 s = l.add(f, q);
        if (lruns == SEG_ONE)
          S.first[quad][q] = s;
        else if (rruns == SEG_ONE)
          S.last[quad][q] = s;
        else
          quad_close(buckets, lkey, s, q);
        if (lruns == SEG_ONE && rruns == SEG_ONE) runs = SEG_ONE;
      } else {
        if (lruns == SEG_SEVERAL) quad_close(buckets, lkey, l, q);
        if (rruns == SEG_SEVERAL)
          quad_close(buckets, rkey, f, q);
        else
          S.last[quad][q] = f;
      }
    }
    if (rruns == SEG_SEVERAL) S.last[quad][q] = S.last[r][q];
    if (q == 0) {
      S.runs[quad] = runs;
      S.key_last[quad] = S.key_last[r];
    }
  }
  __syncthreads();
}

// One workgroup's share of the chunks; its segment goes to seg_pts[2b], [2b + 1]
// and seg_meta[3b ..] (runs, first key, last key).  Only the pieces of long
// runs count: the others were closed by k_close_runs.
__global__ void __launch_bounds__(THREADS)
    k_long_tiles(const uint32_t* __restrict__ keys, const u32* __restrict__ pieces,
                 const uint32_t* __restrict__ counts, uint32_t ch, u32* buckets, uint32_t* __restrict__ seg_meta,
                 u32* __restrict__ seg_pts) {
  if (counts[1] == 0) return;
  __shared__ SegmentLds S;
  const uint32_t N = counts[0];
  const uint32_t nchunks = chunks_of(N, ch);
  const uint32_t quad = threadIdx.x >> 2, q = threadIdx.x & 3;
  const uint32_t per = (nchunks + gridDim.x * LONG_QUADS - 1) / (gridDim.x * LONG_QUADS);
  const uint32_t lo = (blockIdx.x * LONG_QUADS + quad) * per;
  const uint32_t hi = lo + per < nchunks ? lo + per : nchunks;
  SegmentWalk w;
  for (uint32_t base = lo; base < hi; base += 4) {
    // four chunks at a time, their keys looked at by one lane each: bit 0, slot
    // 2u holds a piece of a long run; bit 1, slot 2u + 1 does
    const uint32_t u0 = base + q;
    uint32_t mine = 0, kf = 0, kl = 0;
    if (u0 < hi) {
      kf = keys[u0 * ch];
      kl = keys[u0 + 1 < nchunks ? u0 * ch + ch - 1 : N - 1];
      const bool open_left = u0 > 0 && keys[u0 * ch - 1] == kf;
      if (open_left) {
        // c: the first chunk, within RUN_MAX + 1 before u0, that starts with the
        // run's key; the run starts there or in the chunk before, and is long
        // when the chunk RUN_MAX + 1 after its start still holds it
        uint32_t below = u0 > RUN_MAX + 1 ? u0 - RUN_MAX - 2 : ~0u, c = u0;  // chunk `below` is not looked at
        while (c - below > 1) {
          const uint32_t mid = below + ((c - below) >> 1);
          if (keys[mid * ch] == kf)
            c = mid;
          else
            below = mid;
        }
        const uint32_t t = c > 0 && keys[c * ch - 1] == kf ? c - 1 : c;
        if (u0 - t > RUN_MAX || (t + 1 + RUN_MAX < nchunks && keys[(t + 1 + RUN_MAX) * ch] == kf)) mine = 1;
      }
      // (a chunk that is all the run of slot 2u has nothing in slot 2u + 1)
      if (!(open_left && kl == kf) && u0 + 1 + RUN_MAX < nchunks && keys[(u0 + 1) * ch] == kl &&
          keys[(u0 + 1 + RUN_MAX) * ch] == kl)
        mine |= 2;
    }
    const uint32_t lane0 = __lane_id() & ~3u;
    for (uint32_t j = 0; j < 8; j++) {
      const int from = (int)(lane0 + (j >> 1));
      const uint32_t bits = __shfl(mine, from);
      const uint32_t key_f = __shfl(kf, from), key_l = __shfl(kl, from);
      if ((bits >> (j & 1)) & 1)
        w.piece(S, quad, q, buckets, (j & 1) ? key_l : key_f,
                Quad29::load(pieces + (size_t)(2 * (base + (j >> 1)) + (j & 1)) * 32, q));
    }
  }
  w.finish(S, quad, q);
  join_segments(S, quad, q, buckets);
  if (quad == 0) {
    uint32_t* m = seg_meta + 3 * blockIdx.x;
    if (q == 0) {
      m[0] = S.runs[0];
      m[1] = S.key_first[0];
      m[2] = S.key_last[0];
    }
    if (S.runs[0] != SEG_EMPTY) S.first[0][q].store(seg_pts + (size_t)(2 * blockIdx.x) * 32, q);
    if (S.runs[0] == SEG_SEVERAL) S.last[0][q].store(seg_pts + (size_t)(2 * blockIdx.x + 1) * 32, q);
  }
}

// The tiles' segments joined (one workgroup); the last runs are closed.
__global__ void __launch_bounds__(THREADS)
    k_long_join(const uint32_t* __restrict__ counts, const uint32_t* __restrict__ seg_meta,
                const u32* __restrict__ seg_pts, uint32_t tiles, u32* buckets) {
  if (counts[1] == 0) return;
  __shared__ SegmentLds S;
  const uint32_t quad = threadIdx.x >> 2, q = threadIdx.x & 3;
  SegmentWalk w;
  constexpr uint32_t per = 2 * LONG_TILES / LONG_QUADS;  // a constant: the meta loads go out together
  for (uint32_t v = quad * per; v < (quad + 1) * per; v++) {
    const uint32_t b = v >> 1;
    if (b < tiles && seg_meta[3 * b] > (v & 1))
      w.piece(S, quad, q, buckets, seg_meta[3 * b + 1 + (v & 1)], Quad29::load(seg_pts + (size_t)v * 32, q));
  }
  w.finish(S, quad, q);
  join_segments(S, quad, q, buckets);
  if (quad == 0) {
    if (S.runs[0] != SEG_EMPTY) quad_close(buckets, S.key_first[0], S.first[0][q], q);
    if (S.runs[0] == SEG_SEVERAL) quad_close(buckets, S.key_last[0], S.last[0][q], q);
  }
}

__global__ void __launch_bounds__(THREADS) k_zero_u32(uint32_t* p, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0;
}

__global__ void __launch_bounds__(THREADS) k_fill_identity(u32* pts, uint64_t count) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint4 z = make_uint4(0, 0, 0, 0);
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count * 8; i += stride)
    reinterpret_cast<uint4*>(pts)[i] = z;
}

// dst[0, n16) = src[0, n16) in 16-byte words, src being pinned host memory
// mapped into the device's address space: the host-to-device copies of the
// drop-in msm's points and scalars.  A grid of PULL_BLOCKS workgroups with four
// loads in flight per lane keeps the PCIe link full (57 GB/s measured on
// MI355X for 64 MiB, the link's rate) on a small share of the CUs, so the
// compute stream's sort runs beside it.  DMA copies reach the same rate on some
// copy engines and about half of it on others, and which engine serves a stream
// depends on what the process did before (a one-part 2^20 call took 3.8 ms or
// 4.9 ms that way); the kernel's rate does not.
constexpr uint32_t PULL_BLOCKS = 64;
constexpr int PULL_UNROLL = 4;
__global__ void __launch_bounds__(THREADS) k_pull_host(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                       uint64_t n16) {
  const uint64_t stride = (uint64_t)gridDim.x * THREADS * PULL_UNROLL;
  for (uint64_t base = (uint64_t)blockIdx.x * THREADS * PULL_UNROLL + threadIdx.x; base < n16; base += stride) {
    uint4 v[PULL_UNROLL];
#pragma unroll
    for (int u = 0; u < PULL_UNROLL; u++) {
      const uint64_t i = base + (uint64_t)u * THREADS;
      if (i < n16) v[u] = src[i];
    }
#pragma unroll
    for (int u = 0; u < PULL_UNROLL; u++) {
      const uint64_t i = base + (uint64_t)u * THREADS;
      if (i < n16) dst[i] = v[u];
    }
  }
}

// dst[i] += src[i] over H buckets (XYZZ): a later part's buckets, accumulated
// into a scratch set of their own, join the batch's buckets in one pass with
// no divergence, instead of every run of that part reading and adding its
// bucket inside the accumulation loop.
__global__ void __launch_bounds__(THREADS) k_merge_buckets(u32* __restrict__ dst, const u32* __restrict__ src,
                                                           uint32_t H) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= H) return;
  const G1X29 b = G1X29::load(src + (size_t)i * 32);
  if (b.is_identity()) return;
  u32* d = dst + (size_t)i * 32;
  const G1X29 a = G1X29::load(d);
  (a.is_identity() ? b : a.add(b)).store(d);
}

__global__ void k_set_count(uint32_t* counts, const uint32_t* offsets, uint32_t h) {
  if (threadIdx.x == 0 && blockIdx.x == 0) counts[0] = offsets[h];
}

// ---------------------------------------------------------------- bucket reduction
//
// Per window: S = sum_j j X_j + sum_j Y_j over j < M (M a power of two).  A
// halving level maps the pair (2i, 2i + 1) to
//   X'_i = 2 (X_2i + X_2i+1),   Y'_i = X_2i+1 + Y_2i + Y_2i+1,
// which keeps S = sum_i i X'_i + sum_i Y'_i over M / 2 items; at M = 1,
// S = Y_0.  Level 0 has X = Y = buckets, bucket b at j = b - 1, which makes
// S = sum_b b B_b.  X' and Y' are computed by different threads (different
// waves), so a level is two point operations deep.
// The top window's first top_log levels only fold its buckets' copies,
// X'_i = X_2i + X_2i+1 and Y'_i = Y_2i + Y_2i+1, which leaves
// S = sum_i i X'_i + sum_i Y'_i with one item per digit.

// The first two levels at once, one thread per block of four buckets
// B_0..B_3 (items 4i..4i+3 of a window): X'' = 4T with T = B_0 + .. + B_3, and
// Y'' = B_0 + 2B_1 + 3B_2 + 4B_3 = T + s_1 + s_2 + s_3 with the suffix sums
// s_r = B_r + .. + B_3, so that S = sum_i i X''_i + sum_i Y''_i over M / 4
// items.  Six additions and two doublings (102 products) per four buckets,
// where two halving levels take 51 products per pair, 153 per four buckets.
__global__ void __launch_bounds__(THREADS)
    k_reduce_block4(const u32* __restrict__ B, uint32_t M, uint32_t n_windows, uint32_t fold_top, u32* __restrict__ Xo,
                    u32* __restrict__ Yo) {
  const uint32_t blocks = (M >> 2) * n_windows;
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= blocks) return;
  // folding levels of this window: both, X'' = Y'' = T; the first, X'' = 2T and Y'' = T + s_2
  const uint32_t fold = gid / (M >> 2) == n_windows - 1 ? fold_top : 0;
  const size_t j0 = (size_t)gid * 4;  // windows are consecutive runs of M items: block gid covers 4 gid..4 gid+3
  // s = s_3, s_2, s_1, s_0 = T and y their sum, one addition per loop step so
  // that one copy of its code serves them all; then two doublings of T.
  G1X29 s = G1X29::load(B + (j0 + 3) * 32);
  G1X29 y = s;
#pragma unroll 1
  for (int step = 0; step < 8; step++) {
    const bool to_s = !(step & 1);
    if (fold >= 2 && (!to_s || step >= 6)) continue;
    if (fold == 1) {
      if (step == 1) y = s;
      if (step == 1 || step == 3 || step == 7) continue;
    }
    const G1X29 a = to_s ? s : y;
    G1X29 b = s;
    if (to_s && step < 6) b = G1X29::load(B + (j0 + 2 - (step >> 1)) * 32);
    const G1X29 r = step < 6 ? a.add(b) : s.dbl();
    if (to_s || step >= 6)
      s = r;
    else
      y = r;
    if (step == 5) y.store(Yo + (size_t)gid * 32);
  }
  if (fold >= 2) s.store(Yo + (size_t)gid * 32);
  s.store(Xo + (size_t)gid * 32);
}

// One level over all windows: threads [0, Mo * n_windows) write X', the next
// Mo * n_windows threads write Y' (Mo = M / 2).
__global__ void __launch_bounds__(THREADS)
    k_reduce_level(const u32* __restrict__ X, const u32* __restrict__ Y, uint32_t M, uint32_t n_windows,
                   bool first, bool fold_top, u32* __restrict__ Xo, u32* __restrict__ Yo) {
  const uint32_t Mo = M >> 1;
  const uint32_t items = Mo * n_windows;
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= 2 * items) return;
  const bool yside = gid >= items;
  const uint32_t it = yside ? gid - items : gid;
  const size_t j0 = (size_t)(it / Mo) * M + 2 * (it % Mo);
  const u32* src = yside && !first ? Y : X;
  const G1X29 x1 = G1X29::load(X + (j0 + 1) * 32);
  G1X29 r = G1X29::load(src + j0 * 32);
  G1X29 o = G1X29::load(src + (j0 + 1) * 32);
  const int steps = fold_top && it / Mo == n_windows - 1 ? 1 : 2;
#pragma unroll 1
  for (int step = 0; step < steps; step++) {  // one copy of the addition; X' doubles through it
    r = r.add(o);
    o = yside ? x1 : r;
  }
  r.store((yside ? Yo : Xo) + (size_t)it * 32);
}

// The same level with a quad of lanes per point operation (Quad29): for the narrow levels, where the operations are few and each
// one's latency, not the throughput, sets the time.
__global__ void __launch_bounds__(THREADS)
    k_reduce_level_quad(const u32* __restrict__ X, const u32* __restrict__ Y, uint32_t M, uint32_t n_windows,
                        bool first, bool fold_top, u32* __restrict__ Xo, u32* __restrict__ Yo) {
  const uint32_t Mo = M >> 1;
  const uint32_t items = Mo * n_windows;
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t op = gid >> 2, q = gid & 3;
  if (op >= 2 * items) return;  // whole quads: 2 * items * 4 threads are launched in multiples of 4
  const bool yside = op >= items;
  const uint32_t it = yside ? op - items : op;
  const size_t j0 = (size_t)(it / Mo) * M + 2 * (it % Mo);
  const u32* src = yside && !first ? Y : X;
  const Quad29 x1 = Quad29::load(X + (j0 + 1) * 32, q);
  Quad29 r = Quad29::load(src + j0 * 32, q);
  Quad29 o = Quad29::load(src + (j0 + 1) * 32, q);
  const int steps = fold_top && it / Mo == n_windows - 1 ? 1 : 2;
#pragma unroll 1
  for (int step = 0; step < steps; step++) {
    r = r.add(o, q);
    o = yside ? x1 : r;
  }
  r.store((yside ? Yo : Xo) + (size_t)it * 32, q);
}

// The last levels of window blockIdx.x (M <= RED_TAIL items) in LDS, all in
// one launch, a quad of lanes per point operation; out[w] = S_w.  fold_top: how
// many of the levels fold the top window's copies.  The X' quads of a level of
// P items come first and the Y' quads from the next wave on, so that the two
// waves of the narrow levels run on two SIMDs (waves 0 and 4 of a workgroup
// would share one).
constexpr uint32_t QUAD_TAIL_THREADS = 4 * RED_TAIL;
__global__ void __launch_bounds__(QUAD_TAIL_THREADS)
    k_reduce_tail_quad(const u32* __restrict__ X, const u32* __restrict__ Y, uint32_t M, bool first,
                       uint32_t fold_top, u32* __restrict__ out) {
  __shared__ Quad29 sh[2][RED_TAIL][4];  // X, Y; [item][lane]
  const size_t base = (size_t)blockIdx.x * M;
  const uint32_t op = threadIdx.x >> 2, q = threadIdx.x & 3;
  if (op < M) {
    sh[0][op][q] = Quad29::load(X + (base + op) * 32, q);
    sh[1][op][q] = Quad29::load((first ? X : Y) + (base + op) * 32, q);
  }
  __syncthreads();
  uint32_t fold = blockIdx.x + 1 == gridDim.x ? fold_top : 0;
  for (uint32_t P = M >> 1; P >= 1; P >>= 1) {
    const uint32_t y0 = P < 16 ? 16 : P;  // first Y' quad
    const uint32_t side = op >= y0 ? 1 : 0;
    const uint32_t i = op - (side ? y0 : 0);
    const bool act = i < P;  // the same for the four lanes of a quad
    const int steps = fold > 0 ? 1 : 2;
    if (fold > 0) fold--;
    Quad29 r, o;
    if (act) {
      r = sh[side][2 * i][q];
      o = sh[side][2 * i + 1][q];
#pragma unroll 1
      for (int step = 0; step < steps; step++) {  // X' doubles through the addition
        r = r.add(o, q);
        o = r;
        if (side) o = sh[0][2 * i + 1][q];
      }
    }
    __syncthreads();
    if (act) sh[side][i][q] = r;
    __syncthreads();
  }
  // The host reads G1XYZZ: a coordinate per lane (were the value uniform the
  // compiler would take its products to the scalar unit, 12 us of them).
  if (threadIdx.x < 4) {
    u32 w[8];
    sh[1][0][q].c.to_mont256(w);
    Fq::from_raw(w).store(out + (size_t)blockIdx.x * 32 + 8 * q);
  }
}

// ---------------------------------------------------------------- precompute

// table j (1 <= j < n_precompute) of point i = 2^(j * shift) * P_i, affine
__global__ void __launch_bounds__(THREADS)
    k_precompute(u32* points, uint64_t len, uint32_t n_precompute, uint32_t shift) {
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= len) return;
  G1XYZZ p = G1XYZZ::from_affine(G1Affine::load(points + gid * 16));
  for (uint32_t j = 1; j < n_precompute; j++) {
    for (uint32_t k = 0; k < shift; k++) p = p.dbl();
    p.to_affine().store(points + (gid + j * len) * 16);
  }
}

// out[i] = k_i * G for G = (1, 2), k_i given as Fr Montgomery-form elements;
// double-and-add over the canonical bits, affine output.
__global__ void __launch_bounds__(THREADS)
    k_mul_generator(const u32* __restrict__ scalars, uint64_t n, u32* __restrict__ out) {
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= n) return;
  const Fr k = Fr::load(scalars + gid * 8).to_canonical();
  Fq one = Fq::one();
  const G1Affine g{one, one + one};
  G1XYZZ acc = G1XYZZ::identity();
  for (int bit = 253; bit >= 0; bit--) {
    acc = acc.dbl();
    if ((k.v[bit >> 5] >> (bit & 31)) & 1) acc = acc.add_affine(g);
  }
  acc.to_affine().store(out + gid * 16);
}

// ---------------------------------------------------------------- host orchestration

static inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Device workspace for one MSM of `len` points (per table) and config cfg.
// The pieces of cut runs live in the accumulation only, the sort's temporaries
// (matrix, keys_tmp, vals_tmp, slices) before it and the reduction's levels (red)
// after it, all on one stream, so the pieces lie over the other two.
struct Layout {
  size_t hist, block_sums, cursor, keys0, vals0, counts, pieces, seg_meta, seg_pts, buckets, red[4], sums;
  size_t least, total;  // smallest workspace that does, and the one to ask for
  size_t matrix, keys_tmp, vals_tmp, slices;  // partition sort (when `part`)
  uint32_t max_slices;
  bool part;
  SortPlan sp;
  uint64_t matrix_n;  // nc * tiles + 1
  uint32_t nb_matrix;
  uint32_t H, nb_scan;
  uint64_t n_entries_max;
  Share share;          // how the accumulation is shared out
  uint32_t chunks_max;  // accumulating threads or quads
  uint32_t red_m[MAX_LEVELS];
  int red_levels;  // one-level launches before the in-workgroup tail
  size_t bucket_bytes;  // one bucket set (n_windows * 2^(s-1) XYZZ points)
  uint32_t sets;        // bucket sets from `buckets` on (one per batch of a run)
};

// Partition-sort parameters for `len` points; false when the window is too wide
// for the LDS tables (then the atomic counting sort runs instead).
constexpr uint32_t PART_LDS_MAX = 96 * 1024;
static bool make_sort_plan(const Config& cfg, uint64_t len, SortPlan* sp) {
  const uint32_t bits = cfg.s - 1;  // bucket bits
  uint32_t cb = bits < 5 ? bits : 5;
  uint32_t low = bits - cb;
  if (low > 12) {
    low = 12;
    cb = bits - 12;
  }
  if (cb > 7) return false;  // windows above 20 bits
  sp->low_bits = low;
  sp->nc = cfg.n_windows << cb;
  uint32_t tp = 1024;
  while (tp > 64 && (2ull * sp->nc + 2ull * tp * cfg.actual_windows) * 4 > PART_LDS_MAX) tp >>= 1;
  if ((2ull * sp->nc + 2ull * tp * cfg.actual_windows) * 4 > PART_LDS_MAX) return false;
  sp->tp = tp;
  sp->tiles = (uint32_t)((len + tp - 1) / tp);
  sp->lds_part = (uint32_t)((2ull * sp->nc + 2ull * tp * cfg.actual_windows) * 4);
  return sp->tiles > 0;
}

// Room for pieces beyond the sort's and the reduction's.  The least workspace of a
// length may not grow from one version to the next (a saved plan's buffer has to
// do), nor be smaller than a shorter length's: the first accumulation kept 10.3
// bytes an entry for itself, and the first one with pieces, which lay apart, no
// less than 24 MB from 2.4 M entries on.  Chunks of sixteen entries take 16 bytes
// of pieces an entry and fit there.  The shorter ones of small MSMs, down to four
// entries (65 bytes an entry, at most 10 240 chunks), do not where the reduction has
// no levels, so the size asked for has room for them, and a smaller buffer gets
// longer chunks: 2^10 points, window 8, 250 us, and 281 us in the least workspace.
constexpr uint64_t PIECE_BYTES_PER_ENTRY = 10, PIECE_BYTES_MAX = 24000000;
constexpr uint64_t SHORT_CHUNK_BYTES_PER_ENTRY = 68, SHORT_CHUNK_BYTES_MAX = 2750000;

// The layout in `room` bytes of workspace, at least L->least, at most L->total:
// chunks are as long as room for their pieces asks.
static bool make_layout(const Config& cfg, uint64_t len, Layout* L, uint32_t sets, uint64_t room) {
  memset(L, 0, sizeof(*L));
  if (sets == 0) return false;
  L->sets = sets;
  L->H = cfg.n_windows * cfg.buckets;
  L->nb_scan = div_ceil32((uint64_t)L->H + 1, SCAN_BLOCK);
  if (L->nb_scan > THREADS * 1024) return false;
  L->part = len > 0 && make_sort_plan(cfg, len, &L->sp);
  if (L->part) {
    L->matrix_n = (uint64_t)L->sp.nc * L->sp.tiles + 1;
    if (L->matrix_n >= 0xffffffffull) return false;
    L->nb_matrix = div_ceil32(L->matrix_n, SCAN_BLOCK);
    if (L->nb_matrix > THREADS * 1024) L->part = false;
  }
  L->n_entries_max = len * cfg.actual_windows;
  if (len * cfg.n_precompute >= 0x80000000ull || L->n_entries_max >= 0xffffffffull) return false;
  // reduction level sizes (halving down to RED_TAIL items per window)
  uint32_t M = cfg.buckets;
  int rl = 0;
  uint64_t red_max0 = 0, red_max1 = 0;
  while (M > RED_TAIL) {
    if (rl >= MAX_LEVELS) return false;
    M >>= 1;
    L->red_m[rl] = M;
    if (rl % 2 == 0) red_max0 = M > red_max0 ? M : red_max0;
    else red_max1 = M > red_max1 ? M : red_max1;
    rl++;
  }
  L->red_levels = rl;
  size_t off = 0;
  L->hist = off; off = align256(off + ((size_t)L->H + 1) * 4);
  L->cursor = off; off = align256(off + ((size_t)L->H + 1) * 4);
  L->block_sums = off; off = align256(off + (size_t)(L->nb_scan > L->nb_matrix ? L->nb_scan : L->nb_matrix) * 4);
  L->counts = off; off = align256(off + 2 * 4);
  L->keys0 = off; off = align256(off + L->n_entries_max * 4);
  L->vals0 = off; off = align256(off + L->n_entries_max * 4);
  L->bucket_bytes = align256((size_t)L->H * 128);
  L->buckets = off; off += L->bucket_bytes * sets;
  L->sums = off; off = align256(off + (size_t)cfg.n_windows * 128);
  const size_t shared = off;
  if (L->part) {
    L->matrix = off; off = align256(off + (size_t)L->matrix_n * 4);
    L->keys_tmp = off; off = align256(off + L->n_entries_max * 4);
    L->vals_tmp = off; off = align256(off + L->n_entries_max * 4);
    L->slices = off; off = align256(off + ((size_t)L->sp.nc + 1) * 4);
    L->max_slices = (uint32_t)((L->n_entries_max + SEG_SLICE - 1) / SEG_SLICE) + L->sp.nc;
  }
  // reduction ping-pong: X and Y for even / odd levels
  L->red[0] = off; off = align256(off + (size_t)cfg.n_windows * red_max0 * 128);
  L->red[1] = off; off = align256(off + (size_t)cfg.n_windows * red_max0 * 128);
  L->red[2] = off; off = align256(off + (size_t)cfg.n_windows * (red_max1 ? red_max1 : 1) * 128);
  L->red[3] = off; off = align256(off + (size_t)cfg.n_windows * (red_max1 ? red_max1 : 1) * 128);
  const uint64_t least = PIECE_BYTES_PER_ENTRY * L->n_entries_max, full = SHORT_CHUNK_BYTES_PER_ENTRY * L->n_entries_max;
  L->least = align256(off + (least < PIECE_BYTES_MAX ? least : PIECE_BYTES_MAX));
  L->total = align256(off + (full < SHORT_CHUNK_BYTES_MAX ? full : SHORT_CHUNK_BYTES_MAX));
  if (L->total < L->least) L->total = L->least;
  if (room < L->least) return false;
  // chunks as share_for wants them, longer where their pieces would not fit
  L->share = share_for(L->n_entries_max);
  for (;; L->share.ch += 4) {
    L->chunks_max = (uint32_t)((L->n_entries_max + L->share.ch - 1) / L->share.ch);
    const uint32_t tiles = L->chunks_max > RUN_MAX + 1 ? long_tiles_for(L->chunks_max) : 0;
    L->pieces = shared;
    L->seg_meta = align256(L->pieces + (L->chunks_max > 1 ? (size_t)L->chunks_max * 2 * 128 : 0));
    L->seg_pts = align256(L->seg_meta + (size_t)tiles * 3 * 4);
    if (L->seg_pts + (size_t)tiles * 2 * 128 <= (room < L->total ? room : L->total)) break;
  }
  return true;
}

static inline unsigned grid_for(uint64_t work, unsigned cap) {
  uint64_t g = (work + THREADS - 1) / THREADS;
  if (g > cap) g = cap;
  return g == 0 ? 1u : (unsigned)g;
}

// The partition and segment scatters take more than 64 KB of dynamic LDS; the
// permission is set once per device, at each kernel's largest request, on the
// first MSM there (outside any graph capture a caller may start later).
static std::mutex g_attr_mu;
static bool g_attr_done[64];

static hipError_t ensure_lds_limits() {
  int dev = 0;
  ZKP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_attr_mu);
  if (g_attr_done[dev]) return hipSuccess;
  ZKP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_part_scatter),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)PART_LDS_MAX));
  ZKP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(k_seg_scatter),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)seg_scatter_lds(12)));
  g_attr_done[dev] = true;
  return hipSuccess;
}

struct PhaseTimer {
  bool on;
  hipStream_t s;
  std::vector<hipEvent_t> ev;
  std::vector<const char*> names;
  void mark(const char* name) {
    if (!on) return;
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return;
    (void)hipEventRecord(e, s);
    ev.push_back(e);
    names.push_back(name);
  }
  void report() {
    if (!on || ev.size() < 2) return;
    (void)hipEventSynchronize(ev.back());
    for (size_t i = 1; i < ev.size(); i++) {
      float ms = 0;
      (void)hipEventElapsedTime(&ms, ev[i - 1], ev[i]);
      fprintf(stderr, "[msm] %-12s %.4f ms\n", names[i], ms);
    }
    for (auto e : ev) (void)hipEventDestroy(e);
    ev.clear();
    names.clear();
  }
};

static inline u32* bucket_set(const Layout& L, char* ws, uint32_t set) {
  return reinterpret_cast<u32*>(ws + L.buckets + (size_t)set * L.bucket_bytes);
}

// Zeroes bucket set `set` (fill kernel, safe under graph capture).
static hipError_t reset_buckets(const Config& cfg, const Layout& L, char* ws, uint32_t set, hipStream_t stream) {
  hipLaunchKernelGGL(k_fill_identity, dim3(grid_for((uint64_t)L.H * 8, 16384)), dim3(THREADS), 0, stream,
                     bucket_set(L, ws, set), (uint64_t)L.H);
  return hipGetLastError();
}

// First half of a part: the signed digits of its scalars sorted by bucket into
// keys0 / vals0 (point index and sign), with the entry counts in `counts`.
// Reads only the scalars, so it can run while the part's points are still
// crossing the link.
static hipError_t sort_part(const Config& cfg, const Layout& L, char* ws, const u32* d_scalars, uint64_t len,
                            hipStream_t stream, PhaseTimer& pt) {
  ZKP_CHECK(ensure_lds_limits());
  uint32_t* hist = reinterpret_cast<uint32_t*>(ws + L.hist);
  uint32_t* cursor = reinterpret_cast<uint32_t*>(ws + L.cursor);
  uint32_t* bsums = reinterpret_cast<uint32_t*>(ws + L.block_sums);
  uint32_t* counts = reinterpret_cast<uint32_t*>(ws + L.counts);
  uint32_t* keys0 = reinterpret_cast<uint32_t*>(ws + L.keys0);
  uint32_t* vals0 = reinterpret_cast<uint32_t*>(ws + L.vals0);
  if (L.part) {
    // partition sort (no device atomics); `len` may be below the planned maximum
    SortPlan sp = L.sp;
    sp.tiles = (uint32_t)((len + sp.tp - 1) / sp.tp);
    const uint64_t mn = (uint64_t)sp.nc * sp.tiles + 1;
    uint32_t* matrix = reinterpret_cast<uint32_t*>(ws + L.matrix);
    uint32_t* ktmp = reinterpret_cast<uint32_t*>(ws + L.keys_tmp);
    uint32_t* vtmp = reinterpret_cast<uint32_t*>(ws + L.vals_tmp);
    const uint32_t nbk = 1u << sp.low_bits;
    uint32_t* slices = reinterpret_cast<uint32_t*>(ws + L.slices);
    pt.mark("start");
    hipLaunchKernelGGL(k_part_count, dim3(sp.tiles), dim3(THREADS), sp.nc * 4, stream, d_scalars, len, cfg, sp, matrix,
                       cursor);
    ZKP_CHECK(hipGetLastError());
    pt.mark("count");
    if (mn <= SCAN_SMALL_MAX) {
      hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(SCAN_SMALL_THREADS), (sp.nc + 1) * 4, stream, matrix,
                         (uint32_t)mn, sp, slices, counts);
    } else {
      const uint32_t nbm = div_ceil32(mn, SCAN_BLOCK);
      hipLaunchKernelGGL(k_scan_blocks, dim3(nbm), dim3(THREADS), 0, stream, matrix, (uint32_t)mn, bsums);
      hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(THREADS), 0, stream, bsums, nbm);
      hipLaunchKernelGGL(k_scan_add, dim3(div_ceil32(mn, THREADS)), dim3(THREADS), 0, stream, matrix, (uint32_t)mn,
                         bsums, nullptr);
      hipLaunchKernelGGL(k_seg_plan, dim3(1), dim3(THREADS), (sp.nc + 1) * 4, stream, matrix, sp, slices, counts);
    }
    ZKP_CHECK(hipGetLastError());
    pt.mark("scan");
    hipLaunchKernelGGL(k_part_scatter, dim3(sp.tiles), dim3(THREADS), sp.lds_part, stream, d_scalars, len, cfg, sp,
                       matrix, ktmp, vtmp);
    ZKP_CHECK(hipGetLastError());
    pt.mark("partition");
    hipLaunchKernelGGL(k_seg_hist, dim3(L.max_slices), dim3(THREADS), nbk * 4, stream, ktmp, matrix, slices, sp, cursor);
    hipLaunchKernelGGL(k_seg_scan, dim3(sp.nc), dim3(THREADS), nbk * 4, stream, matrix, slices, sp, cursor);
    const uint32_t lds_seg = seg_scatter_lds(sp.low_bits);
    hipLaunchKernelGGL(k_seg_scatter, dim3(L.max_slices), dim3(THREADS), lds_seg, stream, ktmp, vtmp, matrix, slices,
                       sp, cursor, keys0, vals0);
    ZKP_CHECK(hipGetLastError());
    pt.mark("segsort");
  } else {
  const uint32_t h1 = L.H + 1;
  hipLaunchKernelGGL(k_zero_u32, dim3(grid_for(h1, 4096)), dim3(THREADS), 0, stream, hist, (uint64_t)h1);
  ZKP_CHECK(hipGetLastError());
  pt.mark("start");
  hipLaunchKernelGGL(k_histogram, dim3(grid_for(len, 8192)), dim3(THREADS), 0, stream, d_scalars, len, cfg, hist);
  ZKP_CHECK(hipGetLastError());
  pt.mark("histogram");
  hipLaunchKernelGGL(k_scan_blocks, dim3(L.nb_scan), dim3(THREADS), 0, stream, hist, h1, bsums);
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(THREADS), 0, stream, bsums, L.nb_scan);
  hipLaunchKernelGGL(k_scan_add, dim3(div_ceil32(h1, THREADS)), dim3(THREADS), 0, stream, hist, h1, bsums, cursor);
  hipLaunchKernelGGL(k_set_count, dim3(1), dim3(64), 0, stream, counts, hist, L.H);
  ZKP_CHECK(hipGetLastError());
  pt.mark("scan");
  hipLaunchKernelGGL(k_scatter, dim3(grid_for(len, 8192)), dim3(THREADS), 0, stream, d_scalars, len, cfg, cursor,
                     keys0, vals0);
  ZKP_CHECK(hipGetLastError());
  pt.mark("scatter");
  }
  return hipSuccess;
}

// Launches with at most this many point operations run a quad of lanes per
// operation (their time is the operations' latency, not their count): a quad
// adds in 2.5 us where a lone lane takes 5.6 us, but 65 536 quads already put
// four waves on every SIMD.
constexpr uint64_t QUAD_OPS = 65536;

// Second half: adds the sorted entries' points (n_precompute tables laid out
// table-major at d_points) into bucket set `set`.
static hipError_t accumulate_sorted(const Layout& L, char* ws, uint32_t set, const u32* d_points,
                                    hipStream_t stream, PhaseTimer& pt) {
  uint32_t* counts = reinterpret_cast<uint32_t*>(ws + L.counts);
  uint32_t* keys0 = reinterpret_cast<uint32_t*>(ws + L.keys0);
  uint32_t* vals0 = reinterpret_cast<uint32_t*>(ws + L.vals0);
  u32* pieces = reinterpret_cast<u32*>(ws + L.pieces);
  uint32_t* seg_meta = reinterpret_cast<uint32_t*>(ws + L.seg_meta);
  u32* seg_pts = reinterpret_cast<u32*>(ws + L.seg_pts);
  u32* buckets = bucket_set(L, ws, set);
  const uint32_t ch = L.share.ch;
  if (L.share.quads)
    hipLaunchKernelGGL(k_accumulate<true>, dim3(div_ceil32(4ull * L.chunks_max, THREADS)), dim3(THREADS), 0, stream,
                       keys0, vals0, d_points, counts, ch, buckets, pieces);
  else
    hipLaunchKernelGGL(k_accumulate<false>, dim3(div_ceil32(L.chunks_max, THREADS)), dim3(THREADS), 0, stream, keys0,
                       vals0, d_points, counts, ch, buckets, pieces);
  ZKP_CHECK(hipGetLastError());
  pt.mark("accumulate");
  if (L.chunks_max > 1) {
    if (L.share.quads)
      hipLaunchKernelGGL(k_close_runs<true>, dim3(div_ceil32(4ull * L.chunks_max, THREADS)), dim3(THREADS), 0, stream,
                         keys0, pieces, counts, ch, buckets);
    else
      hipLaunchKernelGGL(k_close_runs<false>, dim3(div_ceil32(L.chunks_max, THREADS)), dim3(THREADS), 0, stream, keys0,
                         pieces, counts, ch, buckets);
    ZKP_CHECK(hipGetLastError());
  }
  if (L.chunks_max > RUN_MAX + 1) {
    const uint32_t tiles = long_tiles_for(L.chunks_max);
    hipLaunchKernelGGL(k_long_tiles, dim3(tiles), dim3(THREADS), 0, stream, keys0, pieces, counts, ch, buckets,
                       seg_meta, seg_pts);
    hipLaunchKernelGGL(k_long_join, dim3(1), dim3(THREADS), 0, stream, counts, seg_meta, seg_pts, tiles, buckets);
    ZKP_CHECK(hipGetLastError());
  }
  pt.mark("runs");
  return hipSuccess;
}

// Adds sum_i k_i P_i for one part (len points, n_precompute tables laid out
// table-major at d_points) into bucket set `set`.
static hipError_t accumulate_part(const Config& cfg, const Layout& L, char* ws, uint32_t set, const u32* d_points,
                                  const u32* d_scalars, uint64_t len, hipStream_t stream, PhaseTimer& pt) {
  ZKP_CHECK(sort_part(cfg, L, ws, d_scalars, len, stream, pt));
  return accumulate_sorted(L, ws, set, d_points, stream, pt);
}

// Reduction of bucket set `set`; the n_windows window sums end at *out_dev (XYZZ).
static hipError_t reduce_buckets(const Config& cfg, const Layout& L, char* ws, uint32_t set, hipStream_t stream,
                                 const u32** out_dev, PhaseTimer& pt) {
  const u32* X = bucket_set(L, ws, set);
  const u32* Y = X;
  uint32_t M = cfg.buckets;
  if (M < 2 || (M & (M - 1))) return hipErrorInvalidValue;  // 2^(s-1) buckets, s >= 2
  int rl0 = 0;
  uint32_t fold = cfg.top_log;  // levels that fold the top window's copies
  // Levels 0 and 1 in one pass, into level 1's buffers, where its blocks are
  // enough to occupy the chip: the pass is a chain of eight point operations
  // (63 us however few blocks), the two levels by quads take 20-30 us up to
  // 32 768 blocks.
  if (L.red_levels >= 2 && (uint64_t)(M >> 2) * cfg.n_windows > QUAD_OPS / 2) {
    u32* Xo = reinterpret_cast<u32*>(ws + L.red[2]);
    u32* Yo = reinterpret_cast<u32*>(ws + L.red[3]);
    const uint32_t blocks = (M >> 2) * cfg.n_windows;
    hipLaunchKernelGGL(k_reduce_block4, dim3(div_ceil32(blocks, THREADS)), dim3(THREADS), 0, stream, X, M,
                       cfg.n_windows, fold, Xo, Yo);
    ZKP_CHECK(hipGetLastError());
    X = Xo;
    Y = Yo;
    M >>= 2;
    rl0 = 2;
    fold -= fold < 2 ? fold : 2;
  }
  for (int rl = rl0; rl < L.red_levels; rl++) {
    u32* Xo = reinterpret_cast<u32*>(ws + L.red[(rl % 2) * 2]);
    u32* Yo = reinterpret_cast<u32*>(ws + L.red[(rl % 2) * 2 + 1]);
    const uint32_t Mo = L.red_m[rl];
    const uint64_t ops = 2ull * Mo * cfg.n_windows;
    if (ops <= QUAD_OPS || rl0 == 0)
      hipLaunchKernelGGL(k_reduce_level_quad, dim3(div_ceil32(4 * ops, THREADS)), dim3(THREADS), 0, stream, X, Y, M,
                         cfg.n_windows, rl == 0, fold > 0, Xo, Yo);
    else
      hipLaunchKernelGGL(k_reduce_level, dim3(div_ceil32(ops, THREADS)), dim3(THREADS), 0, stream, X, Y, M,
                         cfg.n_windows, rl == 0, fold > 0, Xo, Yo);
    ZKP_CHECK(hipGetLastError());
    X = Xo;
    Y = Yo;
    M = Mo;
    fold -= fold > 0 ? 1 : 0;
  }
  u32* sums = reinterpret_cast<u32*>(ws + L.sums);
  hipLaunchKernelGGL(k_reduce_tail_quad, dim3(cfg.n_windows), dim3(QUAD_TAIL_THREADS), 0, stream, X, Y, M,
                     L.red_levels == 0, fold, sums);
  ZKP_CHECK(hipGetLastError());
  *out_dev = sums;
  pt.mark("reduce");
  return hipSuccess;
}

// Host Horner over the window sums: sum_w 2^(s w) S_w.
static G1XYZZ combine_windows(const Config& cfg, const std::vector<G1XYZZ>& sums) {
  G1XYZZ acc = G1XYZZ::identity();
  for (int w = (int)cfg.n_windows - 1; w >= 0; w--) {
    if (!acc.is_identity())
      for (uint32_t k = 0; k < cfg.s; k++) acc = acc.dbl();
    acc = acc.add(sums[w]);
  }
  return acc;
}

static hipError_t fetch_window_sums(const Config& cfg, const u32* d_sums, hipStream_t stream,
                                    std::vector<G1XYZZ>& out) {
  out.resize(cfg.n_windows);
  ZKP_CHECK(hipMemcpyAsync(out.data(), d_sums, sizeof(G1XYZZ) * cfg.n_windows, hipMemcpyDeviceToHost, stream));
  return hipStreamSynchronize(stream);
}

// Full device-resident MSM of one scalar batch: result (XYZZ, host).
static hipError_t msm_device(const Config& cfg, const u32* d_points, const u32* d_scalars, uint64_t len, char* ws,
                             const Layout& L, hipStream_t stream, G1XYZZ* result, bool debug) {
  PhaseTimer pt{debug, stream, {}, {}};
  ZKP_CHECK(reset_buckets(cfg, L, ws, 0, stream));
  if (len > 0) ZKP_CHECK(accumulate_part(cfg, L, ws, 0, d_points, d_scalars, len, stream, pt));
  const u32* d_sums = nullptr;
  ZKP_CHECK(reduce_buckets(cfg, L, ws, 0, stream, &d_sums, pt));
  std::vector<G1XYZZ> sums;
  ZKP_CHECK(fetch_window_sums(cfg, d_sums, stream, sums));
  auto t0 = std::chrono::steady_clock::now();
  *result = combine_windows(cfg, sums);
  if (debug) {
    pt.report();
    auto t1 = std::chrono::steady_clock::now();
    fprintf(stderr, "[msm] host combine %.4f ms\n", std::chrono::duration<double, std::milli>(t1 - t0).count());
  }
  return hipSuccess;
}

// ---------------------------------------------------------------- host-streamed MSM (the drop-in msm)
//
// Plan of one call: each card takes a contiguous range of points, split into
// `parts` pieces that are streamed through its buffer; batches run in groups
// of batch_per_run that share one pass over the parts, each with its own
// bucket set.  Copies go on two copy streams (points, scalars) into
// stage_points / stage_scalars rotating device buffers, ordered against the
// compute stream by events, so the next part's points and the next batch's
// scalars cross the link while the current accumulation runs.  Runs
// alternate the direction of their pass over the parts, so the part a run
// ends with is still resident when the next run starts with it (with one part
// the points cross the link once per call).
struct HostPlan {
  uint64_t part_len;      // points per part (the last may be shorter)
  uint32_t scratch_set;   // bucket set for the parts after a run's first (UINT32_MAX: one part)
  uint32_t stage_points;  // rotating device buffers for point parts
  uint32_t stage_scalars; // rotating device buffers for scalar parts
  uint32_t batch_per_run; // bucket sets
  size_t pts_bytes;       // one point stage: part_len * n_precompute affine points
  size_t sc_bytes;        // one scalar stage: part_len Fr elements
  Layout L;

  size_t total() const { return stage_points * pts_bytes + stage_scalars * sc_bytes + L.least; }
};

static bool make_host_plan(const Config& cfg, uint64_t card_len, uint32_t parts, uint32_t batch_per_run,
                           uint32_t stage_scalars, uint32_t stage_points, HostPlan* P) {
  if (parts == 0 || batch_per_run == 0 || stage_scalars == 0 || stage_points == 0) return false;
  if (batch_per_run > 1024 || stage_scalars > 64 || stage_points > 64) return false;
  P->part_len = (card_len + parts - 1) / parts;
  P->stage_points = stage_points;
  P->stage_scalars = stage_scalars;
  P->batch_per_run = batch_per_run;
  const bool several = P->part_len < card_len;
  P->scratch_set = several ? batch_per_run : UINT32_MAX;
  // (the buffer's size does not come with the call, so the plan is for the least)
  if (!make_layout(cfg, P->part_len ? P->part_len : 1, &P->L, batch_per_run + (several ? 1 : 0), UINT64_MAX) ||
      !make_layout(cfg, P->part_len ? P->part_len : 1, &P->L, batch_per_run + (several ? 1 : 0), P->L.least))
    return false;
  P->pts_bytes = align256((size_t)P->part_len * cfg.n_precompute * 64);
  P->sc_bytes = align256((size_t)P->part_len * 32);
  return true;
}

// One card's streams (compute, point copies, scalar copies), the events that
// order them, and pinned slots for the window sums.  Made once per device and
// kept for the process's lifetime in a free list (stream, event and pinned
// allocations cost more than a small MSM); a call takes one set for itself,
// grows it if its plan needs more stages, and gives it back drained.
struct CardRes {
  hipStream_t s = nullptr, cp = nullptr, cs = nullptr;
  std::vector<hipEvent_t> pt_ready, pt_free, sc_ready, sc_free;
  G1XYZZ* h_sums = nullptr;  // batch_per_run x n_windows window sums (pinned)
  size_t sums_cap = 0;

  hipError_t ensure(const Config& cfg, const HostPlan& P) {
    if (s == nullptr) ZKP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    if (cp == nullptr) ZKP_CHECK(hipStreamCreateWithFlags(&cp, hipStreamNonBlocking));
    if (cs == nullptr) ZKP_CHECK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    auto grow = [](std::vector<hipEvent_t>& v, uint32_t n) -> hipError_t {
      while (v.size() < n) {
        hipEvent_t e;
        ZKP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        v.push_back(e);
      }
      return hipSuccess;
    };
    ZKP_CHECK(grow(pt_ready, P.stage_points));
    ZKP_CHECK(grow(pt_free, P.stage_points));
    ZKP_CHECK(grow(sc_ready, P.stage_scalars));
    ZKP_CHECK(grow(sc_free, P.stage_scalars));
    const size_t need = sizeof(G1XYZZ) * cfg.n_windows * P.batch_per_run;
    if (sums_cap < need) {
      if (h_sums) ZKP_CHECK(hipHostFree(h_sums));
      h_sums = nullptr;
      sums_cap = 0;
      ZKP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&h_sums), need, hipHostMallocDefault));
      sums_cap = need;
    }
    // every stage starts free
    for (uint32_t i = 0; i < P.stage_points; i++) ZKP_CHECK(hipEventRecord(pt_free[i], s));
    for (uint32_t i = 0; i < P.stage_scalars; i++) ZKP_CHECK(hipEventRecord(sc_free[i], s));
    return hipSuccess;
  }
  void drain() {
    for (hipStream_t q : {s, cp, cs})
      if (q) (void)hipStreamSynchronize(q);
  }
};

static std::mutex g_res_mu;
static std::vector<CardRes*>* g_res_free = new std::vector<CardRes*>[64];  // per device; never freed

struct ResLease {
  int dev;
  CardRes* r = nullptr;
  explicit ResLease(int d) : dev(d) {
    std::lock_guard<std::mutex> lock(g_res_mu);
    auto& v = g_res_free[dev];
    if (!v.empty()) {
      r = v.back();
      v.pop_back();
    }
    if (r == nullptr) r = new CardRes;
  }
  ~ResLease() {
    r->drain();  // nothing of this call may still run when the set is reused
    std::lock_guard<std::mutex> lock(g_res_mu);
    g_res_free[dev].push_back(r);
  }
};

// Host-to-device copy of `bytes` on stream s.  With `pull`, pinned host memory
// that the device addresses at the host's own virtual address (hipHostMalloc'd
// or registered memory) is pulled by k_pull_host when both ends are 16-byte
// aligned; any other source (pageable memory), and every copy without `pull`,
// goes through hipMemcpyAsync.
static hipError_t copy_in(void* dst, const void* src, size_t bytes, hipStream_t s, bool pull) {
  if (bytes == 0) return hipSuccess;
  if (!pull) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
  hipPointerAttribute_t a{};
  const hipError_t q = hipPointerGetAttributes(&a, src);
  if (q != hipSuccess) (void)hipGetLastError();  // an unregistered pointer may be reported as an error
  const bool pinned = q == hipSuccess && a.type == hipMemoryTypeHost && a.devicePointer != nullptr &&
                      a.devicePointer == a.hostPointer;
  if (pinned && bytes % 16 == 0 && (uintptr_t)src % 16 == 0 && (uintptr_t)dst % 16 == 0) {
    hipLaunchKernelGGL(k_pull_host, dim3(PULL_BLOCKS), dim3(THREADS), 0, s, static_cast<const uint4*>(src),
                       static_cast<uint4*>(dst), (uint64_t)(bytes / 16));
    return hipGetLastError();
  }
  return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
}

// One card's share: points [c_off, c_off + c_len) of every table, all
// batches; adds the card's partial result of batch b into totals[b].
//
// Per part, each batch's scalars are copied first; the part's sort reads only
// them, so it runs while the part's points are still on the link; the
// accumulation waits for the points.  The next part's points are requested
// as soon as this part's first scalars are on their way, into another point
// stage, so they cross the link during this part's sorts and accumulations.
static hipError_t msm_card(const Config& cfg, const HostPlan& P, unsigned card, char* buf, uint64_t c_off,
                           uint64_t c_len, const u32* const* h_points, unsigned batches, const u32* const* h_scalars,
                           G1XYZZ* totals, bool debug) {
  ZKP_CHECK(hipSetDevice((int)card));
  int dev = 0;
  ZKP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  ResLease lease(dev);
  CardRes& R = *lease.r;
  ZKP_CHECK(R.ensure(cfg, P));
  const Layout& L = P.L;
  char* ws = buf + P.stage_points * P.pts_bytes + P.stage_scalars * P.sc_bytes;
  auto pts = [&](uint32_t st) { return reinterpret_cast<u32*>(buf + st * P.pts_bytes); };
  auto scs = [&](uint32_t st) { return reinterpret_cast<u32*>(buf + P.stage_points * P.pts_bytes + st * P.sc_bytes); };
  const uint32_t nparts = c_len ? (uint32_t)((c_len + P.part_len - 1) / P.part_len) : 0;
  // The copy kernel needs room on the CUs.  With one part the points cross the
  // link beside the sort only; with several, each part's copy runs beside the
  // previous part's accumulation, whose waves hold every CU's registers, and
  // the kernel would wait for them (2^20 points, window 16, four parts: 4.6 ms
  // with the kernel, 3.9 ms with DMA), so those copies go to the DMA engines.
  const bool pull = nparts == 1;
  auto part_off = [&](uint32_t p) { return c_off + (uint64_t)p * P.part_len; };
  auto part_len = [&](uint32_t p) {
    const uint64_t o = part_off(p), end = c_off + c_len;
    return end - o < P.part_len ? end - o : P.part_len;
  };
  // which part each point stage holds (-1: none); the copy has been enqueued
  std::vector<int64_t> held(P.stage_points, -1);
  std::vector<uint64_t> last_use(P.stage_points, 0);
  uint64_t clock = 0;
  uint32_t sc_next = 0;
  // stage holding part p, enqueueing its copy into the least recently used
  // stage other than `keep` when it is not resident; `after` (may be null) is
  // an event the copy waits for first (the scalars that should go first)
  auto points_of = [&](uint32_t p, int64_t keep, hipEvent_t after, uint32_t* out) -> hipError_t {
    for (uint32_t st = 0; st < P.stage_points; st++)
      if (held[st] == (int64_t)p) {
        *out = st;
        last_use[st] = ++clock;
        return hipSuccess;
      }
    uint32_t st = P.stage_points;
    for (uint32_t k = 0; k < P.stage_points; k++)
      if ((int64_t)k != keep && (st == P.stage_points || last_use[k] < last_use[st])) st = k;
    if (st == P.stage_points) st = 0;  // one stage: reuse it after its last reader
    ZKP_CHECK(hipStreamWaitEvent(R.cp, R.pt_free[st], 0));
    if (after != nullptr) ZKP_CHECK(hipStreamWaitEvent(R.cp, after, 0));
    const uint64_t off = part_off(p), n = part_len(p);
    for (uint32_t t = 0; t < cfg.n_precompute; t++)
      ZKP_CHECK(copy_in(pts(st) + (size_t)t * n * 16, h_points[t] + off * 16, n * 64, R.cp, pull));
    ZKP_CHECK(hipEventRecord(R.pt_ready[st], R.cp));
    held[st] = p;
    last_use[st] = ++clock;
    *out = st;
    return hipSuccess;
  };
  for (unsigned r0 = 0, run = 0; r0 < batches; r0 += P.batch_per_run, run++) {
    const uint32_t nb = batches - r0 < P.batch_per_run ? batches - r0 : P.batch_per_run;
    PhaseTimer pt{debug, R.s, {}, {}};
    for (uint32_t j = 0; j < nb; j++) ZKP_CHECK(reset_buckets(cfg, L, ws, j, R.s));
    const bool forward = (run & 1) == 0;
    for (uint32_t idx = 0; idx < nparts; idx++) {
      const uint32_t p = forward ? idx : nparts - 1 - idx;
      const uint64_t off = part_off(p), n = part_len(p);
      int64_t st = -1;
      for (uint32_t j = 0; j < nb; j++) {
        const uint32_t ss = sc_next++ % P.stage_scalars;
        ZKP_CHECK(hipStreamWaitEvent(R.cs, R.sc_free[ss], 0));
        ZKP_CHECK(copy_in(scs(ss), h_scalars[r0 + j] + off * 8, n * 32, R.cs, pull));
        ZKP_CHECK(hipEventRecord(R.sc_ready[ss], R.cs));
        if (j == 0) {
          // the part's points after its first scalars (resident parts are not copied again), then the next
          // part's points into another stage
          uint32_t s0 = 0;
          ZKP_CHECK(points_of(p, -1, R.sc_ready[ss], &s0));
          st = s0;
          if (idx + 1 < nparts && P.stage_points > 1) {
            uint32_t s1 = 0;
            ZKP_CHECK(points_of(forward ? p + 1 : p - 1, st, nullptr, &s1));
          }
        }
        ZKP_CHECK(hipStreamWaitEvent(R.s, R.sc_ready[ss], 0));
        ZKP_CHECK(sort_part(cfg, L, ws, scs(ss), n, R.s, pt));
        ZKP_CHECK(hipEventRecord(R.sc_free[ss], R.s));
        if (j == 0) ZKP_CHECK(hipStreamWaitEvent(R.s, R.pt_ready[st], 0));
        if (idx == 0 || P.scratch_set == UINT32_MAX) {
          ZKP_CHECK(accumulate_sorted(L, ws, j, pts((uint32_t)st), R.s, pt));
        } else {
          ZKP_CHECK(reset_buckets(cfg, L, ws, P.scratch_set, R.s));
          ZKP_CHECK(accumulate_sorted(L, ws, P.scratch_set, pts((uint32_t)st), R.s, pt));
          hipLaunchKernelGGL(k_merge_buckets, dim3(div_ceil32(L.H, THREADS)), dim3(THREADS), 0, R.s,
                             bucket_set(L, ws, j), bucket_set(L, ws, P.scratch_set), L.H);
          ZKP_CHECK(hipGetLastError());
        }
      }
      ZKP_CHECK(hipEventRecord(R.pt_free[st], R.s));
    }
    for (uint32_t j = 0; j < nb; j++) {
      const u32* d_sums = nullptr;
      ZKP_CHECK(reduce_buckets(cfg, L, ws, j, R.s, &d_sums, pt));
      ZKP_CHECK(hipMemcpyAsync(R.h_sums + (size_t)j * cfg.n_windows, d_sums, sizeof(G1XYZZ) * cfg.n_windows,
                               hipMemcpyDeviceToHost, R.s));
    }
    ZKP_CHECK(hipStreamSynchronize(R.s));
    pt.report();
    for (uint32_t j = 0; j < nb; j++) {
      std::vector<G1XYZZ> sums(R.h_sums + (size_t)j * cfg.n_windows, R.h_sums + (size_t)(j + 1) * cfg.n_windows);
      totals[r0 + j] = totals[r0 + j].add(combine_windows(cfg, sums));
    }
  }
  return hipSuccess;
}

}  // namespace msm
}  // namespace zkp

using namespace zkp;
using namespace zkp::msm;

extern "C" {

// Multi-scalar multiplication of host points / host scalars, results to host
// (affine), for MsmConfig (window, target_windows).  Behind msm of
// core/src/msm/src/msm.h:4-9 / msm.cu:9-41, with the same calling convention:
// with buffers == NULL only buffer_sizes[card] (bytes of device memory per
// card) is filled.  Points are split over the cards in contiguous ranges, one
// host thread per card (MultiGPUMSM, msm_impl.cuh:830-909); each card streams
// its range in `parts` pieces with batch_per_run batches per pass, through
// stage_points / stage_scalers rotating buffers on copy streams (MSM::run,
// msm_impl.cuh:374-603); the cards' results are summed on the host.
// Synchronous.  h_points holds n_precompute tables (msm_precompute),
// h_scaler_batch `batches` scalar arrays (Fr Montgomery, no rotation),
// h_result `batches` affine points.  Host arrays in pinned memory (as the
// runtime's CPU pool gives) let the copies overlap the accumulation.
hipError_t zkp_msm_host(unsigned int window, unsigned int target_windows, int debug_flag, void* const* buffers,
                        unsigned long* buffer_sizes, unsigned long long len, unsigned int batch_per_run,
                        unsigned int parts, unsigned int stage_scalers, unsigned int stage_points,
                        unsigned int num_cards, const unsigned int* cards, unsigned int const* const* h_points,
                        unsigned int batches, unsigned int const* const* h_scaler_batch,
                        unsigned int* const* h_result) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return hipErrorInvalidValue;
  if (num_cards == 0 || cards == nullptr) return hipErrorInvalidValue;
  const uint64_t card_len = (len + num_cards - 1) / num_cards;
  HostPlan P;
  if (!make_host_plan(cfg, card_len, parts, batch_per_run, stage_scalers, stage_points, &P))
    return hipErrorInvalidValue;
  if (buffers == nullptr) {
    if (buffer_sizes == nullptr) return hipErrorInvalidValue;
    for (unsigned c = 0; c < num_cards; c++) buffer_sizes[c] = P.total();
    return hipSuccess;
  }
  if (batches > 0 && (h_points == nullptr || h_scaler_batch == nullptr || h_result == nullptr))
    return hipErrorInvalidValue;
  const bool debug = debug_flag != 0;
  std::vector<std::vector<G1XYZZ>> partial(num_cards, std::vector<G1XYZZ>(batches, G1XYZZ::identity()));
  std::vector<hipError_t> errs(num_cards, hipSuccess);
  std::vector<std::thread> threads;
  for (unsigned c = 0; c < num_cards; c++) {
    const uint64_t c_off = c * card_len;
    if (c_off >= len) break;
    const uint64_t c_len = len - c_off < card_len ? len - c_off : card_len;
    auto job = [&, c, c_off, c_len]() {
      errs[c] = msm_card(cfg, P, cards[c], reinterpret_cast<char*>(buffers[c]), c_off, c_len, h_points, batches,
                         h_scaler_batch, partial[c].data(), debug);
    };
    if (num_cards == 1) job();
    else threads.emplace_back(job);
  }
  for (auto& t : threads) t.join();
  for (unsigned c = 0; c < num_cards; c++)
    if (errs[c] != hipSuccess) return errs[c];
  for (unsigned b = 0; b < batches; b++) {
    G1XYZZ total = G1XYZZ::identity();
    for (unsigned c = 0; c < num_cards; c++) total = total.add(partial[c][b]);
    const G1Affine a = total.to_affine();
    memcpy(h_result[b], a.x.v, 32);
    memcpy(h_result[b] + 8, a.y.v, 32);
  }
  return hipSuccess;
}

// Fills tables 1..n_precompute-1: h_points[j][i] = 2^(j * n_windows * s) * h_points[0][i]
// (affine), for MsmConfig (window, target_windows).  Behind msm_precompute of
// core/src/msm/src/msm.h:11 / msm_impl.cuh:776-828.  Synchronous; uses at most max_cards devices.
hipError_t zkp_msm_precompute_host(unsigned int window, unsigned int target_windows, unsigned long long len,
                                   unsigned int* const* h_points, unsigned int max_cards) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return hipErrorInvalidValue;
  if (cfg.n_precompute == 1 || len == 0) return hipSuccess;
  if (h_points == nullptr || max_cards == 0) return hipErrorInvalidValue;
  int devices = 0;
  ZKP_CHECK(hipGetDeviceCount(&devices));
  if (devices < 1) return hipErrorNoDevice;
  if ((unsigned)devices > max_cards) devices = (int)max_cards;
  const uint64_t per_dev = (len + devices - 1) / devices;
  for (int d = 0; d < devices; d++) {
    const uint64_t off = (uint64_t)d * per_dev;
    if (off >= len) break;
    const uint64_t n = len - off < per_dev ? len - off : per_dev;
    ZKP_CHECK(hipSetDevice(d));
    hipStream_t s;
    ZKP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    const uint64_t part = n < (1ull << 20) ? n : (1ull << 20);
    u32* dp = nullptr;
    hipError_t err = hipMalloc(&dp, (size_t)part * 64 * cfg.n_precompute);
    for (uint64_t p = 0; p < n && err == hipSuccess; p += part) {
      const uint64_t cur = n - p < part ? n - p : part;
      err = hipMemcpyAsync(dp, h_points[0] + (off + p) * 16, cur * 64, hipMemcpyHostToDevice, s);
      if (err != hipSuccess) break;
      hipLaunchKernelGGL(k_precompute, dim3(div_ceil32(cur, THREADS)), dim3(THREADS), 0, s, dp, cur,
                         cfg.n_precompute, cfg.n_windows * cfg.s);
      err = hipGetLastError();
      for (uint32_t j = 1; j < cfg.n_precompute && err == hipSuccess; j++)
        err = hipMemcpyAsync(h_points[j] + (off + p) * 16, dp + (size_t)j * cur * 16, cur * 64,
                             hipMemcpyDeviceToHost, s);
      if (err == hipSuccess) err = hipStreamSynchronize(s);
    }
    if (dp) (void)hipFree(dp);
    (void)hipStreamDestroy(s);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

// ---- extension entry points (no counterpart in the reference ABI) ----

// Device workspace bytes for zkp_msm_device with `len` points per table.
unsigned long long zkp_msm_workspace_size(unsigned long long len, unsigned int window, unsigned int target_windows) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return 0;
  Layout L;
  if (!make_layout(cfg, len ? len : 1, &L, 1, UINT64_MAX)) return 0;
  return L.total;
}

// The smallest workspace that zkp_msm_device accepts (0 if the configuration is
// invalid): no larger than an earlier version's size or a longer call's.  Below
// zkp_msm_workspace_size, small MSMs accumulate in longer chains.
unsigned long long zkp_msm_workspace_least(unsigned long long len, unsigned int window, unsigned int target_windows) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return 0;
  Layout L;
  if (!make_layout(cfg, len ? len : 1, &L, 1, UINT64_MAX)) return 0;
  return L.least;
}

// MSM with points (n_precompute tables of len affine points, table-major) and
// scalars already in device memory.  Runs on `stream`, then synchronizes it and
// writes the affine result to host memory h_result[16].
hipError_t zkp_msm_device(const unsigned int* d_points, const unsigned int* d_scalars, unsigned long long len,
                          unsigned int window, unsigned int target_windows, void* d_workspace,
                          unsigned long long workspace_bytes, hipStream_t stream, unsigned int* h_result, int debug) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return hipErrorInvalidValue;
  Layout L;
  if (!make_layout(cfg, len ? len : 1, &L, 1, workspace_bytes)) return hipErrorInvalidValue;
  if (d_workspace == nullptr || h_result == nullptr) return hipErrorInvalidValue;
  if (len > 0 && (d_points == nullptr || d_scalars == nullptr)) return hipErrorInvalidValue;
  G1XYZZ r;
  ZKP_CHECK(msm_device(cfg, d_points, d_scalars, len, reinterpret_cast<char*>(d_workspace), L, stream, &r,
                       debug != 0));
  const G1Affine a = r.to_affine();
  memcpy(h_result, a.x.v, 32);
  memcpy(h_result + 8, a.y.v, 32);
  return hipSuccess;
}

// zkp_msm_device split at the host boundary, for callers that batch MSMs into
// one stream or hipGraph: enqueues the whole device part (digits, sort,
// accumulation, bucket reduction) on `stream` and, when h_sums is not NULL,
// an asynchronous copy of the n_windows window sums (XYZZ, 128 bytes each)
// into h_sums (pinned host memory, n_windows * 128 bytes).  Nothing is
// allocated and nothing waits; zkp_msm_combine turns the sums into the
// result once the stream has passed the copy.  Launch permissions are set on
// the device's first MSM: run one MSM (or this call) outside a capture first.
hipError_t zkp_msm_device_enqueue(const unsigned int* d_points, const unsigned int* d_scalars, unsigned long long len,
                                  unsigned int window, unsigned int target_windows, void* d_workspace,
                                  unsigned long long workspace_bytes, hipStream_t stream, void* h_sums) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return hipErrorInvalidValue;
  Layout L;
  if (!make_layout(cfg, len ? len : 1, &L, 1, workspace_bytes)) return hipErrorInvalidValue;
  if (d_workspace == nullptr) return hipErrorInvalidValue;
  if (len > 0 && (d_points == nullptr || d_scalars == nullptr)) return hipErrorInvalidValue;
  char* ws = reinterpret_cast<char*>(d_workspace);
  PhaseTimer pt{false, stream, {}, {}};
  ZKP_CHECK(reset_buckets(cfg, L, ws, 0, stream));
  if (len > 0) ZKP_CHECK(accumulate_part(cfg, L, ws, 0, d_points, d_scalars, len, stream, pt));
  const u32* d_sums = nullptr;
  ZKP_CHECK(reduce_buckets(cfg, L, ws, 0, stream, &d_sums, pt));
  if (h_sums != nullptr)
    ZKP_CHECK(hipMemcpyAsync(h_sums, d_sums, sizeof(G1XYZZ) * cfg.n_windows, hipMemcpyDeviceToHost, stream));
  return hipSuccess;
}

// Result of an MSM from its window sums (as zkp_msm_device_enqueue copied
// them): Horner over the windows on the host, affine into h_result[16].
hipError_t zkp_msm_combine(unsigned int window, unsigned int target_windows, const void* h_sums,
                           unsigned int* h_result) {
  Config cfg;
  if (!make_config(window, target_windows, &cfg)) return hipErrorInvalidValue;
  if (h_sums == nullptr || h_result == nullptr) return hipErrorInvalidValue;
  const G1XYZZ* p = reinterpret_cast<const G1XYZZ*>(h_sums);
  std::vector<G1XYZZ> sums(p, p + cfg.n_windows);
  const G1Affine a = combine_windows(cfg, sums).to_affine();
  memcpy(h_result, a.x.v, 32);
  memcpy(h_result + 8, a.y.v, 32);
  return hipSuccess;
}

// out[i] = k_i * G (affine, Fq Montgomery) for Fr Montgomery scalars k_i on the
// device; asynchronous on stream.
hipError_t zkp_g1_mul_generator(const unsigned int* d_scalars, unsigned long long n, unsigned int* d_out,
                                hipStream_t stream) {
  if (n == 0) return hipSuccess;
  if (d_scalars == nullptr || d_out == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mul_generator, dim3(div_ceil32(n, THREADS)), dim3(THREADS), 0, stream, d_scalars, (uint64_t)n,
                     d_out);
  return hipGetLastError();
}

// Derived configuration for (window, target_windows): {window,
// actual_windows, n_windows, n_precompute, buckets}; returns 0 if invalid.
int zkp_msm_config(unsigned int window, unsigned int target_windows, unsigned int* out5) {
  Config c;
  if (!make_config(window, target_windows, &c)) return 0;
  out5[0] = c.s;
  out5[1] = c.actual_windows;
  out5[2] = c.n_windows;
  out5[3] = c.n_precompute;
  out5[4] = c.buckets;
  return 1;
}

}  // extern "C"
