// BN254 Fr in nine signed 29-bit limbs: the butterflies of the transforms
// (host + device).
//
// A value is sum_i l_i 2^(29 i) with signed 32-bit limbs; it stands for an
// element x 2^256 mod r of bn254.hpp's form, reduced only as far as the next
// step needs it.  What that buys against eight 32-bit limbs, per butterfly:
//  * a limb product is one v_mad_i64_i32 into a 64-bit column that never
//    overflows, where 32-bit limbs spend a second instruction folding each
//    carry: 205 VALU instructions a product against 281 (with 221, before chain()
//    below, 910 against 1 190 SIMD cycles per wave at four waves per SIMD);
//  * a + t and a - t are nine v_add_u32 / v_sub_u32 with no carry and no
//    conditional subtraction (2.3 cycles each; a carry chain's v_addc takes 4.2):
//    about 50 cycles where the two lazy 32-bit additions and the reduction of
//    a took 175.
//
// Product: mul(x, w) = x w 2^-256 mod r for a multiplier w unpacked with a 5-bit
// shift (w 2^5, radix 2^261).  Each digit is m = T r^-1 mod 2^29 (r = 1 + 2^28
// mod 2^29 is its own inverse: one shift-add) and T gains m (-r).
// Bounds, with N = 2^29:
//  * limbs of x in (-3N, 3N), of w in [0, N); -r is written in balanced limbs
//    (|.| <= N / 2): a column is below 9 3N^2 + 9 N^2 / 2 + carry < 2^63;
//  * the result has limbs 0..7 in [0, N) (limb 8 signed), and for |x| <= X r and
//    w < r it lies in (-0.19 X r - r, 0.19 X r], since T / 2^261 = x w / 2^256
//    and r / 2^256 < 0.19.  So a butterfly takes X to at most 1.19 X + 1, ten
//    stages take 2 to 36, and limb 8 (x >> 232, 22 bits per r) stays below 2^28.
//  * norm() brings limbs 0..7 back to [0, N).  a + t and a - t with a and t
//    normalised have limbs in (-N, 2N), one stage more in (-2N, 3N): a normalised
//    value survives two stages before it is a factor or needs norm().
//  * reduce() brings any value with |limb 8| < 2^30 to [0, 1.0002 r).
#pragma once
#include "bn254.hpp"

namespace zkp {

struct Fr29 {
  int32_t l[9];

  static constexpr int32_t MASK = (1 << 29) - 1;
  // -r in balanced limbs
  static constexpr int32_t NEG_R[9] = {0x0fffffff,  0x00f05360,  -0x0e5c2451, -0x07d090f3, 0x0a7a2d7d,
                                       -0x02db40c1, -0x00a6e141, -0x0e5c2634, -0x0030644e};

  // (words << SHIFT) for a 256-bit little-endian value, SHIFT 0 or 5.
  template <int SHIFT>
  ZKP_HD static Fr29 from_words(const u32 (&w)[8]) {
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      const int s = 29 * i - SHIFT;  // first source bit of limb i
      u32 v;
      if (s < 0) {
        v = w[0] << (-s);
      } else {
        const int word = s >> 5, off = s & 31;
        const u32 lo = w[word], hi = word + 1 < 8 ? w[word + 1] : 0u;
        v = off ? (lo >> off) | (hi << (32 - off)) : lo;
      }
      r.l[i] = i < 8 ? (int32_t)(v & MASK) : (int32_t)v;
    }
    return r;
  }
  // Packs normalised limbs of a value in [0, 2^256).
  ZKP_HD void to_words(u32 (&w)[8]) const {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int b = 32 * k, i = b / 29, o = b % 29;
      u32 v = (u32)l[i] >> o;
      v |= (u32)l[i + 1] << (29 - o);
      if (58 - o < 32 && i + 2 < 9) v |= (u32)l[i + 2] << (58 - o);
      w[k] = v;
    }
  }

  ZKP_HD Fr29 operator+(const Fr29& b) const {
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = l[i] + b.l[i];
    return r;
  }
  ZKP_HD Fr29 operator-(const Fr29& b) const {
    Fr29 r;
#pragma unroll
    for (int i = 0; i < 9; i++) r.l[i] = l[i] - b.l[i];
    return r;
  }

  // limbs 0..7 carried into [0, 2^29), value unchanged
  ZKP_HD Fr29 norm() const {
    Fr29 r;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int32_t t = l[i] + c;
      r.l[i] = t & MASK;
      c = t >> 29;
    }
    r.l[8] = l[8] + c;
    return r;
  }

  // Keeps a column's additions in one chain of multiply-adds that starts from
  // the carry: after it the factors f count as newer than acc, and the compiler,
  // which adds the newest values last, adds acc first.  Left to itself it sums
  // the products apart and joins them with a v_lshl_add_u64, 16 a product.  (A
  // multiply-add written in asm gets an s_nop behind it.)
  ZKP_HD static void chain(int64_t& acc, int32_t (&f)[9], int n) {
#if defined(__HIP_DEVICE_COMPILE__)
    switch (n) {  // n is a constant where the column loop is unrolled
      case 1: asm("" : "+v"(acc), "+v"(f[0])); break;
      case 2: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1])); break;
      case 3: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2])); break;
      case 4: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3])); break;
      case 5: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4])); break;
      case 6: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5])); break;
      case 7: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6])); break;
      case 8: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7])); break;
      default: asm("" : "+v"(acc), "+v"(f[0]), "+v"(f[1]), "+v"(f[2]), "+v"(f[3]), "+v"(f[4]), "+v"(f[5]), "+v"(f[6]), "+v"(f[7]), "+v"(f[8])); break;
    }
#endif
  }

  // x w 2^-256 (bounds above); w from from_words<5>
  ZKP_HD static Fr29 mul(Fr29 x, const Fr29& w) {
    int32_t m[9];
    Fr29 r;
    int64_t acc = 0;
#pragma unroll
    for (int k = 0; k < 17; k++) {
      if (k) chain(acc, x.l, 9);
#pragma unroll
      for (int i = 0; i < 9; i++) {
        const int j = k - i;
        if (j >= 0 && j <= 8) acc += (int64_t)x.l[i] * w.l[j];
      }
      if (k) chain(acc, m, k);
#pragma unroll
      for (int i = 0; i < 9; i++) {
        const int j = k - i;
        if (i < k && j >= 1 && j <= 8) acc += (int64_t)m[i] * NEG_R[j];
      }
      if (k < 9) {
        const u32 lo = (u32)acc;
        m[k] = (int32_t)((lo + (lo << 28)) & (u32)MASK);
        acc += (int64_t)m[k] * NEG_R[0];  // clears the low 29 bits
      } else {
        r.l[k - 9] = (int32_t)((u32)acc & (u32)MASK);
      }
      acc >>= 29;
    }
    r.l[8] = (int32_t)acc;
    return r;
  }

  // The representative in [0, 1.0002 r), normalised, for |limb 8| < 2^30.
  // top = limb 8 + (limb 7 >> 29) differs from x / 2^232 by less than 2, that is
  // 6.4e-7 of r, and the float quotient from top / (r / 2^232) by less than 2^-14;
  // so q = floor(quotient - 2^-13) never exceeds x / r and falls short of it by less
  // than 1.0002.
  ZKP_HD Fr29 reduce() const {
    const int32_t top = l[8] + (l[7] >> 29);
    const int32_t q = (int32_t)floorf((float)top * (1.0f / 3171406.449f) - 0x1p-13f);
    Fr29 r;
    int64_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      c += (int64_t)q * NEG_R[i] + l[i];
      r.l[i] = (int32_t)((u32)c & (u32)MASK);
      c >>= 29;
    }
    r.l[8] = l[8] + q * NEG_R[8] + (int32_t)c;
    return r;
  }
};

}  // namespace zkp
