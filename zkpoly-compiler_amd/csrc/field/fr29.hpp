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

// ---------------------------------------------------------------- inversion
//
// mul's two operands stand for x 2^256 and y 2^256 when the second is unpacked 5
// bits up; a value that serves as second operand again has to keep the factor 32
// itself.  Call a value "up" when it is 32 x 2^256 mod r: up * up is up, and
// plain * up is plain.  Unpacked words are up below 32 r, for which mul's result
// is below 6.1 r in magnitude, and results of mul are normalised, so chains of
// products go on without end in either operand.
//
// inverse(x, c) = x^-1 c 2^-261 mod r for a normalised x in [0, 2 r); 0 where x
// is 0 mod r.  With c = INV_PLAIN it maps x 2^256 to x^-1 2^256, with INV_UP an up value of x
// to x^-1 2^256.
//
// By the division steps of Bernstein and Yang (Fast constant-time gcd computation
// and modular inversion, 2019, definition 8.1), with f = r, g = x and delta = 1: f is
// odd, and a step takes
//   (delta, f, g) to (1 - delta, g, (g - f) / 2) if delta > 0 and g is odd,
//                    (1 + delta, f, (g + (g mod 2) f) / 2) otherwise.
// 29 steps at a time are taken on the low words and collected in a matrix that is
// then applied to f and g (exactly divisible by 2^29) and, mod r, to d and e with
// d x = f, e x = g (mod r).
// A batch changes |d| and |e| by at most r, so limb 8 stays below 2^28 for the at
// most 26 batches (754 steps; the paper bounds 256-bit inputs by 741).
struct Fr29Inverse {
  static constexpr int32_t R[9] = {0x10000001, 0x1f0fac9f, 0x0e5c2450, 0x07d090f3,
                                  0x1585d283, 0x02db40c0, 0x00a6e141, 0x0e5c2634, 0x0030644e};
  static constexpr int32_t INV_PLAIN[9] = {0x17e007f8, 0x1c5b7cb8, 0x0ad4a06c, 0x08aaffa3,
                                  0x13abc077, 0x0f7013f7, 0x190d945a, 0x1b1dfff5, 0x001be8b5};
  static constexpr int32_t INV_UP[9] = {0x1c00feee, 0x1c5573e0, 0x18197fea, 0x08b5c34c,
                                  0x120f41ae, 0x1a97f167, 0x15f6b4bb, 0x01454f10, 0x00160937};

  int32_t u, v, q, r;  // 2^29 (f', g') = [u v; q r] (f, g)

  // 29 division steps on the low 32 bits of f (odd) and g: after k of them 32 - k
  // bits of g are still right.  The matrix is kept times 2^k, so that steps which
  // shift g down shift f's row up.  Steps that do the same are taken together:
  //  * those that find g even halve it and count;
  //  * with g odd and delta > 0 f and g change places: written as (f, g) = (g, -f)
  //    with delta = -delta, what is left of that step is one of the third kind;
  //  * with delta <= 0 the next 1 - delta steps keep f, and k of them take g to
  //    (g + w f) / 2^k, the w < 2^k that makes the sum divisible: w = -g / f.  An odd f
  //    is its own inverse mod 8 and a Newton step x (2 - f x) from there is right mod
  //    64, so w = g f (f^2 - 2) mod 2^k up to k = 6.
  // The shift by k is left to the next round, which finds those zeros.  (Gathering
  // variable-time steps, up to six of the last kind, is public practice: libsecp256k1
  // does so.  With no more than three a lone inversion took 0.8 us more.)
  ZKP_HD void steps(u32 f, u32 g, int32_t& delta) {
    u32 fu = 1, fv = 0, gu = 0, gv = 1;  // 2^k f' = fu f + fv g, 2^k g' = gu f + gv g
    for (u32 left = 29;;) {
      const u32 k = (u32)__builtin_ctz(g | 1u << left);
      g >>= k;
      fu <<= k;
      fv <<= k;
      delta += (int32_t)k;
      left -= k;
      if (left == 0) break;
      if (delta > 0) {
        const u32 f0 = f, u0 = fu, v0 = fv;
        f = g;
        fu = gu;
        fv = gv;
        g = 0u - f0;
        gu = 0u - u0;
        gv = 0u - v0;
        delta = -delta;
      }
      // k = min(6, 1 - delta, left), as a mask; delta <= 0 here
      const u32 mask = (delta < -4 ? 63u : ~(~0u << (1 - delta))) & ~(~0u << left);
      const u32 w = g * (f * (f * f - 2)) & mask;
      g += w * f;
      gu += w * fu;
      gv += w * fv;
    }
    u = (int32_t)fu;
    v = (int32_t)fv;
    q = (int32_t)gu;
    r = (int32_t)gv;
  }

  // (a x + b y) / 2^29: exact with mod = 0, mod r with mod = MASK
  ZKP_HD static Fr29 row(int32_t a, const Fr29& x, int32_t b, const Fr29& y, int32_t mod) {
    Fr29 o;
    int64_t acc = (int64_t)a * x.l[0] + (int64_t)b * y.l[0];
    const u32 lo = (u32)acc;
    const int32_t m = (int32_t)(lo + (lo << 28)) & mod;
    acc += (int64_t)m * Fr29::NEG_R[0];
    acc >>= 29;
#pragma unroll
    for (int i = 1; i < 9; i++) {
      acc += (int64_t)a * x.l[i] + (int64_t)b * y.l[i];
      acc += (int64_t)m * Fr29::NEG_R[i];
      o.l[i - 1] = (int32_t)((u32)acc & (u32)Fr29::MASK);
      acc >>= 29;
    }
    o.l[8] = (int32_t)acc;
    return o;
  }

  // On the device the lanes of a wave work together (all of them call, with the
  // same x): the steps run on the scalar unit, and lanes 0..3 of every quad form f,
  // g, d and e, each from the pair (p, q) = (f, g) or (d, e) that it keeps a copy
  // of.  12 us as a launch of one wave.  (With all of it on one lane of the vector
  // unit the batched inversion took 119 us where it took 92 with this.)
  ZKP_HD static Fr29 inverse(const Fr29& x, const int32_t (&c)[9]) {
    Fr29 w;
    int32_t delta = 1;
    Fr29Inverse s;
#if defined(__HIP_DEVICE_COMPILE__)
    const u32 lane = threadIdx.x;
    const bool second = lane & 1, mod_r = lane & 2;
    const int32_t mod = mod_r ? Fr29::MASK : 0;
    Fr29 p, q;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      p.l[i] = mod_r ? 0 : R[i];
      q.l[i] = mod_r ? (i == 0 ? 1 : 0) : x.l[i];
      w.l[i] = c[i];
    }
#pragma unroll 1
    for (int n = 0; n < 26; n++) {
      int32_t any = 0;
#pragma unroll
      for (int i = 0; i < 9; i++) any |= q.l[i];
      if (__builtin_amdgcn_readfirstlane(any) == 0) break;
      s.steps((u32)__builtin_amdgcn_readfirstlane(p.l[0] | p.l[1] << 29),
              (u32)__builtin_amdgcn_readfirstlane(q.l[0] | q.l[1] << 29), delta);
      const Fr29 o = row(second ? s.q : s.u, p, second ? s.r : s.v, q, mod);
#pragma unroll
      for (int i = 0; i < 9; i++) {
        p.l[i] = __builtin_amdgcn_update_dpp(0, o.l[i], 0xa0, 0xf, 0xf, true);  // quad_perm 0, 0, 2, 2
        q.l[i] = __builtin_amdgcn_update_dpp(0, o.l[i], 0xf5, 0xf, 0xf, true);  // quad_perm 1, 1, 3, 3
      }
    }
    const int32_t top = __builtin_amdgcn_readfirstlane(p.l[8]);
    Fr29 d;
#pragma unroll
    for (int i = 0; i < 9; i++) d.l[i] = __builtin_amdgcn_update_dpp(0, p.l[i], 0xaa, 0xf, 0xf, true);  // lane 2's
#else
    Fr29 f, g = x, d, e;
    for (int i = 0; i < 9; i++) {
      f.l[i] = R[i];
      d.l[i] = 0;
      e.l[i] = i == 0 ? 1 : 0;
      w.l[i] = c[i];
    }
    for (int n = 0; n < 26; n++) {
      int32_t any = 0;
      for (int i = 0; i < 9; i++) any |= g.l[i];
      if (any == 0) break;
      s.steps((u32)f.l[0] | (u32)f.l[1] << 29, (u32)g.l[0] | (u32)g.l[1] << 29, delta);
      const Fr29 f1 = row(s.u, f, s.v, g, 0), d1 = row(s.u, d, s.v, e, Fr29::MASK);
      g = row(s.q, f, s.r, g, 0);
      e = row(s.q, d, s.r, e, Fr29::MASK);
      f = f1;
      d = d1;
    }
    const int32_t top = f.l[8];
#endif
    // f = 1, -1, or r times one of them where x = 0 (mod r)
    const int32_t sign = top == 0 ? 1 : top == -1 ? -1 : 0;
#pragma unroll
    for (int i = 0; i < 9; i++) d.l[i] *= sign;
    return Fr29::mul(d, w);
  }
};

}  // namespace zkp
