// BN254 G1 XYZZ points over Fq29 (nine 29-bit limbs, radix 2^261): the
// buckets of the MSM (host + device).
//
// Same formulas as G1XYZZ in g1.hpp (EFD "xyzz", a = 0: madd-2008-s,
// add-2008-s, dbl-2008-s-1, with the equal and opposite point cases handled
// exactly), with Fq29's lazy reduction.  Invariant of every point passed
// between operations: X < 8p, Y < 4p, ZZ, ZZZ < 2p, limbs normalised; the
// identity has every limb zero (ZZ = 0 is the test).  Each formula below keeps
// it, with these bounds (A B <= 168 for every product, A B + C D for a pair
// that shares one reduction):
//  madd:  U2 = x ZZ (32 x 2), S2 = y ZZZ; P = U2 + 8p - X < 10p,
//         R = S2 + 4p - Y < 6p; PP = P^2 (100), PPP = P PP, Q = X PP, R^2 (36);
//         X3 = R^2 + 6p - PPP - 2Q < 8p; Y3 = R (Q + 8p - X3) + (4p - Y) PPP (60 + 8) < 2p
//  add:   U1, U2, S1, S2 < 2p; P, R < 4p; X3 < 8p; Q - X3 < 10p; Y3 = R (Q + 8p - X3) + (4p - S1) PPP
//  dbl:   U = 2Y < 8p; V = U^2 (64), X^2 (64); M = 3 X^2 < 6p; X3 = M^2 + 4p - 2S < 6p;
//         Y3 = M (S + 8p - X3) + (4p - Y) W (60 + 8) < 2p
// Y3's two products share a reduction: 90 limb products fewer of about 1 700.
// Equal operands double through the addition's own steps: with P = 2Y, R = 3 X^2,
// Q = X P^2 and no P^3 in X3 they are dbl-2008-s-1's, so the case costs one more
// product in its branch and no second formula in the code.  The instruction
// cache (64 KB per two CUs) holds a loop over one addition but not the 80 to
// 313 KB that kernels with a doubling inlined in every addition took.
// Affine inputs come from HBM in the form of bn254.hpp and are read as
// x 2^261 below 32p (Fq29::load_mont256); they meet only ZZ and ZZZ in
// products (32 x 2), and are brought below 2p (Fq29::reduce_2p) where they
// become a point's X and Y.
// In HBM a point is four packed elements (128 bytes); X is brought below 2p
// first so that every coordinate is below 2^256.
#pragma once
#include "../field/fq29.hpp"

namespace zkp {

struct Affine29 {
  Fq29 x, y;  // below 32p
  bool inf;

  // An affine point of G1Affine's layout (x, y in the form of bn254.hpp, (0, 0) the identity).
  __device__ __forceinline__ static Affine29 load(const u32* p, bool negate) {
    u32 wx[8], wy[8];
    Fq29::load_words(p, wx);
    Fq29::load_words(p + 8, wy);
    u32 any = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) any |= wx[i] | wy[i];
    Affine29 a;
    a.inf = any == 0;
    a.x = Fq29::from_words<5>(wx);
    a.y = Fq29::from_words<5>(wy);
    // -y = 32 p - y (below 32 p; y = 0 only for points of order 2, which G1 has none of)
    if (negate) a.y = Fq29::zero().sub<32>(a.y);
    return a;
  }
};

struct G1X29 {
  Fq29 x, y, zz, zzz;

  ZKP_HD static G1X29 identity() { return G1X29{Fq29::zero(), Fq29::zero(), Fq29::zero(), Fq29::zero()}; }
  ZKP_HD bool is_identity() const { return zz.all_zero(); }

  // (reduce_2p, not a product by one: a run's first point takes this path in
  // a few lanes of the wave while the others wait)
  ZKP_HD static G1X29 from_affine(const Affine29& a) {
    const Fq29 one = Fq29::one();
    return G1X29{a.x.reduce_2p(), a.y.reduce_2p(), one, one};
  }

  __device__ __forceinline__ static G1X29 load(const u32* p) {
    return G1X29{Fq29::load(p), Fq29::load(p + 8), Fq29::load(p + 16), Fq29::load(p + 24)};
  }
  __device__ __forceinline__ void store(u32* p) const {
    x.reduce_2p().store(p);
    y.store(p + 8);
    zz.store(p + 16);
    zzz.store(p + 24);
  }
  // dbl-2008-s-1
  ZKP_HD G1X29 dbl() const {
    if (is_identity()) return *this;
    const Fq29 u = y + y;
    const Fq29 v = u * u;
    const Fq29 x2 = x * x;
    const Fq29 m = (x2 + x2 + x2).norm();
    const Fq29 w = u * v;
    const Fq29 s = x * v;
    const Fq29 m2 = m * m;
    G1X29 r;
    r.zz = v * zz;
    r.x = m2.sub<4>(s + s);
    r.y = Fq29::mul_add(m, s.sub<8>(r.x), y.neg<4>(), w);
    r.zzz = w * zzz;
    return r;
  }

  // madd-2008-s: this + a
  ZKP_HD G1X29 add_affine(const Affine29& a) const {
    if (a.inf) return *this;
    if (is_identity()) return from_affine(a);
    const Fq29 u2 = a.x * zz;
    const Fq29 s2 = a.y * zzz;
    Fq29 p = u2.sub<8>(x);
    Fq29 rr = s2.sub<4>(y);
    bool same = false;
    if (p.is_zero_modp()) {
      if (!rr.is_zero_modp()) return identity();
      doubling_steps(p, rr);
      same = true;
    }
    return finish(p, rr, x, y, zz, zzz, same);
  }

  // add-2008-s: this + o
  ZKP_HD G1X29 add(const G1X29& o) const {
    if (o.is_identity()) return *this;
    if (is_identity()) return o;
    Fq29 u1 = x * o.zz;
    const Fq29 u2 = o.x * zz;
    Fq29 s1 = y * o.zzz;
    const Fq29 s2 = o.y * zzz;
    Fq29 p = u2.sub<2>(u1);
    Fq29 rr = s2.sub<2>(s1);
    Fq29 zz12 = zz * o.zz;
    Fq29 zzz12 = zzz * o.zzz;
    bool same = false;
    if (p.is_zero_modp()) {
      if (!rr.is_zero_modp()) return identity();
      doubling_steps(p, rr);
      u1 = x;
      s1 = y;
      zz12 = zz;
      zzz12 = zzz;
      same = true;
    }
    return finish(p, rr, u1, s1, zz12, zzz12, same);
  }

 private:
  // P and R of the addition's last steps when they double this point.
  ZKP_HD void doubling_steps(Fq29& p, Fq29& rr) const {
    const Fq29 x2 = x * x;
    p = (y + y).norm();
    rr = (x2 + x2 + x2).norm();
  }
  // X3, Y3, ZZ3, ZZZ3 from P, R, U1, S1, ZZ1 ZZ2 and ZZZ1 ZZZ2.
  ZKP_HD static G1X29 finish(const Fq29& p, const Fq29& rr, const Fq29& u1, const Fq29& s1, const Fq29& zz12,
                             const Fq29& zzz12, bool same) {
    const Fq29 pp = p * p;
    const Fq29 r2 = rr * rr;
    const Fq29 ppp = p * pp;
    const Fq29 q = u1 * pp;
    G1X29 r;
    r.zz = zz12 * pp;
    r.x = r2.sub<6>((same ? Fq29::zero() : ppp) + q + q);
    r.y = Fq29::mul_add(rr, q.sub<8>(r.x), s1.neg<4>(), ppp);
    r.zzz = zzz12 * ppp;
    return r;
  }
};

// ---- quad-cooperative XYZZ arithmetic (device) ----
//
// Where few point operations are left (the last levels of the bucket
// reduction, the accumulation of a small MSM) each one would run on a single
// lane with its products one after another.  Here a point lies across the four
// lanes of a quad (q = lane & 3), lane 0 holding X, 1 Y, 2 ZZ and 3 ZZZ, and a
// phase of independent products is one product on every lane: add-2008-s takes
// four product latencies instead of 14 (4, 4, 3 and 3 products), madd-2008-s
// four instead of 10, doubling (equal operands) one more.  DPP quad permutes
// move factors between the lanes, nine moves each; a first form in which all
// four lanes held all four coordinates spent twice as many moves and selects
// and four times the registers.  Every branch depends only on values that the
// whole quad shares, so its lanes always run together.
template <int L0, int L1, int L2, int L3>
__device__ __forceinline__ u32 quad_perm(u32 x) {
  return (u32)__builtin_amdgcn_mov_dpp((int)x, L0 | L1 << 2 | L2 << 4 | L3 << 6, 0xf, 0xf, false);
}
template <int L0, int L1, int L2, int L3>
__device__ __forceinline__ Fq29 quad_perm(const Fq29& x) {
  Fq29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = quad_perm<L0, L1, L2, L3>(x.l[i]);
  return r;
}
template <int L>
__device__ __forceinline__ Fq29 quad_lane(const Fq29& x) {
  return quad_perm<L, L, L, L>(x);
}
// lane by lane: c ? a : b
__device__ __forceinline__ Fq29 lane_pick(bool c, const Fq29& a, const Fq29& b) {
  Fq29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = c ? a.l[i] : b.l[i];
  return r;
}

struct Quad29 {
  Fq29 c;  // this lane's coordinate

  __device__ __forceinline__ static Quad29 identity() { return Quad29{Fq29::zero()}; }
  __device__ __forceinline__ static Quad29 load(const u32* p, u32 q) { return Quad29{Fq29::load(p + 8 * q)}; }
  __device__ __forceinline__ void store(u32* p, u32 q) const { c.reduce_2p().store(p + 8 * q); }
  __device__ __forceinline__ bool is_identity() const {
    u32 any = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) any |= c.l[i];
    return quad_perm<2, 2, 2, 2>(any) == 0;
  }
  // lane 0's coordinate x and lane 1's y of an affine point (lanes 2 and 3 hold them too)
  __device__ __forceinline__ static Quad29 from_affine(const Fq29& xy, u32 q) {
    return Quad29{lane_pick(q < 2, xy.reduce_2p(), Fq29::one())};
  }

  // P (lane 0) and R (lane 1) in d; r1: U1 (lane 0) and S1 (lane 1); zz: ZZ1
  // ZZ2 (lane 2) and ZZZ1 ZZZ2 (lane 3); r2: P^2 (lane 0) and R^2 (lane 1).
  __device__ __forceinline__ static Quad29 finish(const Fq29& d, const Fq29& r1, const Fq29& zz, const Fq29& r2,
                                                  bool same, u32 q) {
    const Fq29 g = lane_pick(q == 0, d, lane_pick(q == 1, quad_lane<0>(r1), zz));
    const Fq29 r3 = g * quad_lane<0>(r2);  // PPP, Q, ZZ3
    const Fq29 ppp = quad_lane<0>(r3), qq = quad_lane<1>(r3);
    const Fq29 x3 = quad_lane<1>(r2).sub<6>((same ? Fq29::zero() : ppp) + qq + qq);
    const Fq29 h1 = lane_pick(q == 0, quad_lane<1>(d), lane_pick(q == 1, r1.neg<4>(), zz));
    const Fq29 r4 = h1 * lane_pick(q == 0, qq.sub<8>(x3), ppp);  // R (Q - X3), -S1 PPP, , ZZZ3
    const Fq29 y3 = (r4 + quad_lane<0>(r4)).norm();
    return Quad29{lane_pick(q < 2, lane_pick(q == 0, x3, y3), lane_pick(q == 2, r3, r4))};
  }
  // d for doubling this point: 2Y on lane 0, 3 X^2 on the others
  __device__ __forceinline__ Fq29 doubling_steps(u32 q) const {
    const Fq29 x2 = quad_lane<0>(c * c), y = quad_lane<1>(c);
    return lane_pick(q == 0, y + y, x2 + x2 + x2).norm();
  }

  __device__ __forceinline__ Quad29 add(const Quad29& o, u32 q) const {
    if (o.is_identity()) return *this;
    if (is_identity()) return o;
    Fq29 r1 = c * quad_perm<2, 3, 0, 1>(o.c);        // U1, S1, U2, S2
    Fq29 d = quad_perm<2, 3, 0, 1>(r1).sub<2>(r1);  // P, R
    Fq29 f = o.c;
    bool same = false;
    const u32 zero = d.is_zero_modp() ? 1u : 0u;
    if (quad_perm<0, 0, 0, 0>(zero)) {
      if (!quad_perm<1, 1, 1, 1>(zero)) return identity();
      d = doubling_steps(q);
      r1 = c;
      f = Fq29::one();  // ZZ 1 and ZZZ 1: the doubled point's own
      same = true;
    }
    const Fq29 r2 = lane_pick(q < 2, d, c) * lane_pick(q < 2, d, f);  // PP, R^2, ZZ1 ZZ2, ZZZ1 ZZZ2
    return finish(d, r1, r2, r2, same, q);
  }

  // this + an affine point, xy as in from_affine (below 32p)
  __device__ __forceinline__ Quad29 add_affine(const Fq29& xy, bool inf, u32 q) const {
    if (inf) return *this;
    if (is_identity()) return from_affine(xy, q);
    Fq29 d = (xy * quad_perm<2, 3, 2, 3>(c)).sub<8>(c);  // U2 - X, S2 - Y (below 10p)
    bool same = false;
    const u32 zero = d.is_zero_modp() ? 1u : 0u;
    if (quad_perm<0, 0, 0, 0>(zero)) {
      if (!quad_perm<1, 1, 1, 1>(zero)) return identity();
      d = doubling_steps(q);
      same = true;
    }
    return finish(d, c, c, d * d, same, q);
  }
};

}  // namespace zkp
