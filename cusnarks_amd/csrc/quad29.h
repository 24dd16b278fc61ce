// Point additions spread over a group of lanes, for the reductions that follow
// the bucket accumulation: long dependency chains with fewer additions than
// lanes.
//
// G1: the lanes 4i .. 4i + 3 (a quad, the unit of the DPP quad_perm moves) hold
// the coordinates X, Y, ZZ, ZZZ of one point, one each, on 29-bit limbs in the
// ranges of the stored slots (G1 X < 8q, G2 X < 4q per component, the rest < 2q).
// An addition's 14 products then take four rounds, one product or one two-term
// sum per lane and round:
//   1  X1 ZZ2 | Y1 ZZZ2 | ZZ1 X2 | ZZZ1 Y2      = U1 | S1 | U2 | S2
//   2  P^2    | R^2     | ZZ1 ZZ2 | ZZZ1 ZZZ2   = PP | RR | Z2 | Z3
//   3  P PP   | U1 PP   | Z2 PP  |              = PPP | Qv | ZZ3 |
//   4         | R T - S1 PPP |   | Z3 PPP       =     | Y3 |    | ZZZ3
// with P = U2 - U1, R = S2 - S1, X3 = R^2 - PPP - 2 Qv and T = Qv - X3 (formed in
// the second lane).  G2: eight lanes, the quad of the c0 components in this order
// and that of the c1 components mirrored (lane i and lane 7 - i hold the two
// components of a coordinate, so the partner is one half-row mirror away); each
// lane forms its component of the round's Fq2 product in one reduction.
//
// A quad adds two G1 points in about 1300 instructions, where one lane takes
// about 3700, while the wave takes 1.4 times the instructions per addition, so it
// is the faster form until the additions in flight fill the SIMDs several waves
// deep.  Eight lanes add two G2 points in about 2200 instructions (one lane: about
// 9500; four lanes of both components: 5100).
#pragma once
#include "field.h"
#include "field29.h"

namespace csk {

template <int CTRL, int BANKS> __device__ __forceinline__ void grp_move(Fq29 &r, const Fq29 &a) {
#pragma unroll
  for (int i = 0; i < 9; i++)
    r.l[i] = BANKS == 0xf ? (uint32_t)__builtin_amdgcn_mov_dpp((int)a.l[i], CTRL, 0xf, 0xf, true)
                          : (uint32_t)__builtin_amdgcn_update_dpp((int)r.l[i], (int)a.l[i], CTRL, 0xf, BANKS, true);
}
__device__ __forceinline__ Fq29 grp_sel(bool c, const Fq29 &a, const Fq29 &b) {
  Fq29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = c ? a.l[i] : b.l[i];
  return r;
}

// The field steps the formulas are written in.  coord: which of X, Y, ZZ, ZZZ
// this lane holds; swap: coordinate i takes i ^ 2; all<c>: every lane takes
// coordinate c; kX: the bound on X in units of q.
template <class F> struct Grp;

template <> struct Grp<Fq> {
  static constexpr int N = 4, kX = 8;
  __device__ __forceinline__ static uint32_t coord() { return threadIdx.x & 3; }
  __device__ __forceinline__ static uint32_t word() { return 9 * (threadIdx.x & 3); }  // of the slot
  __device__ __forceinline__ static Fq29 swap(const Fq29 &a) {
    Fq29 r;
    grp_move<0x4E, 0xf>(r, a);
    return r;
  }
  template <int C> __device__ __forceinline__ static Fq29 all(const Fq29 &a) {
    Fq29 r;
    grp_move<C * 0x55, 0xf>(r, a);
    return r;
  }
  // f holds for coordinate c of this lane's point
  __device__ __forceinline__ static bool flag(bool f, uint32_t c) {
    return (__ballot(f) >> ((threadIdx.x & 60) + c)) & 1;
  }
  __device__ __forceinline__ static Fq29 mul(const Fq29 &a, const Fq29 &b) { return mul29_2c(a, b); }
  // a b + c (2q - d) in one reduction
  __device__ __forceinline__ static Fq29 dot(const Fq29 &a, const Fq29 &b, const Fq29 &c, const Fq29 &d) {
    return dot29(a, b, c, sub29<2>(Fq29{}, d));
  }
  __device__ __forceinline__ static Fq29 stored_x(const Fq29 &a) { return a; }
};

template <> struct Grp<Fq2> {
  static constexpr int N = 8, kX = 4;
  __device__ __forceinline__ static bool c1() { return threadIdx.x & 4; }
  __device__ __forceinline__ static uint32_t coord() { return (threadIdx.x & 3) ^ (c1() ? 3 : 0); }
  __device__ __forceinline__ static uint32_t word() { return 18 * coord() + (c1() ? 9 : 0); }
  __device__ __forceinline__ static Fq29 swap(const Fq29 &a) {
    Fq29 r;
    grp_move<0x4E, 0xf>(r, a);
    return r;
  }
  template <int C> __device__ __forceinline__ static Fq29 all(const Fq29 &a) {
    Fq29 r;
    grp_move<C * 0x55, 0xf>(r, a);
    grp_move<(3 - C) * 0x55, 0xA>(r, a);  // the mirrored quads
    return r;
  }
  __device__ __forceinline__ static bool flag(bool f, uint32_t c) {
    const uint64_t b = __ballot(f) >> (threadIdx.x & 56);
    return (b >> c) & (b >> (7 - c)) & 1;
  }
  // the other component of the same coordinate
  __device__ __forceinline__ static Fq29 other(const Fq29 &a) {
    Fq29 r;
    grp_move<0x141, 0xf>(r, a);
    return r;
  }
  // c0 = a0 b0 + a1 (6q - b1), c1 = a1 b0 + a0 b1 (b < 5.9q)
  __device__ __forceinline__ static Fq29 mul(const Fq29 &a, const Fq29 &b) {
    const bool c = c1();
    const Fq29 ao = other(a), bo = other(b);
    return dot29(grp_sel(c, ao, a), b, grp_sel(c, a, ao), grp_sel(c, bo, neg29_loose<6>(bo)));
  }
  // a b + c (2q - d) in one reduction (columns below (3 * 4.5 + 2 * 9) 2^59)
  __device__ __forceinline__ static Fq29 dot(const Fq29 &a, const Fq29 &b, const Fq29 &c, const Fq29 &d) {
    const bool h = c1();
    const Fq29 ao = other(a), bo = other(b), co = other(c), dd = other(d);
    return dot4_29(grp_sel(h, ao, a), b, grp_sel(h, a, ao), grp_sel(h, bo, sub29<6>(Fq29{}, bo)), grp_sel(h, co, c),
                   neg29_loose<2>(d), grp_sel(h, c, co), grp_sel(h, neg29_loose<2>(dd), dd));
  }
  __device__ __forceinline__ static Fq29 stored_x(const Fq29 &a) { return csub29(a, Q29::p4); }
};

// a = 2a (dbl-2008-s), a not at infinity.  Products below 72 q^2.
template <class F> __device__ __forceinline__ void grp_dbl(Fq29 &a) {
  using G = Grp<F>;
  const uint32_t c = G::coord();
  const Fq29 u = grp_sel(c == 1, add29<1>(a, a), a);  // X | U = 2Y < 4q | ZZ | ZZZ
  const Fq29 r1 = G::mul(u, u);                        // xx | V
  const Fq29 xx = G::template all<0>(r1), V = G::template all<1>(r1);
  const Fq29 M = add29<2>(xx, xx);                                        // < 6q
  const Fq29 r2 = G::mul(grp_sel(c == 3, M, u), grp_sel(c == 3, M, V));  // S = X V | W = U V | ZZ3 | M^2
  const Fq29 S = G::template all<0>(r2), W = G::template all<1>(r2), MM = G::template all<3>(r2);
  const Fq29 X3 = G::stored_x(sub29<4>(MM, add29<1>(S, S)));  // < 6q, G2 < 4q
  const Fq29 Tv = sub29<G::kX>(S, X3);                         // G1 < 10q, G2 < 6q
  // Y3 = M T - W Y in lane 1; ZZZ3 = ZZZ W (and W times 0) in lane 3
  const Fq29 r3 = G::dot(grp_sel(c == 3, a, M), grp_sel(c == 3, W, Tv), W, grp_sel(c == 1, a, Fq29{}));
  a = grp_sel(c == 0, X3, grp_sel(c == 2, r2, r3));
}

// a += b (add-2008-s), either may be at infinity (ZZ = 0 mod q)
template <class F> __device__ __forceinline__ void grp_add(Fq29 &a, const Fq29 &b) {
  using G = Grp<F>;
  const uint32_t c = G::coord();
  const bool za = G::flag(is_zero29(a), 2), zb = G::flag(is_zero29(b), 2);
  if (__all(zb)) return;
  const Fq29 p = G::mul(a, G::swap(b));                              // U1 | S1 | U2 | S2
  const Fq29 d = sub29<2>(G::swap(p), p);                            // P | R (< 4q)
  const Fq29 r2 = G::mul(grp_sel(c < 2, d, a), grp_sel(c < 2, d, b));  // PP | RR | Z2 | Z3
  const bool zp = is_zero29(r2);
  const bool same_x = G::flag(zp, 0), same_y = G::flag(zp, 1);
  const Fq29 PP = G::template all<0>(r2), U1 = G::template all<0>(p);
  const Fq29 r3 = G::mul(grp_sel(c == 0, d, grp_sel(c == 1, U1, r2)), PP);  // PPP | Qv | ZZ3
  const Fq29 PPP = G::template all<0>(r3);
  const Fq29 X3 = G::stored_x(sub29<6>(r2, add29<2>(PPP, r3)));  // lane 1: < 8q, G2 < 4q
  const Fq29 Tv = sub29<G::kX>(r3, X3);                           // lane 1: G1 < 10q, G2 < 6q
  // Y3 = R T - S1 PPP in lane 1; ZZZ3 = Z3 PPP (and S2 times 0) in lane 3
  const Fq29 r4 = G::dot(grp_sel(c == 3, r2, d), grp_sel(c == 3, PPP, Tv), p, grp_sel(c == 3, Fq29{}, PPP));
  const Fq29 s = grp_sel(c == 0, G::template all<1>(X3), grp_sel(c == 2, r3, r4));
  const bool special = same_x && !za && !zb;
  Fq29 sp = a;
  if (__any(special)) {  // equal points double, opposite ones cancel
    Fq29 dd = a;
    grp_dbl<F>(dd);
    sp = grp_sel(same_y, dd, Fq29{});
  }
  a = grp_sel(zb, a, grp_sel(za, b, grp_sel(special, sp, s)));
}

// this lane's words of a stored slot
template <class F> __device__ __forceinline__ void grp_load(const uint32_t *slot, Fq29 &a) {
  const uint32_t *s = slot + Grp<F>::word();
#pragma unroll
  for (int i = 0; i < 9; i++) a.l[i] = s[i];
}
template <class F> __device__ __forceinline__ void grp_store(uint32_t *slot, const Fq29 &a) {
  uint32_t *s = slot + Grp<F>::word();
#pragma unroll
  for (int i = 0; i < 9; i++) s[i] = a.l[i];
}

}  // namespace csk
