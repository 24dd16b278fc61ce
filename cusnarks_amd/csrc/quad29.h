// Point additions spread over four lanes, for the reductions that follow the
// bucket accumulation: long dependency chains with fewer additions than lanes.
//
// The lanes 4i .. 4i + 3 (a quad, the unit of the DPP quad_perm moves) hold the
// coordinates X, Y, ZZ, ZZZ of one point, one each, on 29-bit limbs (Fq29 for
// G1, Fq2_29 for G2) in the ranges of the stored slots (G1 X < 8q, G2 X < 4q
// per component, the rest < 2q).  An addition's 14 products then take four
// rounds, one product or one two-term sum per lane and round:
//   1  X1 ZZ2 | Y1 ZZZ2 | ZZ1 X2 | ZZZ1 Y2      = U1 | S1 | U2 | S2
//   2  P^2    | R^2     | ZZ1 ZZ2 | ZZZ1 ZZZ2   = PP | RR | Z2 | Z3
//   3  P PP   | U1 PP   | Z2 PP  |              = PPP | Qv | ZZ3 |
//   4         | R T - S1 PPP |   | Z3 PPP       =     | Y3 |    | ZZZ3
// with P = U2 - U1, R = S2 - S1, X3 = R^2 - PPP - 2 Qv and T = Qv - X3 (formed in
// the second lane).  A quad adds two points in about a third of the time one
// lane takes (about 1300 instructions against 3700 on G1) while the wave takes
// 1.4 times the instructions per addition, so it is the faster form until the
// additions in flight fill the SIMDs several waves deep.
#pragma once
#include "field29.h"

namespace csk {

// lane i of every quad takes lane (sel >> 2i) & 3
template <int SEL> __device__ __forceinline__ Fq29 quad_perm(const Fq29 &a) {
  Fq29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = (uint32_t)__builtin_amdgcn_mov_dpp((int)a.l[i], SEL, 0xf, 0xf, true);
  return r;
}
template <int SEL> __device__ __forceinline__ Fq2_29 quad_perm(const Fq2_29 &a) {
  return {quad_perm<SEL>(a.c0), quad_perm<SEL>(a.c1)};
}
constexpr int kQuadSwap = 0x4E;                                 // lane i <- i ^ 2
constexpr int kQuadB0 = 0x00, kQuadB1 = 0x55, kQuadB3 = 0xFF;  // broadcasts of lane 0, 1, 3

// the flag of lane `lane` of this lane's quad
__device__ __forceinline__ bool quad_flag(bool f, uint32_t lane) {
  return (__ballot(f) >> ((threadIdx.x & 60) + lane)) & 1;
}

__device__ __forceinline__ Fq29 qsel(bool c, const Fq29 &a, const Fq29 &b) {
  Fq29 r;
#pragma unroll
  for (int i = 0; i < 9; i++) r.l[i] = c ? a.l[i] : b.l[i];
  return r;
}
__device__ __forceinline__ Fq2_29 qsel(bool c, const Fq2_29 &a, const Fq2_29 &b) {
  return {qsel(c, a.c0, b.c0), qsel(c, a.c1, b.c1)};
}

// The field steps the formulas are written in, for Fq and Fq2 (ranges per
// component).  kX is the bound on X in units of q.
template <class T> struct QuadX;
template <> struct QuadX<Fq29> { static constexpr int kX = 8; };
template <> struct QuadX<Fq2_29> { static constexpr int kX = 4; };
__device__ __forceinline__ Fq29 qmul(const Fq29 &a, const Fq29 &b) { return mul29_2c(a, b); }
__device__ __forceinline__ Fq2_29 qmul(const Fq2_29 &a, const Fq2_29 &b) {  // b <= 6q
  return f2mul29(a, b, sub29<6>(Fq29{}, b.c1));
}
template <int K> __device__ __forceinline__ Fq29 qsub(const Fq29 &a, const Fq29 &b) { return sub29<K>(a, b); }
template <int K> __device__ __forceinline__ Fq2_29 qsub(const Fq2_29 &a, const Fq2_29 &b) { return f2sub29<K>(a, b); }
template <int k> __device__ __forceinline__ Fq29 qadd(const Fq29 &a, const Fq29 &b) { return add29<k>(a, b); }
template <int k> __device__ __forceinline__ Fq2_29 qadd(const Fq2_29 &a, const Fq2_29 &b) {
  return {add29<k>(a.c0, b.c0), add29<k>(a.c1, b.c1)};
}
__device__ __forceinline__ bool qzero(const Fq29 &a) { return is_zero29(a); }
__device__ __forceinline__ bool qzero(const Fq2_29 &a) { return is_zero2_29(a); }
// a value below 8q to the stored range of X
__device__ __forceinline__ Fq29 qx(const Fq29 &a) { return a; }
__device__ __forceinline__ Fq2_29 qx(const Fq2_29 &a) { return {csub29(a.c0, Q29::p4), csub29(a.c1, Q29::p4)}; }
// a b + c (2q - d) in one reduction (c, d <= 2q; G2 b <= 6q)
__device__ __forceinline__ Fq29 qdot(const Fq29 &a, const Fq29 &b, const Fq29 &c, const Fq29 &d) {
  return dot29(a, b, c, sub29<2>(Fq29{}, d));
}
__device__ __forceinline__ Fq2_29 qdot(const Fq2_29 &a, const Fq2_29 &b, const Fq2_29 &c, const Fq2_29 &d) {
  const Fq29 nb1 = sub29<6>(Fq29{}, b.c1), nd0 = sub29<2>(Fq29{}, d.c0), nd1 = sub29<2>(Fq29{}, d.c1);
  Fq2_29 r;
  dot4x2(a.c0, b.c0, a.c1, nb1, c.c0, nd0, c.c1, d.c1, a.c0, b.c1, a.c1, b.c0, c.c0, nd1, c.c1, nd0, r.c0, r.c1);
  return r;
}

// a = 2a (dbl-2008-s), a not at infinity.  Products below 72 q^2.
template <class T> __device__ __forceinline__ void quad_dbl(T &a) {
  const uint32_t c = threadIdx.x & 3;
  const T u = qsel(c == 1, qadd<1>(a, a), a);  // X | U = 2Y < 4q | ZZ | ZZZ
  const T r1 = qmul(u, u);                      // xx | V
  const T xx = quad_perm<kQuadB0>(r1), V = quad_perm<kQuadB1>(r1);
  const T M = qadd<2>(xx, xx);                                // < 6q
  const T r2 = qmul(qsel(c == 3, M, u), qsel(c == 3, M, V));  // S = X V | W = U V | ZZ3 | M^2
  const T S = quad_perm<kQuadB0>(r2), W = quad_perm<kQuadB1>(r2), MM = quad_perm<kQuadB3>(r2);
  const T X3 = qx(qsub<4>(MM, qadd<1>(S, S)));  // < 6q, G2 < 4q
  const T Tv = qsub<QuadX<T>::kX>(S, X3);       // G1 < 10q, G2 < 6q
  // Y3 = M T - W Y in lane 1; ZZZ3 = ZZZ W (and W times 0) in lane 3
  const T r3 = qdot(qsel(c == 3, a, M), qsel(c == 3, W, Tv), W, qsel(c == 3, T{}, a));
  a = qsel(c == 0, X3, qsel(c == 2, r2, r3));
}

// a += b (add-2008-s), either may be at infinity (ZZ = 0 mod q)
template <class T> __device__ __forceinline__ void quad_add(T &a, const T &b) {
  const uint32_t c = threadIdx.x & 3;
  const bool za = quad_flag(qzero(a), 2), zb = quad_flag(qzero(b), 2);
  if (__all(zb)) return;
  const T p = qmul(a, quad_perm<kQuadSwap>(b));           // U1 | S1 | U2 | S2
  const T d = qsub<2>(quad_perm<kQuadSwap>(p), p);        // P | R (< 4q)
  const T r2 = qmul(qsel(c < 2, d, a), qsel(c < 2, d, b));  // PP | RR | Z2 | Z3
  const bool zp = qzero(r2);
  const bool same_x = quad_flag(zp, 0), same_y = quad_flag(zp, 1);
  const T PP = quad_perm<kQuadB0>(r2), U1 = quad_perm<kQuadB0>(p);
  const T r3 = qmul(qsel(c == 0, d, qsel(c == 1, U1, r2)), PP);  // PPP | Qv | ZZ3
  const T PPP = quad_perm<kQuadB0>(r3);
  const T X3 = qx(qsub<6>(r2, qadd<2>(PPP, r3)));  // lane 1: < 8q, G2 < 4q
  const T Tv = qsub<QuadX<T>::kX>(r3, X3);         // lane 1: G1 < 10q, G2 < 6q
  // Y3 = R T - S1 PPP in lane 1; ZZZ3 = Z3 PPP (and S2 times 0) in lane 3
  const T r4 = qdot(qsel(c == 3, r2, d), qsel(c == 3, PPP, Tv), p, qsel(c == 3, T{}, PPP));
  const T s = qsel(c == 0, quad_perm<kQuadB1>(X3), qsel(c == 2, r3, r4));
  const bool special = same_x && !za && !zb;
  T sp = a;
  if (__any(special)) {  // equal points double, opposite ones cancel
    T dd = a;
    quad_dbl(dd);
    sp = qsel(same_y, dd, T{});
  }
  a = qsel(zb, a, qsel(za, b, qsel(special, sp, s)));
}

// coordinate words of a stored slot (36 / 72 words: X, Y, ZZ, ZZZ, components in
// turn)
__device__ __forceinline__ void quad_load(const uint32_t *slot, Fq29 &a) {
  const uint32_t *s = slot + 9 * (threadIdx.x & 3);
#pragma unroll
  for (int i = 0; i < 9; i++) a.l[i] = s[i];
}
__device__ __forceinline__ void quad_load(const uint32_t *slot, Fq2_29 &a) {
  const uint32_t *s = slot + 18 * (threadIdx.x & 3);
#pragma unroll
  for (int i = 0; i < 9; i++) {
    a.c0.l[i] = s[i];
    a.c1.l[i] = s[9 + i];
  }
}
__device__ __forceinline__ void quad_store(uint32_t *slot, const Fq29 &a) {
  uint32_t *s = slot + 9 * (threadIdx.x & 3);
#pragma unroll
  for (int i = 0; i < 9; i++) s[i] = a.l[i];
}
__device__ __forceinline__ void quad_store(uint32_t *slot, const Fq2_29 &a) {
  uint32_t *s = slot + 18 * (threadIdx.x & 3);
#pragma unroll
  for (int i = 0; i < 9; i++) {
    s[i] = a.c0.l[i];
    s[9 + i] = a.c1.l[i];
  }
}

}  // namespace csk
