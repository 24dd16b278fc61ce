// Field products spread over a row of lanes, for code that has one wave and a
// serial chain of formulas (the window combination of a multiexp).
//
// A row is 16 consecutive lanes (the unit of the DPP lane moves); lane k < 9
// holds limb k of an element on 29-bit limbs (field29.h: Montgomery form,
// radix 2^261) and lanes 9..15 hold 0.  A wave works on four products at a
// time.  In a product lane k sums column k: nine multiply-adds of a broadcast
// limb of a by b moved up the row, then as many for the reduction's digits
// (T mod 2^261 times -1/q mod 2^261, all digits at once) and for the digits
// times q.  Carries are not chained: a column above 29 bits hands its upper
// parts to the next two lanes once, and what is left once more, so limbs stay
// below 2^29 + 4 ("loose").  The low nine columns are a multiple of 2^261,
// whose quotient is read off the top three of them.
//
// About 110 instructions a product, against about 330 for one lane that
// computes the whole product in latency order: a wave that has its SIMD to
// itself issues one instruction every few cycles whatever it computes, so the
// instruction count is the time.
//
// Ranges.  For operands with limbs <= 2^29 + 4, a sum of products s gives a
// value below s / 2^261 + 1.001 q with limbs <= 2^29 + 3; up to four products
// of values whose sum s is below 169 q^2 give a value below 2q.  Column sums
// stay below 2^64 (4 * 9 * (2^29 + 4)^2 + 9 * 2^29 (2^29 + 2)).
#pragma once
#include "field.h"
#include "field29.h"

namespace csk {

// zero-padded so that lane k reads entry k - j of a constant at [8 + k - j]
__constant__ uint32_t kRowQ[24] = {0, 0, 0, 0, 0, 0, 0, 0, 410844487u, 17064118u, 477274959u, 47522512u, 361093496u,
                                   47923392u, 10936641u, 240920116u, 3171406u};
// -q^-1 mod 2^261
__constant__ uint32_t kRowNp[24] = {0, 0, 0, 0, 0, 0, 0, 0, 75916169u, 512769047u, 312128097u, 486197821u, 497551853u,
                                    99093529u, 296706751u, 384971025u, 267745826u};
// K q for K = 0, 2, 4, 6, 8, 10 with the low eight limbs raised by 2^30 (two
// units of the next limb): a - b is a + D - b, every limb >= 0 for b <= K q
// with limbs <= 2^30 - 2
__constant__ uint32_t kRowD[6][16] = {
    {0},
    {1358559886u, 1107870059u, 1491420828u, 1168786847u, 1259057902u, 1169588607u, 1095615104u, 1555582054u, 6342810u},
    {1106507036u, 1141998297u, 1372228922u, 1263831873u, 1444373982u, 1265435392u, 1117488386u, 1500551374u,
     12685623u},
    {1391325098u, 1176126534u, 1253037016u, 1358876899u, 1092819150u, 1361282178u, 1139361668u, 1445520694u,
     19028436u},
    {1139272248u, 1210254772u, 1133845110u, 1453921925u, 1278135230u, 1457128963u, 1161234950u, 1390490014u,
     25371249u},
    {1424090310u, 1244383009u, 1551524116u, 1548966950u, 1463451310u, 1552975748u, 1183108232u, 1335459334u,
     31714062u}};

// 2^256 mod q (to the 2^256 form)
__constant__ uint32_t kRowFrom[16] = {93261213u,  451550318u, 297979764u, 299258347u, 342016167u,
                                      297253948u, 482187706u, 406012155u, 920183u};

// lane moves within the row; lanes without a source take 0
template <int N> __device__ __forceinline__ uint32_t row_bcast(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x150 + N, 0xf, 0xf, true);
}
template <int N> __device__ __forceinline__ uint32_t row_up(uint32_t x) {  // lane k takes lane k - N
  if constexpr (N == 0) return x;
  else return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x110 + N, 0xf, 0xf, true);
}
template <int N> __device__ __forceinline__ uint32_t row_down(uint32_t x) {  // lane k takes lane k + N
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x100 + N, 0xf, 0xf, true);
}
template <int N> __device__ __forceinline__ uint64_t row_up64(uint64_t x) {
  return (uint64_t)row_up<N>((uint32_t)x) | ((uint64_t)row_up<N>((uint32_t)(x >> 32)) << 32);
}
template <int N> __device__ __forceinline__ uint64_t row_down64(uint64_t x) {
  return (uint64_t)row_down<N>((uint32_t)x) | ((uint64_t)row_down<N>((uint32_t)(x >> 32)) << 32);
}

// this lane's constants
struct RowK {
  uint32_t np[9], q[9];  // entries lane - j of -1/q and q
  uint32_t q8, m8;       // lane 8: q's top limb and all ones; 0 elsewhere
  __device__ __forceinline__ RowK() {
    const uint32_t k = threadIdx.x & 15;
#pragma unroll
    for (int j = 0; j < 9; j++) {
      np[j] = kRowNp[8 + k - j];
      q[j] = kRowQ[8 + k - j];
    }
    m8 = k == 8 ? 0xFFFFFFFFu : 0u;
    q8 = kRowQ[16] & m8;
  }
};

// column sums of a product being built: t of column `lane` (0..15), t16 of
// column 16 on lane 8
struct RowT {
  uint64_t t = 0, t16 = 0;
};

namespace row_detail {
template <int J> __device__ __forceinline__ void conv_step(RowT &s, uint32_t a, uint32_t b) {
  mad29(s.t, row_bcast<J>(a), row_up<J>(b));
  if constexpr (J < 8) conv_step<J + 1>(s, a, b);
}
template <int J> __device__ __forceinline__ void const_step(uint64_t &t, uint32_t a, const uint32_t (&c)[9]) {
  mad29(t, row_bcast<J>(a), c[J]);
  if constexpr (J < 8) const_step<J + 1>(t, a, c);
}
}  // namespace row_detail

__device__ __forceinline__ void row_conv(const RowK &k, RowT &s, uint32_t a, uint32_t b) {
  row_detail::conv_step<0>(s, a, b);
  mad29(s.t16, row_bcast<8>(a), b & k.m8);
}

// a column's parts above 29 and 58 bits to the next two lanes
__device__ __forceinline__ uint32_t row_carry64(uint64_t t) {
  const uint32_t l = (uint32_t)t & Q29::M, c1 = (uint32_t)(t >> 29) & Q29::M, c2 = (uint32_t)(t >> 58);
  return l + row_up<1>(c1) + row_up<2>(c2);
}
// limbs below 2^32 -> loose (top limb below 2^29)
__device__ __forceinline__ uint32_t row_norm(uint32_t x) { return (x & Q29::M) + row_up<1>(x >> 29); }

// Montgomery reduction of the column sums
__device__ __forceinline__ uint32_t row_redc(const RowK &k, RowT &s) {
  const uint32_t t = row_carry64(s.t);  // lanes 0..8: T mod 2^261
  uint64_t mm = 0;
  row_detail::const_step<0>(mm, t, k.np);
  const uint32_t m = row_norm(row_carry64(mm));  // lanes 0..8: the digits
  row_detail::const_step<0>(s.t, m, k.q);
  mad29(s.t16, row_bcast<8>(m), k.q8);
  // carry out of the low nine columns: column 8 plus what columns 7 and 6
  // hand up (low by at most one), whose exact sum is a multiple of 2^29
  const uint64_t x = s.t + row_up64<1>(s.t >> 29);
  const uint64_t c = (s.t + row_up64<1>(x >> 29) + 4) >> 29;
  const uint64_t c8 = (uint64_t)((uint32_t)c & k.m8) | ((uint64_t)((uint32_t)(c >> 32) & k.m8) << 32);
  // columns 9..16 move to lanes 0..7
  const uint64_t h = row_down64<9>(s.t) + row_down64<8>(c8) + row_down64<1>(s.t16);
  return row_norm(row_carry64(h));
}

__device__ __forceinline__ uint32_t row_mul(const RowK &k, uint32_t a, uint32_t b) {
  RowT s;
  row_conv(k, s, a, b);
  return row_redc(k, s);
}
__device__ __forceinline__ uint32_t row_dot(const RowK &k, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  RowT s;
  row_conv(k, s, a, b);
  row_conv(k, s, c, d);
  return row_redc(k, s);
}

// Exact limbs of a loose element (each round passes every carry one lane on)
__device__ __forceinline__ uint32_t row_exact(uint32_t x) {
#pragma unroll
  for (int i = 0; i < 9; i++) x = row_norm(x);
  return x;
}

// x in row 0 is 0 or q (x loose, below 2q): the same answer in every lane.
// The low limb is exact modulo 2^29, so the full comparison is rarely made.
__device__ __forceinline__ bool row_is_zero(uint32_t x) {
  const uint32_t l0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)x) & Q29::M;
  if (l0 != 0 && l0 != Q29::p[0]) return false;
  const uint32_t e = row_exact(x), k = threadIdx.x & 15;
  const uint64_t z = __ballot(e == 0), q = __ballot(e == kRowQ[8 + k]);
  return (z & 0xFFFF) == 0xFFFF || (q & 0xFFFF) == 0xFFFF;
}

// each row's element gathered into its lanes, exact limbs
__device__ __forceinline__ Fq29 row_gather(uint32_t x) {
  x = row_exact(x);
  return {{row_bcast<0>(x), row_bcast<1>(x), row_bcast<2>(x), row_bcast<3>(x), row_bcast<4>(x), row_bcast<5>(x),
           row_bcast<6>(x), row_bcast<7>(x), row_bcast<8>(x)}};
}

// an element held by every lane to the rows
__device__ __forceinline__ uint32_t row_scatter(const Fq29 &a) {
  const uint32_t k = threadIdx.x & 15;
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < 9; i++) r = k == (uint32_t)i ? a.l[i] : r;
  return r;
}
// canonical words of each row's element (below 2q)
__device__ __forceinline__ void row_words(uint32_t x, uint32_t (&w)[8]) { pack29(canon29(row_gather(x)), w); }
// words of 2^522 mod q: over a 2^261-form number, the 2^261 form of its inverse
struct Row522 {
  static constexpr uint32_t v[8] = {1704700944u, 3785531508u, 1409679450u, 1670927750u,
                                    759047730u,  4283745664u, 887776678u,  705799820u};
};
// the inverse of an element every row holds (2^261 form, below 2q, not 0)
__device__ __forceinline__ uint32_t row_inverse(uint32_t x) {
  uint32_t w[8], p[8], s[8], o[8];
  row_words(x, w);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    p[i] = FieldConst<0>::p[i];
    s[i] = Row522::v[i];
  }
  i30_inverse<true>(w, p, FieldConst<0>::np, o, s);
  return row_scatter(unpack29(o));
}

// rows 0, 2 hold one value and rows 1, 3 another: both in every row
__device__ __forceinline__ void row_spread2(uint32_t r, uint32_t &even, uint32_t &odd) {
  const auto s = __builtin_amdgcn_permlane16_swap(r, r, false, false);
  even = s[0];
  odd = s[1];
}
// four rows' values in every row
__device__ __forceinline__ void row_spread4(uint32_t r, uint32_t &r0, uint32_t &r1, uint32_t &r2, uint32_t &r3) {
  uint32_t e, o;
  row_spread2(r, e, o);
  const auto a = __builtin_amdgcn_permlane32_swap(e, e, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(o, o, false, false);
  r0 = a[0];
  r2 = a[1];
  r1 = b[0];
  r3 = b[1];
}

// ------------------------------------------------------------------ G1
// A point held by a wave, each coordinate in every row.  Ranges as the 29-bit
// slots: X < 8q, Y, ZZ, ZZZ < 2q.  The formulas are xdbl29's and xadd29's.
struct RowG1 {
  uint32_t X, Y, ZZ, ZZZ;
};
struct RowG1K : RowK {
  uint32_t d2, d4, d6, d8;
  bool odd, hi;  // rows 1, 3; rows 2, 3
  __device__ __forceinline__ RowG1K() {
    const uint32_t k = threadIdx.x & 15;
    d2 = kRowD[1][k];
    d4 = kRowD[2][k];
    d6 = kRowD[3][k];
    d8 = kRowD[4][k];
    odd = (threadIdx.x >> 4) & 1;
    hi = (threadIdx.x >> 5) & 1;
  }
  __device__ __forceinline__ uint32_t pick(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3) const {
    const uint32_t a = odd ? r1 : r0, b = odd ? r3 : r2;
    return hi ? b : a;
  }
};

// words s[0..9) of a 29-bit element to the rows
__device__ __forceinline__ uint32_t row_load(const uint32_t *s) {
  const uint32_t k = threadIdx.x & 15;
  return k < 9 ? s[k] : 0u;
}
__device__ __forceinline__ RowG1 row_load_g1(const uint32_t *s) {
  return {row_load(s), row_load(s + 9), row_load(s + 18), row_load(s + 27)};
}

// p = 2p (p not at infinity)
__device__ __forceinline__ void row_dbl(const RowG1K &k, RowG1 &p) {
  uint32_t V, xx, W, S, MM, ZZ3, Y3, ZZZ3;
  const uint32_t U = row_norm(p.Y << 1);  // < 4q
  const uint32_t a = k.odd ? p.X : U;
  row_spread2(row_mul(k, a, a), V, xx);
  const uint32_t M = row_norm(3 * xx);  // < 6q
  row_spread4(row_mul(k, k.pick(U, p.X, M, V), k.pick(V, V, M, p.ZZ)), W, S, MM, ZZ3);
  const uint32_t X3 = row_norm(MM + k.d4 - 2 * S);  // < 6q
  const uint32_t T = row_norm(S + k.d6 - X3), nY = row_norm(k.d2 - p.Y);
  // M T - W Y | W ZZZ
  row_spread2(row_dot(k, k.odd ? W : M, k.odd ? p.ZZZ : T, k.odd ? 0u : W, nY), Y3, ZZZ3);
  p = {X3, Y3, ZZ3, ZZZ3};
}

// p += q (neither at infinity); sets inf when q == -p
__device__ __forceinline__ void row_add(const RowG1K &k, RowG1 &p, const RowG1 &q, bool &inf) {
  uint32_t U1, U2, S1, S2, PP, RR, Z2, Z3, PPP, Qv, ZZ3, x, Y3, ZZZ3;
  row_spread4(row_mul(k, k.pick(p.X, q.X, p.Y, q.Y), k.pick(q.ZZ, p.ZZ, q.ZZZ, p.ZZZ)), U1, U2, S1, S2);
  const uint32_t P = row_norm(U2 + k.d2 - U1), R = row_norm(S2 + k.d2 - S1);  // < 4q
  row_spread4(row_mul(k, k.pick(P, R, p.ZZ, p.ZZZ), k.pick(P, R, q.ZZ, q.ZZZ)), PP, RR, Z2, Z3);
  if (row_is_zero(PP)) {
    if (row_is_zero(RR)) row_dbl(k, p);  // q == p
    else inf = true;                     // q == -p
    return;
  }
  row_spread4(row_mul(k, k.pick(P, U1, Z2, Z2), PP), PPP, Qv, ZZ3, x);
  const uint32_t X3 = row_norm(RR + k.d6 - row_norm(PPP + 2 * Qv));  // < 8q
  const uint32_t T = row_norm(Qv + k.d8 - X3), nP = row_norm(k.d2 - PPP);
  // R (Qv - X3) - S1 PPP | Z3 PPP
  row_spread2(row_dot(k, k.odd ? Z3 : R, k.odd ? PPP : T, k.odd ? 0u : S1, nP), Y3, ZZZ3);
  p = {X3, Y3, ZZ3, ZZZ3};
}

}  // namespace csk
