// The G2 window combination (the serial Horner chain that closes a multiexp):
// point formulas over Fq2 as programs that a workgroup of sixteen rows of
// lanes runs (row29.h: a row of 16 lanes holds one 9-limb element and forms
// one product at a time).
//
// Every value of a formula lives in an LDS slot (one Fq component, limb k at
// word k).  A formula is a program of rounds; in a round, row i executes
// operation i (a one-reduction sum of two or four products, or sums and
// differences), reading its operands from slots and writing its result to a
// slot, and the round ends with a barrier.  The independent products of a step
// thus run on different rows at once.  A round keeps to one class of
// operations (sums, products, four-term products, or the chain from X3 to the
// products of Y3), so the rows of a wave do not take turns.
//
// Ranges: X < 8q per component, Y, ZZ, ZZZ < 2q; each operation's bound is
// noted in its program.
#pragma once
#include "curve.h"
#include "row29.h"

namespace csk {

enum : uint8_t {
  // sums and differences
  C29_COPY,   // d = a0
  C29_ADD1,   // d = a0 + a1
  C29_SUB2,   // d = a0 + 2q - a1
  C29_SUB8,   // d = a0 + 8q - a1
  C29_SUB4D,  // d = a0 + 4q - 2 a1
  C29_NSUB,   // d = 4q - (a0 + 2q - a1)
  // products
  C29_DOT,    // d = a0 a1 + a2 a3
  C29_DOTN,   // d = a0 a1 + a2 a3; a4 = 2q - d
  C29_DOTM,   // d = 3 (a0 a1 + a2 a3)
  C29_DOTMN,  // d = 3 (a0 a1 + a2 a3); a4 = 6q - d
  C29_DOT4,   // d = a0 a1 + a2 a3 + a4 a5 + a6 a7
  // the chain of a doubling (a0 = MM, a1 = S): each row computes it whole
  C29_X3D,    // d = x = a0 + 4q - 2 a1
  C29_TD,     // d = t = a1 + 6q - x
  C29_NTD,    // d = 8q - t
  // the chain of an addition (a0 = RR, a1 = PPP, a2 = Qv)
  C29_X3A,    // d = x = a0 + 6q - (a1 + 2 a2)
  C29_TA,     // d = t = a2 + 8q - x
  C29_NTA,    // d = 10q - t
};
struct C29Op {
  uint8_t k, d, a[8];
};

namespace {  // programs (one copy per translation unit)

// ---- G2: acc components X0 X1 Y0 Y1 ZZ0 ZZ1 ZZZ0 ZZZ1 in 0-7, addend in
// 8-15, zero in 16.  An Fq2 product is two reductions: c0 = a0 b0 + a1 (Kq -
// b1), c1 = a0 b1 + a1 b0 (squares too, with the negated a1).
enum : uint8_t { H_X0, H_X1, H_Y0, H_Y1, H_ZZ0, H_ZZ1, H_ZZZ0, H_ZZZ1,
                 H_QX0, H_QX1, H_QY0, H_QY1, H_QZZ0, H_QZZ1, H_QZZZ0, H_QZZZ1, H_ZERO };

// 2 acc: U = 2Y < 4q; V = U^2 (32 q^2), xx = X^2 (128 q^2); M = 3 xx < 6q; M^2
// (72 q^2); X3 = M^2 - 2S < 6q; T = S - X3 < 8q; Y3 = M T - W Y (104 q^2)
enum : uint8_t { D2_U0 = 17, D2_U1, D2_NY0, D2_NY1, D2_NZZ1, D2_NZZZ1, D2_NX1, D2_NU1, D2_V0, D2_V1, D2_XX0, D2_XX1,
                 D2_M0, D2_M1, D2_NV1, D2_NM1, D2_W0, D2_W1, D2_S0, D2_S1, D2_MM0, D2_MM1, D2_ZZ30, D2_ZZ31,
                 D2_S20, D2_S21, D2_X30, D2_X31, D2_T0, D2_T1, D2_NT1, D2_Y30, D2_Y31, D2_ZZZ30, D2_ZZZ31,
                 D2_OY1, D2_OZZZ0, D2_OZZZ1 };
// The last rounds write the accumulator slots in place (X3 and ZZ3 once no
// later round reads the old X and ZZ, Y3 and ZZZ3 from copies of the old
// Y1, ZZZ0, ZZZ1 taken in the first round), so no round of copies follows.
__constant__ C29Op kG2Dbl[] = {
    {C29_ADD1, D2_U0, {H_Y0, H_Y0}}, {C29_ADD1, D2_U1, {H_Y1, H_Y1}}, {C29_SUB2, D2_NY0, {H_ZERO, H_Y0}},
    {C29_SUB2, D2_NY1, {H_ZERO, H_Y1}}, {C29_SUB2, D2_NZZ1, {H_ZERO, H_ZZ1}}, {C29_SUB2, D2_NZZZ1, {H_ZERO, H_ZZZ1}},
    {C29_SUB8, D2_NX1, {H_ZERO, H_X1}}, {C29_SUB4D, D2_NU1, {H_ZERO, H_Y1}},  // 4q - U1
    {C29_COPY, D2_OY1, {H_Y1}}, {C29_COPY, D2_OZZZ0, {H_ZZZ0}}, {C29_COPY, D2_OZZZ1, {H_ZZZ1}},
    // V = U^2 (and 2q - V1); M = 3 X^2 (and 6q - M1)
    {C29_DOT, D2_V0, {D2_U0, D2_U0, D2_U1, D2_NU1}}, {C29_DOTN, D2_V1, {D2_U0, D2_U1, D2_U1, D2_U0, D2_NV1}},
    {C29_DOTM, D2_M0, {H_X0, H_X0, H_X1, D2_NX1}}, {C29_DOTMN, D2_M1, {H_X0, H_X1, H_X1, H_X0, D2_NM1}},
    {C29_DOT, D2_W0, {D2_U0, D2_V0, D2_U1, D2_NV1}}, {C29_DOT, D2_W1, {D2_U0, D2_V1, D2_U1, D2_V0}},
    {C29_DOT, D2_S0, {H_X0, D2_V0, H_X1, D2_NV1}},   {C29_DOT, D2_S1, {H_X0, D2_V1, H_X1, D2_V0}},
    {C29_DOT, D2_MM0, {D2_M0, D2_M0, D2_M1, D2_NM1}}, {C29_DOT, D2_MM1, {D2_M0, D2_M1, D2_M1, D2_M0}},
    {C29_DOT, D2_ZZ30, {D2_V0, H_ZZ0, D2_V1, D2_NZZ1}}, {C29_DOT, D2_ZZ31, {D2_V0, H_ZZ1, D2_V1, H_ZZ0}},
    // X3 = MM - 2S < 6q; T = S - X3 < 8q; 8q - T1
    {C29_X3D, H_X0, {D2_MM0, D2_S0}}, {C29_X3D, H_X1, {D2_MM1, D2_S1}},
    {C29_TD, D2_T0, {D2_MM0, D2_S0}},   {C29_TD, D2_T1, {D2_MM1, D2_S1}},
    {C29_NTD, D2_NT1, {D2_MM1, D2_S1}}, {C29_COPY, H_ZZ0, {D2_ZZ30}}, {C29_COPY, H_ZZ1, {D2_ZZ31}},
    // ZZZ3 as four-term sums with two zero terms: the same column sums as
    // C29_DOT, so the same result, and the round runs one operation kind
    {C29_DOT4, H_Y0, {D2_M0, D2_T0, D2_M1, D2_NT1, D2_W0, D2_NY0, D2_W1, D2_OY1}},
    {C29_DOT4, H_Y1, {D2_M0, D2_T1, D2_M1, D2_T0, D2_W0, D2_NY1, D2_W1, D2_NY0}},
    {C29_DOT4, H_ZZZ0, {D2_W0, D2_OZZZ0, D2_W1, D2_NZZZ1, H_ZERO, H_ZERO, H_ZERO, H_ZERO}},
    {C29_DOT4, H_ZZZ1, {D2_W0, D2_OZZZ1, D2_W1, D2_OZZZ0, H_ZERO, H_ZERO, H_ZERO, H_ZERO}},
};
__constant__ uint8_t kG2DblR[] = {11, 4, 8, 7, 4};

// acc + q, part 1: U1 = X qZZ, U2 = qX ZZ, S1 = Y qZZZ, S2 = qY ZZZ, ZZ qZZ,
// ZZZ qZZZ (16 q^2 each); P, R < 4q; PP, RR (32 q^2)
enum : uint8_t { E_NQZZ1 = 17, E_NQZZZ1, E_NZZ1, E_NZZZ1, E_U10, E_U11, E_U20, E_U21, E_S10, E_S11, E_S20, E_S21,
                 E_Z20, E_Z21, E_Z30, E_Z31, E_P0, E_P1, E_R0, E_R1, E_NP1, E_NR1, E_PP0, E_PP1, E_RR0, E_RR1,
                 E_NPP1, E_PPP0, E_PPP1, E_QV0, E_QV1, E_ZZ30, E_ZZ31, E_NPPP1, E_NP0, E_T10, E_T11, E_X30, E_X31,
                 E_T0, E_T1, E_NT1, E_Y30, E_Y31, E_ZZZ30, E_ZZZ31, E_NSLOT };
__constant__ C29Op kG2Add1[] = {
    {C29_SUB2, E_NQZZ1, {H_ZERO, H_QZZ1}}, {C29_SUB2, E_NQZZZ1, {H_ZERO, H_QZZZ1}},
    {C29_SUB2, E_NZZ1, {H_ZERO, H_ZZ1}},   {C29_SUB2, E_NZZZ1, {H_ZERO, H_ZZZ1}},
    {C29_DOT, E_U10, {H_X0, H_QZZ0, H_X1, E_NQZZ1}},     {C29_DOT, E_U11, {H_X0, H_QZZ1, H_X1, H_QZZ0}},
    {C29_DOT, E_U20, {H_QX0, H_ZZ0, H_QX1, E_NZZ1}},     {C29_DOT, E_U21, {H_QX0, H_ZZ1, H_QX1, H_ZZ0}},
    {C29_DOT, E_S10, {H_Y0, H_QZZZ0, H_Y1, E_NQZZZ1}},   {C29_DOT, E_S11, {H_Y0, H_QZZZ1, H_Y1, H_QZZZ0}},
    {C29_DOT, E_S20, {H_QY0, H_ZZZ0, H_QY1, E_NZZZ1}},   {C29_DOT, E_S21, {H_QY0, H_ZZZ1, H_QY1, H_ZZZ0}},
    {C29_DOT, E_Z20, {H_ZZ0, H_QZZ0, H_ZZ1, E_NQZZ1}},   {C29_DOT, E_Z21, {H_ZZ0, H_QZZ1, H_ZZ1, H_QZZ0}},
    {C29_DOT, E_Z30, {H_ZZZ0, H_QZZZ0, H_ZZZ1, E_NQZZZ1}}, {C29_DOT, E_Z31, {H_ZZZ0, H_QZZZ1, H_ZZZ1, H_QZZZ0}},
    {C29_SUB2, E_P0, {E_U20, E_U10}}, {C29_SUB2, E_P1, {E_U21, E_U11}},
    {C29_SUB2, E_R0, {E_S20, E_S10}}, {C29_SUB2, E_R1, {E_S21, E_S11}},
    {C29_NSUB, E_NP1, {E_U21, E_U11}}, {C29_NSUB, E_NR1, {E_S21, E_S11}},  // 4q - P1, 4q - R1
    {C29_DOT, E_PP0, {E_P0, E_P0, E_P1, E_NP1}}, {C29_DOT, E_PP1, {E_P0, E_P1, E_P1, E_P0}},
    {C29_DOT, E_RR0, {E_R0, E_R0, E_R1, E_NR1}}, {C29_DOT, E_RR1, {E_R0, E_R1, E_R1, E_R0}},
};
__constant__ uint8_t kG2Add1R[] = {4, 12, 6, 4};
// part 2: PPP, Qv, ZZ3 (16 q^2); X3 = RR - PPP - 2Qv < 8q; T = Qv - X3 < 10q;
// Y3 = R T - S1 PPP (88 q^2); ZZZ3
__constant__ C29Op kG2Add2[] = {
    {C29_SUB2, E_NPP1, {H_ZERO, E_PP1}},
    {C29_DOT, E_PPP0, {E_P0, E_PP0, E_P1, E_NPP1}},  {C29_DOT, E_PPP1, {E_P0, E_PP1, E_P1, E_PP0}},
    {C29_DOT, E_QV0, {E_U10, E_PP0, E_U11, E_NPP1}}, {C29_DOT, E_QV1, {E_U10, E_PP1, E_U11, E_PP0}},
    {C29_DOT, E_ZZ30, {E_Z20, E_PP0, E_Z21, E_NPP1}}, {C29_DOT, E_ZZ31, {E_Z20, E_PP1, E_Z21, E_PP0}},
    {C29_SUB2, E_NPPP1, {H_ZERO, E_PPP1}}, {C29_SUB2, E_NP0, {H_ZERO, E_PPP0}},
    {C29_X3A, H_X0, {E_RR0, E_PPP0, E_QV0}}, {C29_X3A, H_X1, {E_RR1, E_PPP1, E_QV1}},  // in place, as in kG2Dbl
    {C29_TA, E_T0, {E_RR0, E_PPP0, E_QV0}},   {C29_TA, E_T1, {E_RR1, E_PPP1, E_QV1}},
    {C29_NTA, E_NT1, {E_RR1, E_PPP1, E_QV1}}, {C29_COPY, H_ZZ0, {E_ZZ30}}, {C29_COPY, H_ZZ1, {E_ZZ31}},
    {C29_DOT4, H_Y0, {E_R0, E_T0, E_R1, E_NT1, E_S10, E_NP0, E_S11, E_PPP1}},
    {C29_DOT4, H_Y1, {E_R0, E_T1, E_R1, E_T0, E_S10, E_NPPP1, E_S11, E_NP0}},
    {C29_DOT4, H_ZZZ0, {E_Z30, E_PPP0, E_Z31, E_NPPP1, H_ZERO, H_ZERO, H_ZERO, H_ZERO}},
    {C29_DOT4, H_ZZZ1, {E_Z30, E_PPP1, E_Z31, E_PPP0, H_ZERO, H_ZERO, H_ZERO, H_ZERO}},
};
__constant__ uint8_t kG2Add2R[] = {1, 6, 2, 7, 4};

}  // namespace

// The interpreter.  Slot s is at words [16 s, 16 s + 16): limb k at word k, zeros
// above.  The biases K q of the differences are slots of their own after the
// formulas' (D index = K / 2).  Every row of a workgroup of kRows rows takes
// part; row i of a round with more than i operations executes operation i.
template <class F> struct Coop29;
template <> struct Coop29<Fq2> {
  static constexpr int NC = 8;
  static constexpr int kRows = 16;
  static constexpr int kForm = E_NSLOT > D2_OZZZ1 + 1 ? E_NSLOT : D2_OZZZ1 + 1;
  static constexpr int kSlots = kForm + 6;

  // One row's operation of a round, as word offsets of its lane: fetched once
  // for the rounds of the doubling, which run back to back.
  struct Op {
    uint32_t k = 0;
    uint32_t d = 0, a[8] = {};
    bool live = false;
    __device__ __forceinline__ void fetch(const C29Op *ops, uint32_t off, uint32_t n) {
      const uint32_t row = threadIdx.x >> 4, lane = threadIdx.x & 15;
      live = row < n;
      const C29Op o = ops[off + (live ? row : 0)];
      k = o.k;
      d = 16u * o.d + lane;
#pragma unroll
      for (int i = 0; i < 8; i++) a[i] = 16u * o.a[i] + lane;
    }
  };
  RowK rk;
  Op dbl_op[5];
  uint32_t *sh;

  // sh: kSlots * 16 words, zeroed here but for the biases
  __device__ __forceinline__ explicit Coop29(uint32_t *lds) : sh(lds) {
    for (uint32_t i = threadIdx.x; i < kSlots * 16; i += blockDim.x)
      sh[i] = i < kForm * 16 ? 0u : kRowD[i / 16 - kForm][i & 15];
    uint32_t off = 0;
#pragma unroll
    for (int r = 0; r < 5; r++) {
      dbl_op[r].fetch(kG2Dbl, off, kG2DblR[r]);
      off += kG2DblR[r];
    }
    __syncthreads();
  }

  __device__ __forceinline__ uint32_t bias(int i) const { return sh[16 * (kForm + i) + (threadIdx.x & 15)]; }

  template <bool WITH_NSUB> __device__ __forceinline__ void lin(const Op &o) {
    if (o.live) {
      const int di = o.k == C29_SUB2 || o.k == C29_NSUB ? 1 : o.k == C29_SUB4D ? 2 : o.k == C29_SUB8 ? 4 : 0;
      const uint32_t m = o.k == C29_ADD1 ? 1u : o.k == C29_COPY ? 0u : o.k == C29_SUB4D ? (uint32_t)-2 : (uint32_t)-1;
      uint32_t r = row_norm(sh[o.a[0]] + bias(di) + m * sh[o.a[1]]);
      if (WITH_NSUB) {
        const uint32_t n = row_norm(bias(2) - r);
        if (o.k == C29_NSUB) r = n;
      }
      sh[o.d] = r;
    }
    __syncthreads();
  }
  // POST: some operations of the round derive more from the product
  template <bool POST> __device__ __forceinline__ void dot(const Op &o) {
    if (o.live) {
      uint32_t r = row_dot(rk, sh[o.a[0]], sh[o.a[1]], sh[o.a[2]], sh[o.a[3]]);
      if (POST) {
        const uint32_t r3 = row_norm(3 * r);
        if (o.k == C29_DOTM || o.k == C29_DOTMN) r = r3;
        const uint32_t n = row_norm(bias(o.k == C29_DOTMN ? 3 : 1) - r);
        if (o.k == C29_DOTN || o.k == C29_DOTMN) sh[o.a[4]] = n;
      }
      sh[o.d] = r;
    }
    __syncthreads();
  }
  __device__ __forceinline__ void dot4(const Op &o) {
    if (o.live) {
      uint32_t x[8];
#pragma unroll
      for (int i = 0; i < 8; i++) x[i] = sh[o.a[i]];
      RowT s;
#pragma unroll
      for (int i = 0; i < 8; i += 2) row_conv(rk, s, x[i], x[i + 1]);
      sh[o.d] = row_redc(rk, s);
    }
    __syncthreads();
  }
  template <bool ADD> __device__ __forceinline__ void chain(const Op &o) {
    if (o.live) {
      const uint32_t a0 = sh[o.a[0]], a1 = sh[o.a[1]], sv = ADD ? sh[o.a[2]] : a1;
      const uint32_t x = ADD ? row_norm(a0 + bias(3) - row_norm(a1 + 2 * sv)) : row_norm(a0 + bias(2) - 2 * sv);
      const uint32_t t = row_norm(sv + bias(ADD ? 4 : 3) - x);
      const uint32_t n = row_norm(bias(ADD ? 5 : 4) - t);
      sh[o.d] = o.k == C29_COPY                            ? a0
                : o.k == C29_X3D || o.k == C29_X3A ? x
                : o.k == C29_TD || o.k == C29_TA   ? t
                                                   : n;
    }
    __syncthreads();
  }

  // acc = 2 acc
  __device__ __forceinline__ void dbl() {
    lin<false>(dbl_op[0]);
    dot<true>(dbl_op[1]);
    dot<false>(dbl_op[2]);
    chain<false>(dbl_op[3]);
    dot4(dbl_op[4]);
  }
  // acc + q up to PP and RR; the accumulator is left alone
  __device__ __forceinline__ void add1() {
    Op o;
    o.fetch(kG2Add1, 0, kG2Add1R[0]);
    lin<false>(o);
    o.fetch(kG2Add1, kG2Add1R[0], kG2Add1R[1]);
    dot<false>(o);
    o.fetch(kG2Add1, kG2Add1R[0] + kG2Add1R[1], kG2Add1R[2]);
    lin<true>(o);
    o.fetch(kG2Add1, kG2Add1R[0] + kG2Add1R[1] + kG2Add1R[2], kG2Add1R[3]);
    dot<false>(o);
  }
  // acc += q
  __device__ __forceinline__ void add2() {
    Op o;
    o.fetch(kG2Add2, 0, kG2Add2R[0]);
    lin<false>(o);
    o.fetch(kG2Add2, kG2Add2R[0], kG2Add2R[1]);
    dot<false>(o);
    o.fetch(kG2Add2, kG2Add2R[0] + kG2Add2R[1], kG2Add2R[2]);
    lin<false>(o);
    o.fetch(kG2Add2, kG2Add2R[0] + kG2Add2R[1] + kG2Add2R[2], kG2Add2R[3]);
    chain<true>(o);
    o.fetch(kG2Add2, kG2Add2R[0] + kG2Add2R[1] + kG2Add2R[2] + kG2Add2R[3], kG2Add2R[4]);
    dot4(o);
  }

  static constexpr uint8_t ZZ[2] = {H_ZZ0, H_ZZ1}, QZZ[2] = {H_QZZ0, H_QZZ1}, PP[2] = {E_PP0, E_PP1},
                           RR[2] = {E_RR0, E_RR1};
  // zero mod q in both component slots (values below 2q): the same answer in
  // every lane of the workgroup
  __device__ __forceinline__ bool is_zero(const uint8_t (&s)[2]) const {
    const uint32_t k = threadIdx.x & 15;
    const uint32_t x = sh[16 * s[0] + k], y = sh[16 * s[1] + k];
    return row_is_zero(x) && row_is_zero(y);
  }
};

// ------------------------------------------------------------ accumulators
// A running point over stored 29-bit slots (limbs below 2^29 + 4 allowed): G1 in
// the registers of one wave, G2 in LDS, held by a workgroup of four.  Infinity
// is tracked in a flag every lane holds.
template <class F> struct RowAcc;
template <> struct RowAcc<Fq> {
  static constexpr int SW = 36;
  RowG1K k;
  RowG1 p;
  bool inf;
  __device__ __forceinline__ void clear() {
    p = {0, 0, 0, 0};
    inf = true;
  }
  __device__ __forceinline__ void set(const uint32_t *slot) {
    p = row_load_g1(slot);
    inf = row_is_zero(p.ZZ);
  }
  __device__ __forceinline__ void dbl(uint32_t n) {
    if (inf) return;
#pragma unroll 1
    for (uint32_t i = 0; i < n; i++) row_dbl(k, p);
  }
  __device__ __forceinline__ void add(const uint32_t *slot) {
    const RowG1 q = row_load_g1(slot);
    if (row_is_zero(q.ZZ)) return;
    if (inf) {
      p = q;
      inf = false;
    } else {
      row_add(k, p, q, inf);
    }
  }
  __device__ __forceinline__ void store(uint32_t *slot) const {
    const uint32_t l = threadIdx.x & 63;
    if (l < 9) {
      slot[l] = p.X;
      slot[9 + l] = p.Y;
      slot[18 + l] = inf ? 0u : p.ZZ;
      slot[27 + l] = inf ? 0u : p.ZZZ;
    }
  }
  // canonical affine words, by one wave
  __device__ __forceinline__ void store_affine_to(uint32_t *out) const {
    const uint32_t l = threadIdx.x & 63;
    uint32_t w[8];
    if (inf) {
      for (int i = 0; i < 8; i++) w[i] = l ? FieldConst<0>::one[i] : 0u;
    } else {
      const uint32_t t = row_inverse(row_mul(k, p.ZZ, p.ZZZ));
      const uint32_t i = row_mul(k, t, k.odd ? p.ZZ : p.ZZZ);  // 1/ZZ | 1/ZZZ
      const uint32_t v = row_mul(k, i, k.odd ? p.Y : p.X);
      row_words(row_mul(k, v, kRowFrom[l & 15]), w);
    }
    if (l == 0 || l == 16) st8(out + l / 2, w);
  }
};

template <> struct RowAcc<Fq2> {
  using C = Coop29<Fq2>;
  static constexpr int N = 16 * C::kRows, kLds = C::kSlots * 16, SW = 72;
  C prog;
  uint32_t *sh;
  bool inf;
  // slot word of element word i of a stored slot
  __device__ __forceinline__ static uint32_t at(uint32_t i) { return 16 * (i / 9) + i % 9; }
  __device__ __forceinline__ RowAcc(uint32_t *lds, const uint32_t *slot) : prog(lds), sh(lds) {
    if (threadIdx.x < SW) sh[at(threadIdx.x)] = slot[threadIdx.x];
    __syncthreads();
    inf = prog.is_zero(C::ZZ);
  }
  __device__ __forceinline__ void dbl(uint32_t n) {
    if (inf) return;
#pragma unroll 1
    for (uint32_t i = 0; i < n; i++) prog.dbl();
  }
  __device__ __forceinline__ void add(const uint32_t *slot) {
    __syncthreads();  // every wave is done with the last addend
    if (threadIdx.x < SW) sh[16 * C::NC + at(threadIdx.x)] = slot[threadIdx.x];
    __syncthreads();
    if (prog.is_zero(C::QZZ)) return;
    if (inf) {
      if (threadIdx.x < 16 * C::NC) sh[threadIdx.x] = sh[16 * C::NC + threadIdx.x];
      __syncthreads();
      inf = false;
      return;
    }
    prog.add1();
    if (prog.is_zero(C::PP)) {
      const bool same = prog.is_zero(C::RR);
      __syncthreads();  // every wave has read PP and RR
      if (same) prog.dbl();  // acc == q
      else inf = true;       // acc == -q
      return;
    }
    prog.add2();
  }
  __device__ __forceinline__ void store(uint32_t *slot) const {
    if (threadIdx.x < SW) slot[threadIdx.x] = inf && threadIdx.x >= SW / 2 ? 0u : sh[at(threadIdx.x)];
  }
  // canonical affine words, by the first wave
  __device__ __forceinline__ void store_affine_to(uint32_t *out) const {
    if (threadIdx.x >= 64) return;
    const uint32_t l = threadIdx.x, ln = l & 15;
    uint32_t w[8];
    if (inf) {
      for (int i = 0; i < 8; i++) w[i] = l == 32 ? FieldConst<0>::one[i] : 0u;  // (0, 0, 1, 0)
    } else {
      const RowK &k = prog.rk;
      const bool odd = (l >> 4) & 1, hi = (l >> 5) & 1;
      auto v = [&](int i) { return sh[16 * i + ln]; };
      auto neg = [&](uint32_t x) { return row_norm(kRowD[1][ln] - x); };  // 2q - x
      // rows 2h, 2h + 1: the components of a_h b_h
      auto mul2 = [&](uint32_t a00, uint32_t a01, uint32_t b00, uint32_t b01, uint32_t a10, uint32_t a11,
                      uint32_t b10, uint32_t b11) {
        const uint32_t a0 = hi ? a10 : a00, a1 = hi ? a11 : a01, b0 = hi ? b10 : b00, b1 = hi ? b11 : b01;
        return row_dot(k, a0, odd ? b1 : b0, a1, odd ? b0 : neg(b1));
      };
      const uint32_t zz0 = v(H_ZZ0), zz1 = v(H_ZZ1), z30 = v(H_ZZZ0), z31 = v(H_ZZZ1);
      uint32_t t0, t1, u0, u1, a0, a1, b0, b1;
      row_spread2(mul2(zz0, zz1, z30, z31, zz0, zz1, z30, z31), t0, t1);  // ZZ ZZZ
      const uint32_t n = row_inverse(row_dot(k, t0, t0, t1, t1));       // its inverse: (t0 - t1 u) / (t0^2 + t1^2)
      row_spread2(row_mul(k, odd ? neg(t1) : t0, n), u0, u1);
      row_spread4(mul2(u0, u1, z30, z31, u0, u1, zz0, zz1), a0, a1, b0, b1);  // 1/ZZ, 1/ZZZ
      const uint32_t r = mul2(v(H_X0), v(H_X1), a0, a1, v(H_Y0), v(H_Y1), b0, b1);
      row_words(row_mul(k, r, kRowFrom[ln]), w);
    }
    if (ln == 0) st8(out + l / 2, w);
  }
};

}  // namespace csk
