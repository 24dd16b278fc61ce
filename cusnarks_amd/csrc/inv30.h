// Modular inversion by division steps, for the inversions that close a multiexp
// and the per-point ones of the table builders.
//
// Bernstein and Yang, "Fast constant-time gcd computation and modular
// inversion" (2019), define for odd f the step
//   (delta, f, g) -> (1 - delta, g, (g - f) / 2)                delta > 0, g odd
//                    (1 + delta, f, (g + (g mod 2) f) / 2)      otherwise
// and prove that from delta = 1 at most (49 b + 57) / 17 of them bring numbers of
// b bits to g = 0, f = +-gcd: 741 for b = 256.
//
// A batch is 30 steps on the low 30 bits of f and g, which is all that they look
// at, and its matrix (u v; q r), 2^30 (f', g') = (u f + v g, q f + r g), with
// |u| + |v| and |q| + |r| at most 2^30.  A row is kept as one 64-bit number
// u + 2^32 v: doubling, adding and subtracting rows are then single operations,
// exact as long as the entries fit (they do), and the entries are read off at the
// end.  f, g and the pair d, e with d a = s f, e a = s g mod p (s: the scale) are
// nine 30-bit limbs, the top one signed, and take the matrix once a batch; for d and
// e a multiple m p, |m| <= 2^29, makes the sum divisible by 2^30, so that they grow
// by at most p / 2: after the 25 batches that can be needed both are within 13.5 p,
// and only the result is brought to [0, p).  About 18 batches end with g = 0.  The
// scale makes the caller's factor (Montgomery's) part of the inverse.
#pragma once
#include <stdint.h>

namespace csk {

struct I30 {
  int32_t l[9];
};

// words of a number below 2^256 -> nine 30-bit limbs
__device__ __forceinline__ I30 i30_from(const uint32_t *w) {
  I30 r;
#pragma unroll
  for (int i = 0; i < 9; i++) {
    const int b = 30 * i, wi = b >> 5, sh = b & 31;
    uint32_t x = w[wi] >> sh;
    if (sh > 2 && wi < 7) x |= w[wi + 1] << (32 - sh);
    r.l[i] = (int32_t)(x & 0x3FFFFFFFu);
  }
  return r;
}

// the compiler knows the masked limbs to be nonnegative and would form their
// signed products from unsigned ones and corrections
#ifdef __HIP__
__device__ __forceinline__ int32_t i30_signed(int32_t x) {
  asm("" : "+v"(x));
  return x;
}
// the first lane's value, in a scalar register
template <bool UNIFORM> __device__ __forceinline__ uint32_t i30_low(int32_t x) {
  return (uint32_t)(UNIFORM ? __builtin_amdgcn_readfirstlane(x) : x);
}
#else
static inline int32_t i30_signed(int32_t x) { return x; }
template <bool UNIFORM> static inline uint32_t i30_low(int32_t x) { return (uint32_t)x; }
#endif

struct I30Row {
  int32_t x, y;  // x + 2^32 y
};
__device__ __forceinline__ I30Row i30_row(uint64_t r) {
  const uint32_t lo = (uint32_t)r;
  return {(int32_t)lo, (int32_t)((uint32_t)(r >> 32) + (lo >> 31))};
}

// 30 division steps; the rows of their matrix in top and bottom.  On the scalar unit a
// step is five instructions, nine more where g is odd and up to five for a turn.
// Unrolled, as one wave waits for them: a table run of 64 G1 points, an inversion and
// little else, 177 us, 179 with five steps to a trip, 186 with one.
__device__ __forceinline__ void i30_steps(int32_t &delta, uint32_t f, uint32_t g, I30Row &top, I30Row &bottom) {
  uint64_t a = 1, b = 1ull << 32;
#pragma unroll
  for (int k = 0; k < 30; k++) {
    if (g & 1) {
      if (delta > 0) {  // a quarter turn: the sum below is then g - f, beside f = g
        const uint32_t h = f;
        const uint64_t c = a;
        f = g;
        g = 0 - h;
        a = b;
        b = 0 - c;
        delta = -delta;
      }
      g += f;
      b += a;
    }
    g >>= 1;
    a += a;
    delta++;
  }
  top = i30_row(a);
  bottom = i30_row(b);
}

// (x X + y Y + m P) / 2^30, an exact division
__device__ __forceinline__ I30 i30_combine(const I30Row &r, const I30 &X, const I30 &Y, int32_t m, const I30 &P) {
  I30 o;
  int64_t c = 0;
#pragma unroll
  for (int i = 0; i < 9; i++) {
    c += (int64_t)r.x * X.l[i];
    c += (int64_t)r.y * Y.l[i];
    c += (int64_t)m * P.l[i];
    if (i > 0) o.l[i - 1] = i30_signed((int32_t)c & 0x3FFFFFFF);
    c >>= 30;
  }
  o.l[8] = (int32_t)c;
  return o;
}

// the m of -2^29 .. 2^29 - 1 for which x X + y Y + m p is divisible by 2^30;
// np = -1/p mod 2^32
__device__ __forceinline__ int32_t i30_multiple(const I30Row &r, const I30 &X, const I30 &Y, uint32_t np) {
  const uint32_t t = (uint32_t)r.x * (uint32_t)X.l[0] + (uint32_t)r.y * (uint32_t)Y.l[0];
  return (int32_t)(t * np << 2) >> 2;
}

// words of scale / a mod p (scale below p, 1 if null) for 0 < a < 2^256 coprime to
// p (p odd, below 2^255); pw: words of p, np = -1/p mod 2^32.  UNIFORM: every
// active lane has the same a, so the division steps run on the scalar unit.
template <bool UNIFORM>
__device__ __forceinline__ void i30_inverse(const uint32_t *a, const uint32_t *pw, uint32_t np, uint32_t *out,
                                            const uint32_t *scale = nullptr) {
  const I30 p = i30_from(pw), zero = {};
  I30 f = p, g = i30_from(a), d = {}, e = {};
  e.l[0] = 1;
  if (scale) e = i30_from(scale);
  int32_t delta = 1, left;
  do {
    I30Row t, b;
    i30_steps(delta, i30_low<UNIFORM>(f.l[0]), i30_low<UNIFORM>(g.l[0]), t, b);
    const I30 f1 = i30_combine(t, f, g, 0, zero), d1 = i30_combine(t, d, e, i30_multiple(t, d, e, np), p);
    g = i30_combine(b, f, g, 0, zero);
    e = i30_combine(b, d, e, i30_multiple(b, d, e, np), p);
    f = f1;
    d = d1;
    left = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) left |= g.l[i];
  } while (i30_low<UNIFORM>(left) != 0);
  // f = +-1: the result is f d, within 13.5 p; as a number of [0, 28 p) it loses 14 p,
  // 7 p, 4 p, 2 p and p where it is at least that
  const int32_t sign = f.l[8] < 0 ? -1 : 1;
  int32_t k = 14;
#pragma unroll 1
  for (int pass = 0; pass < 6; pass++) {
    I30 x;
    int64_t c = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      c += pass == 0 ? (int64_t)sign * d.l[i] : (int64_t)d.l[i];
      c += (int64_t)k * p.l[i];
      x.l[i] = i < 8 ? (int32_t)c & 0x3FFFFFFF : (int32_t)c;
      c >>= 30;
    }
    const bool take = pass == 0 || x.l[8] >= 0;
#pragma unroll
    for (int i = 0; i < 9; i++) d.l[i] = take ? x.l[i] : d.l[i];
    k = pass == 0 ? -14 : pass == 1 ? -7 : pass == 2 ? -4 : k / 2;
  }
#pragma unroll
  for (int k2 = 0; k2 < 8; k2++) {  // 30-bit limbs -> words
    uint32_t x = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      const int lo = 30 * i - 32 * k2;
      if (lo >= 32 || lo + 30 <= 0) continue;
      x |= lo >= 0 ? ((uint32_t)d.l[i] << lo) : ((uint32_t)d.l[i] >> -lo);
    }
    out[k2] = x;
  }
}

}  // namespace csk
