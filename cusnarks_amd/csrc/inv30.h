// Modular inversion by division steps (Bernstein and Yang, "Fast
// constant-time gcd computation and modular inversion", 2019; the variant
// that starts at delta = 1/2), for the inversions that close a multiexp and
// the per-point ones of the table builders.
//
// f = p, g = a and the cofactors d, e (d a = f, e a = g mod p) are signed
// numbers of nine 30-bit limbs.  A batch takes 30 division steps on the low
// words alone, several at a time where the low bits of g can be cleared
// together, and collects them in a 2x2 matrix; f, g, d and e then take the
// matrix once, exactly divided by 2^30 (d, e modulo p).  About 18 batches end
// with g = 0, f = +-1.  A binary extended Euclid, which this replaced, shifted
// and added whole numbers bit by bit (the window combination of a one-window
// table run, an inversion and little else: 167 us, now 33).
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

// p^-1 mod 2^30 from np = -p^-1 mod 2^32
__device__ __forceinline__ constexpr uint32_t i30_pinv(uint32_t np) { return (0u - np) & 0x3FFFFFFFu; }

// 30 division steps on the low bits of f (odd) and g; eta = -2 delta.  The
// matrix (u v; q r) satisfies 2^30 (f', g') = (u f + v g, q f + r g) with
// |u| + |v| <= 2^30, |q| + |r| <= 2^30.
__device__ __forceinline__ int32_t i30_divsteps(int32_t eta, uint32_t f, uint32_t g, int32_t &u, int32_t &v,
                                                int32_t &q, int32_t &r) {
  uint32_t uu = 1, vv = 0, qq = 0, rr = 1;
  int32_t i = 30;
  for (;;) {
    // g even: halve it (a step with delta + 1 each); the sentinel stops at i
    const int32_t z = __builtin_ctz(g | (0xFFFFFFFFu << i));
    g >>= z;
    uu <<= z;
    vv <<= z;
    eta -= 2 * z;
    i -= z;
    if (i == 0) break;
    if (eta < 0) {  // delta > 0 and g odd: (f, g) <- (g, -f)
      eta = -eta;
      uint32_t t = f;
      f = g;
      g = 0u - t;
      t = uu;
      uu = qq;
      qq = 0u - t;
      t = vv;
      vv = rr;
      rr = 0u - t;
    }
    // the next (eta + 1) / 2 steps cannot swap: add the multiple w f of f
    // that clears that many low bits of g (at most 6: 1/f = f (2 - f f) mod 64)
    int32_t lim = (eta + 1) >> 1;
    if (lim > i) lim = i;
    if (lim > 6) lim = 6;
    const uint32_t w = (f * g * (f * f - 2u)) & ((1u << lim) - 1u);
    g += f * w;
    qq += uu * w;
    rr += vv * w;
  }
  u = (int32_t)uu;
  v = (int32_t)vv;
  q = (int32_t)qq;
  r = (int32_t)rr;
  return eta;
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

// words of a^-1 mod p for 0 < a < 2^256 coprime to p (p odd, below 2^255);
// pw: words of p, np = -p^-1 mod 2^32.  UNIFORM: every active lane has the same
// a, so the division steps run on the scalar unit.
template <bool UNIFORM>
__device__ __forceinline__ void i30_inverse(const uint32_t *a, const uint32_t *pw, uint32_t np, uint32_t *out) {
  constexpr int32_t M30 = 0x3FFFFFFF;
  const uint32_t pinv = i30_pinv(np);
  const I30 p = i30_from(pw);
  I30 f = p, g = i30_from(a), d = {}, e = {};
  e.l[0] = 1;
  int32_t eta = -1;  // delta = 1/2
  for (;;) {
    int32_t u, v, q, r;
    eta = i30_divsteps(eta, i30_low<UNIFORM>(f.l[0]), i30_low<UNIFORM>(g.l[0]), u, v, q, r);
    // d, e in (-2p, p) stay there: a negative one counts as itself plus p, and
    // the multiple of p that makes the sum divisible by 2^30 is taken in (-2^30, 0]
    const int32_t sd = d.l[8] >> 31, se = e.l[8] >> 31;
    int32_t md = (u & sd) + (v & se), me = (q & sd) + (r & se);
    int64_t cd = (int64_t)u * d.l[0] + (int64_t)v * e.l[0], ce = (int64_t)q * d.l[0] + (int64_t)r * e.l[0];
    md -= (int32_t)((pinv * (uint32_t)cd + (uint32_t)md) & (uint32_t)M30);
    me -= (int32_t)((pinv * (uint32_t)ce + (uint32_t)me) & (uint32_t)M30);
    cd += (int64_t)p.l[0] * md;
    ce += (int64_t)p.l[0] * me;
    int64_t cf = (int64_t)u * f.l[0] + (int64_t)v * g.l[0], cg = (int64_t)q * f.l[0] + (int64_t)r * g.l[0];
    cd >>= 30;
    ce >>= 30;
    cf >>= 30;
    cg >>= 30;
    int32_t nz = 0;
#pragma unroll
    for (int i = 1; i < 9; i++) {
      const int32_t di = d.l[i], ei = e.l[i], fi = f.l[i], gi = g.l[i];
      cd += (int64_t)u * di + (int64_t)v * ei + (int64_t)p.l[i] * md;
      ce += (int64_t)q * di + (int64_t)r * ei + (int64_t)p.l[i] * me;
      cf += (int64_t)u * fi + (int64_t)v * gi;
      cg += (int64_t)q * fi + (int64_t)r * gi;
      d.l[i - 1] = i30_signed((int32_t)cd & M30);
      e.l[i - 1] = i30_signed((int32_t)ce & M30);
      f.l[i - 1] = i30_signed((int32_t)cf & M30);
      g.l[i - 1] = i30_signed((int32_t)cg & M30);
      nz |= g.l[i - 1];
      cd >>= 30;
      ce >>= 30;
      cf >>= 30;
      cg >>= 30;
    }
    d.l[8] = (int32_t)cd;
    e.l[8] = (int32_t)ce;
    f.l[8] = (int32_t)cf;
    g.l[8] = (int32_t)cg;
    nz |= g.l[8];
    if (i30_low<UNIFORM>(nz) == 0) break;
  }
  // f = +-1 and d a = f: the inverse is f d in (-2p, 2p), brought to [0, p)
  const int32_t sf = f.l[8] >> 31;
#pragma unroll
  for (int i = 0; i < 9; i++) d.l[i] = (d.l[i] ^ sf) - sf;
#pragma unroll 1
  for (int k = 0; k < 5; k++) {  // + p twice, into (0, 4p); - p while it is at least p
    const int32_t keep = k < 2 ? 0 : -1, sg = k < 2 ? 0 : -1;
    int32_t x[9], c = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      const int32_t t = d.l[i] + ((p.l[i] ^ sg) - sg) + c;
      x[i] = i < 8 ? (t & M30) : t;
      c = t >> 30;
    }
    const bool lt = (x[8] & keep) < 0;
#pragma unroll
    for (int i = 0; i < 9; i++) d.l[i] = lt ? d.l[i] : x[i];
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {  // 30-bit limbs -> words
    uint32_t x = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      const int lo = 30 * i - 32 * k;
      if (lo >= 32 || lo + 30 <= 0) continue;
      x |= lo >= 0 ? ((uint32_t)d.l[i] << lo) : ((uint32_t)d.l[i] >> -lo);
    }
    out[k] = x;
  }
}

}  // namespace csk
