// Scalar splitting along the curve's endomorphism.
//
// BN254 has j-invariant 0, so phi(x, y) = (beta x, y) with beta^3 = 1 is an
// endomorphism of G1 and of the twist, and on the order-r subgroup it is the
// multiplication by a cube root of unity lambda mod r.  A scalar k < r splits
// as k = k1 + k2 lambda mod r with |k1|, |k2| < 2^126 (Gallant, Lambert and
// Vanstone, "Faster point multiplication on elliptic curves with efficient
// endomorphisms", 2001), so k P = k1 P + k2 phi(P).
//
// lambda = 4407920970296243842393367215006156084916469457145843978461.  The
// lattice of (a, b) with a + b lambda = 0 mod r has the short vectors
// (s, -n1) and (n2, s), s^2 + n1 n2 = r:
//   s  = 9931322734385697763
//   n1 = 147946756881789319000765030803803410728
//   n2 = 147946756881789319010696353538189108491
// (k, 0) is c1 (s, -n1) + c2 (n2, s) for c1 = s k / r, c2 = n1 k / r; with the
// nearest whole numbers the rest is
//   k1 = k - c1 s - c2 n2,  k2 = c1 n1 - c2 s,
// at most (1/2 + 2^-33)(s + n2) < 2^126 in size.  c1 and c2 come from
// products by round(2^288 s / r) and round(2^288 n1 / r).
//
// On the twist psi(x, y) = (conj(x) gx, conj(y) gy), the q-power Frobenius seen
// through the twist (gx = (9 + u)^((q - 1) / 3), gy = (9 + u)^((q - 1) / 2)), is the
// multiplication by mu = q mod r = 6 x^2, x the curve's parameter, and psi^2 = -phi:
// k = k0 + k1 mu + k2 mu^2 + k3 mu^3 with |ki| < 2^64 (Galbraith and Scott,
// "Exponentiation in pairing-friendly groups using homomorphisms", 2008).  A reduced
// basis of the lattice of (a0, .., a3) with sum a_i mu^i = 0 mod r:
//   (2x, x + 1, -x, x), (x, -x, x, 2x + 1), (x + 1, x, x, -2x), (2x + 1, -x, -x - 1, -x)
// (k, 0, 0, 0) is the sum of the rows times k (6x^3 - x) / r, k (6x^3 + 6x^2 + 2x) / r,
// k (6x^3 + 6x^2 + 4x + 1) / r and k (6x^3 + 6x^2 + x) / r.  Their nearest whole numbers
// c_j leave k0 .. k3, at most half the sums of the columns: 0.81 2^64.
#pragma once
#include <stdint.h>

namespace csk {

// bits of a half (its size is below 2^kGlvBits), of a quarter and of a whole scalar
static constexpr uint32_t kGlvBits = 126, kGlsBits = 64, kScalarBits = 254;

namespace glv_detail {
struct K {
  static constexpr uint32_t g1[4] = {1857668884u, 3353392087u, 3642565422u, 2u};
  static constexpr uint32_t g2[6] = {2783153403u, 958312845u, 2054937044u, 2809385679u, 1288630292u, 2u};
  static constexpr uint32_t h0[7] = {2099248942u, 2513771441u, 1190444457u, 4235297966u, 149281382u, 2967022483u, 2659201418u};
  static constexpr uint32_t h1[7] = {893176993u, 853813032u, 771696917u, 2749716351u, 1437911675u, 2967022485u, 2659201418u};
  static constexpr uint32_t h2[7] = {2750845877u, 4207205119u, 119295043u, 2749716354u, 1437911675u, 2967022485u, 2659201418u};
  static constexpr uint32_t h3[7] = {587435050u, 3472084287u, 3245381501u, 2749716349u, 1437911675u, 2967022485u, 2659201418u};
  static constexpr uint64_t x = 4965661367192848881ull;
  static constexpr uint32_t s[2] = {2496795619u, 2312316264u};
  static constexpr uint32_t n1[4] = {2102333736u, 2182200299u, 4005059068u, 1867350600u};
  static constexpr uint32_t n2[4] = {304162059u, 199549268u, 4005059069u, 1867350600u};
};

// words 9 .. 9 + NO of a b + 2^287
template <int NB, int NO> __device__ __forceinline__ void mul_hi(const uint32_t *a, const uint32_t (&b)[NB], uint32_t *o) {
  uint32_t t[8 + NB];
#pragma unroll
  for (int i = 0; i < 8 + NB; i++) t[i] = i == 8 ? 0x80000000u : 0u;
#pragma unroll
  for (int j = 0; j < NB; j++) {
    uint64_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      c += (uint64_t)a[i] * b[j] + t[i + j];
      t[i + j] = (uint32_t)c;
      c >>= 32;
    }
    // row j ends at word j + 8, which only the rounding bit has reached
    c += t[j + 8];
    t[j + 8] = (uint32_t)c;
    if (j + 9 < 8 + NB) t[j + 9] += (uint32_t)(c >> 32);
  }
#pragma unroll
  for (int i = 0; i < NO; i++) o[i] = t[9 + i];
}

// r = (r + sign a b) mod 2^128
template <int NA, int NB, bool SUB>
__device__ __forceinline__ void mul_add(uint32_t *r, const uint32_t *a, const uint32_t (&b)[NB]) {
  uint32_t p[4] = {0, 0, 0, 0};
#pragma unroll
  for (int j = 0; j < NB; j++) {
    uint64_t c = 0;
#pragma unroll
    for (int i = 0; i < NA; i++) {
      if (i + j > 3) continue;
      c += (uint64_t)a[i] * b[j] + p[i + j];
      p[i + j] = (uint32_t)c;
      c >>= 32;
    }
    if (j + NA < 4) p[j + NA] = (uint32_t)c;
  }
  uint64_t c = SUB ? 1 : 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    c += (uint64_t)r[i] + (SUB ? ~p[i] : p[i]);
    r[i] = (uint32_t)c;
    c >>= 32;
  }
}

// size and sign of a 128-bit two's complement number
__device__ __forceinline__ uint32_t size_sign(uint32_t *r) {
  const uint32_t neg = r[3] >> 31, m = 0u - neg;
  uint64_t c = neg;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    c += r[i] ^ m;
    r[i] = (uint32_t)c;
    c >>= 32;
  }
  return neg;
}
}  // namespace glv_detail

// k < r (8 words) -> |k1|, |k2| (4 words each); bit h of the result is set
// when k_(h+1) is negative
__device__ __forceinline__ uint32_t glv_split(const uint32_t *k, uint32_t *k1, uint32_t *k2) {
  using namespace glv_detail;
  uint32_t c1[2], c2[4];
  mul_hi<4, 2>(k, K::g1, c1);
  mul_hi<6, 4>(k, K::g2, c2);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    k1[i] = k[i];
    k2[i] = 0;
  }
  mul_add<2, 2, true>(k1, c1, K::s);
  mul_add<4, 4, true>(k1, c2, K::n2);
  mul_add<2, 4, false>(k2, c1, K::n1);
  mul_add<4, 2, true>(k2, c2, K::s);
  const uint32_t a = size_sign(k1), b = size_sign(k2);
  return a | (b << 1);
}

// k < r (8 words) -> |k0| .. |k3| (2 words each); bit i of the result is set when
// k_i is negative.  All modulo 2^128: c_j has up to 190 bits, but k_i is small.
__device__ __forceinline__ uint32_t gls_split(const uint32_t *k, uint32_t (*o)[2]) {
  using namespace glv_detail;
  typedef unsigned __int128 u128;
  uint32_t w[4][4];
  mul_hi<7, 4>(k, K::h0, w[0]);
  mul_hi<7, 4>(k, K::h1, w[1]);
  mul_hi<7, 4>(k, K::h2, w[2]);
  mul_hi<7, 4>(k, K::h3, w[3]);
  auto u = [](const uint32_t *v) {
    return ((u128)((uint64_t)v[3] << 32 | v[2]) << 64) | ((uint64_t)v[1] << 32 | v[0]);
  };
  const u128 c0 = u(w[0]), c1 = u(w[1]), c2 = u(w[2]), c3 = u(w[3]);
  const u128 d = c0 - c1, e = c2 - c3;
  uint32_t neg = 0;
  auto put = [&](int i, u128 r) {
    const bool n = (r >> 127) != 0;
    const uint64_t v = n ? 0 - (uint64_t)r : (uint64_t)r;
    o[i][0] = (uint32_t)v;
    o[i][1] = (uint32_t)(v >> 32);
    neg |= (uint32_t)n << i;
  };
  put(0, u(k) - (K::x * (c0 + c0 + c1 + c2 + c3 + c3) + c2 + c3));
  put(1, 0 - (K::x * (d + e) + c0));
  put(2, K::x * (d - e) + c3);
  put(3, 0 - (K::x * (c0 + c1 + c1 - c2 - c2 - c3) + c1));
  return neg;
}

}  // namespace csk
