// Pippenger kernels and the per-curve launch sequence (see msm.hip for the
// pipeline overview).  Included by msm_g1.hip and msm_g2.hip so that the two
// curves compile as separate translation units.
#pragma once
#include <algorithm>
#include <type_traits>
#include "internal.h"
#include "curve.h"
#include "field29.h"
#include "coop29.h"
#include "glv.h"
#include "quad29.h"
#include "msm.h"

namespace csk {


__constant__ uint32_t kR1[8] = {4026531841u, 1138881939u, 2042196113u, 674490440u,
                                2172737629u, 3092268470u, 3778125865u, 811880050u};
__constant__ uint32_t kR2[8] = {3758096386u, 2277763879u, 4084392226u, 1348980880u,
                                50507962u,   1889569645u, 3261284435u, 1623760101u};
__constant__ uint32_t kR4[8] = {3221225476u, 260560463u,  3873817157u, 2697961761u,
                                101015924u,  3779139290u, 2227601574u, 3247520203u};

__device__ __forceinline__ void cond_sub(uint32_t *k, const uint32_t *m) {
  uint32_t d[8], borrow = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    uint64_t t = (uint64_t)k[i] - m[i] - borrow;
    d[i] = (uint32_t)t;
    borrow = (uint32_t)(t >> 63);
  }
#pragma unroll
  for (int i = 0; i < 8; i++) k[i] = borrow ? k[i] : d[i];
}

// k < 2^256 -> k mod r (2^256 < 6r, so three conditional subtractions)
__device__ __forceinline__ void reduce_mod_r(uint32_t *k) {
  cond_sub(k, kR4);
  cond_sub(k, kR2);
  cond_sub(k, kR1);
}

// ------------------------------------------------------------------ members
// largest j < J with segs[j].tbase <= b (the member of pass-1 workgroup b)
__device__ __forceinline__ uint32_t member_of_tile(const MsmSeg *segs, uint32_t J, uint32_t b) {
  uint32_t lo = 0, hi = J;
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (segs[mid].tbase <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

// beta of phi(x, y) = (beta x, y) in the 2^261 form: on G2 the other cube root
// of unity, so that phi is the multiplication by the same lambda
template <class F> struct Beta29;
template <> struct Beta29<Fq> {
  static constexpr uint32_t v[9] = {171145621u, 361569571u, 412916632u, 318393925u, 408922844u,
                                    24572269u,  250450874u, 338235712u, 789246u};
};
template <> struct Beta29<Fq2> {
  static constexpr uint32_t v[9] = {416069521u, 391846970u, 193189602u, 244240497u, 310558434u,
                                    69340804u,  535036287u, 352865610u, 1478937u};
};

// psi of the twist, (x, y) -> (conj(x) gx, conj(y) gy) (glv.h): both components and
// the first's negative
struct Psi29 {
  static constexpr uint32_t x0[9] = {77959568u, 116720857u, 200831163u, 387972444u, 449106301u,
                                     79574741u, 198110247u, 444835091u, 2396851u};
  static constexpr uint32_t x1[9] = {286535409u, 187804871u, 492312764u, 403373079u, 442701694u,
                                     360078139u, 294614062u, 104485018u, 1269326u};
  static constexpr uint32_t nx0[9] = {332884919u, 437214173u, 276443795u, 196420980u, 448858106u,
                                      505219562u, 349697305u, 332955936u, 774554u};
  static constexpr uint32_t y0[9] = {455018104u, 57932550u, 320278461u, 408777911u, 37819167u,
                                     383878197u, 519288526u, 32534274u, 1918653u};
  static constexpr uint32_t y1[9] = {430327765u, 436072363u, 496131354u, 220163167u, 145517765u,
                                     530932250u, 323946238u, 161949718u, 1410845u};
  static constexpr uint32_t ny0[9] = {492697295u, 496002479u, 156996497u, 175615513u, 323274328u,
                                      200916107u, 28519026u, 208385841u, 1252753u};
};

__device__ __forceinline__ void store29(uint32_t *d, const Fq29 &v) {
  uint32_t o[8];
  pack29(canon29(v), o);
  st8(d, o);
}

// the point in the 2^261 form (field29.h), packed words, component by
// component; with E = 2 followed by phi of it; with E = 4 by psi, -psi^2 = phi and
// -psi^3 of it
template <class F, int E> __device__ __forceinline__ void store_point29(uint32_t *d, const uint32_t *comps) {
  constexpr int NC = FieldIO<F>::NW / 8, PW = 2 * FieldIO<F>::NW;  // components per coordinate, words per point
  Fq29 v[2 * NC];
#pragma unroll
  for (int k = 0; k < 2 * NC; k++) {
    uint32_t in[8];
#pragma unroll
    for (int i = 0; i < 8; i++) in[i] = comps[8 * k + i];
    v[k] = mul29(unpack29(in), f29_const(Q29::to));
    store29(d + 8 * k, v[k]);
    if (E > 1) {
      Fq29 t = v[k];
      if (k < NC) t = mul29(t, f29_const(Beta29<F>::v));
      store29(d + (E / 2) * PW + 8 * k, t);
    }
  }
  if constexpr (E == 4) {
    const Fq29 s[4] = {dot29(v[0], f29_const(Psi29::x0), v[1], f29_const(Psi29::x1)),
                       dot29(v[0], f29_const(Psi29::x1), v[1], f29_const(Psi29::nx0)),
                       dot29(v[2], f29_const(Psi29::y0), v[3], f29_const(Psi29::y1)),
                       dot29(v[2], f29_const(Psi29::y1), v[3], f29_const(Psi29::ny0))};
#pragma unroll
    for (int k = 0; k < 4; k++) {
      store29(d + PW + 8 * k, s[k]);
      Fq29 t = s[k];
      if (k < 2) t = mul29(t, f29_const(Beta29<F>::v));
      store29(d + 3 * PW + 8 * k, t);
    }
  }
}
template <int E> __device__ __forceinline__ void store_point29(uint32_t *d, const Affine<Fq> &p) {
  uint32_t w[16];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    w[i] = p.x.v[i];
    w[8 + i] = p.y.v[i];
  }
  store_point29<Fq, E>(d, w);
}
template <int E> __device__ __forceinline__ void store_point29(uint32_t *d, const Affine<Fq2> &p) {
  uint32_t w[32];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    w[i] = p.x.c0.v[i];
    w[8 + i] = p.x.c1.v[i];
    w[16 + i] = p.y.c0.v[i];
    w[24 + i] = p.y.c1.v[i];
  }
  store_point29<Fq2, E>(d, w);
}

// ------------------------------------------------------------------ digits
// Signed c-bit digits of a number of NW words below 2^bits, lowest first:
// take() gives the next digit's bucket (|d| - 1, or 2^32 - 1 for d == 0) and
// whether d is negative.
template <int NW> struct Digits {
  uint32_t k[NW + 1];
  uint32_t c, B, mask, carry;
  __device__ __forceinline__ void set(const uint32_t *v, uint32_t c_) {
    c = c_;
    B = 1u << (c - 1);
    mask = (1u << c) - 1;
    carry = 0;
#pragma unroll
    for (int i = 0; i < NW; i++) k[i] = v[i];
    k[NW] = 0;
  }
  __device__ __forceinline__ uint32_t take(bool &neg) {
    uint32_t raw = (k[0] & mask) + carry;
#pragma unroll
    for (int i = 0; i < NW; i++) k[i] = __builtin_amdgcn_alignbit(k[i + 1], k[i], c);
    neg = raw > B;
    carry = neg;
    if (neg) raw = (1u << c) - raw;
    return raw - 1;
  }
};

// One workgroup per (member j, tile) of kSortTile points, E of them for each of
// the caller's (E = 2: P_i and phi(P_i) with the halves of k_i, glv.h; points
// 2i and 2i + 1 of the member; E = 4 on G2: P_i, psi(P_i) and so on with the
// quarters); block b covers the tiles in member order
// (member j's tiles start at b = tbase_j / W).  Member j's digits occupy
// D[W*pbase_j + w*n_j + i], b | neg << 31 for the nonzero signed digit d of
// window w (b = |d| - 1 < B), or 0xFFFFFFFF when d == 0 or the point is at
// infinity.  The workgroup also counts its digits per (window, hi = b >> s) in
// LDS and writes the counts as pass 1 of the sort expects them:
// cnt[cbase_j + (w*HB + hi)*NT_j + tile].  It also writes each point in the
// 2^261 form for the bucket loop, at concatenated point number pbase_j + i of
// pts29.
//
// Splitting halves the windows and doubles the points: as many entries, half
// the buckets to reduce and half the doublings of the window combination, for
// one product more per point and the second point's 64 B (128 B on G2) here.  G2's
// quarters halve them again for 14 products and 256 B more a point (5003 points: 46
// -> 55 us here, 757 -> 538 us in all).
//
// APART: the first `tiles` workgroups write only the digits and others the points, a
// thread each.  Few tiles leave most of the CUs idle, and the products of 4096 points
// keep one CU for 20 us and more.
template <class F, int E, bool APART>
__global__ void __launch_bounds__(1024) k_digits(const MsmSeg *__restrict__ segs, uint32_t J, uint32_t c,
                                                 uint32_t W, uint32_t s, uint32_t ts, uint32_t HB, uint32_t tiles,
                                                 uint32_t *__restrict__ digits, uint32_t *__restrict__ cnt,
                                                 uint32_t *__restrict__ pts29) {
  extern __shared__ uint32_t hist[];  // W * HB counters
  constexpr uint32_t TS = kSortTile / E;  // scalars of a tile
  constexpr int PW = 2 * FieldIO<F>::NW;
  if (APART && blockIdx.x >= tiles) {
    const uint32_t u = (blockIdx.x - tiles) * blockDim.x + threadIdx.x, g = u / TS;
    const uint32_t j = member_of_tile(segs, J, W * g);
    const uint64_t i = (uint64_t)(g - segs[j].tbase / W) * TS + u % TS;
    if (E * i < segs[j].n)
      store_point29<E>(pts29 + (segs[j].pbase + E * i) * PW, load_affine<F>(segs[j].points + i * PW));
    return;
  }
  const uint32_t j = member_of_tile(segs, J, W * blockIdx.x);
  const uint32_t tile = blockIdx.x - segs[j].tbase / W;
  const uint64_t pbase = segs[j].pbase, n = segs[j].n;
  const uint32_t NT = segs[j].NT;
  for (uint32_t i = threadIdx.x; i < W * HB; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  uint32_t *dj = digits + W * pbase;
  for (uint32_t t = threadIdx.x; t < TS; t += blockDim.x) {
    const uint64_t i = (uint64_t)tile * TS + t;
    if (E * i >= n) break;
    uint32_t k[8];
    ld8(k, segs[j].scalars + i * 8);
    reduce_mod_r(k);
    const Affine<F> p = load_affine<F>(segs[j].points + i * PW);
    const bool zero = affine_is_inf(p);
    if (!APART) store_point29<E>(pts29 + (pbase + E * i) * PW, p);
    auto entry = [&](uint32_t w, uint32_t b, bool neg) -> uint32_t {
      const bool live = b != 0xFFFFFFFFu && !zero;
      if (live) atomicAdd(&hist[w * HB + (b >> (w == W - 1 ? ts : s))], 1u);
      return live ? b | ((uint32_t)neg << 31) : 0xFFFFFFFFu;
    };
    uint32_t parts[E][8 / E], sg = 0;
    if constexpr (E == 4) sg = gls_split(k, parts) ^ 12u;  // points 2 and 3 are -psi^2 and -psi^3
    else if constexpr (E == 2) sg = glv_split(k, parts[0], parts[1]);
    else
      for (int e = 0; e < 8; e++) parts[0][e] = k[e];
    Digits<8 / E> d[E];
#pragma unroll
    for (int e = 0; e < E; e++) d[e].set(parts[e], c);
    for (uint32_t w = 0; w < W; w++) {
      uint32_t o[E];
#pragma unroll
      for (int e = 0; e < E; e++) {
        bool neg;
        const uint32_t b = d[e].take(neg);
        o[e] = entry(w, b, neg != (bool)((sg >> e) & 1));
      }
      uint32_t *q = dj + (uint64_t)w * n + E * i;
      if constexpr (E == 4) *reinterpret_cast<uint4 *>(q) = make_uint4(o[0], o[1], o[2], o[3]);
      else if constexpr (E == 2) *reinterpret_cast<uint2 *>(q) = make_uint2(o[0], o[1]);
      else *q = o[0];
    }
  }
  __syncthreads();
  const uint32_t cb = segs[j].cbase + tile;
  for (uint32_t i = threadIdx.x; i < W * HB; i += blockDim.x) cnt[cb + (uint64_t)i * NT] = hist[i];
}

template <class F, bool APART> static auto digits_kernel(uint32_t E) {
  if constexpr (std::is_same<F, Fq2>::value)
    if (E == 4) return k_digits<F, 4, APART>;
  return E == 2 ? k_digits<F, 2, APART> : k_digits<F, 1, APART>;
}

namespace {  // curve-independent kernels: one private copy per translation unit

// ------------------------------------------------------------------ scan
static constexpr int SCAN_THREADS = 256;
static constexpr int SCAN_ITEMS = 8;
static constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_reduce(const uint32_t *__restrict__ in, uint32_t K,
                                                              uint32_t *__restrict__ bsum) {
  __shared__ uint32_t sh[SCAN_THREADS];
  uint32_t base = blockIdx.x * SCAN_TILE;
  uint32_t s = 0;
  for (int j = 0; j < SCAN_ITEMS; j++) {
    uint32_t idx = base + j * SCAN_THREADS + threadIdx.x;
    if (idx < K) s += in[idx];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int st = SCAN_THREADS / 2; st > 0; st >>= 1) {
    if ((int)threadIdx.x < st) sh[threadIdx.x] += sh[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = sh[0];
}

// exclusive scan of the block sums in place (any nb)
__global__ void __launch_bounds__(1024) k_scan_blocks(uint32_t *__restrict__ bsum, uint32_t nb) {
  __shared__ uint32_t sh[1024];
  const uint32_t per = (nb + 1023) / 1024;
  uint32_t lo = threadIdx.x * per, s = 0;
  for (uint32_t j = 0; j < per; j++)
    if (lo + j < nb) s += bsum[lo + j];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int st = 1; st < 1024; st <<= 1) {
    uint32_t v = threadIdx.x >= (uint32_t)st ? sh[threadIdx.x - st] : 0;
    __syncthreads();
    sh[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = sh[threadIdx.x] - s;  // exclusive prefix of this thread's run
  for (uint32_t j = 0; j < per; j++)
    if (lo + j < nb) {
      uint32_t v = bsum[lo + j];
      bsum[lo + j] = run;
      run += v;
    }
}

// out[0..K] = exclusive prefix sums of in[0..K) (out[K] = total); in == out allowed
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_final(const uint32_t *in, uint32_t K,
                                                             const uint32_t *__restrict__ bsum, uint32_t *out) {
  __shared__ uint32_t sh[SCAN_THREADS];
  uint32_t base = blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_ITEMS;  // contiguous items per thread
  uint32_t v[SCAN_ITEMS], s = 0;
  for (int j = 0; j < SCAN_ITEMS; j++) {
    uint32_t idx = base + j;
    v[j] = idx < K ? in[idx] : 0;
    s += v[j];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int st = 1; st < SCAN_THREADS; st <<= 1) {
    uint32_t t = threadIdx.x >= (uint32_t)st ? sh[threadIdx.x - st] : 0;
    __syncthreads();
    sh[threadIdx.x] += t;
    __syncthreads();
  }
  uint32_t run = bsum[blockIdx.x] + sh[threadIdx.x] - s;
  for (int j = 0; j < SCAN_ITEMS; j++) {
    uint32_t idx = base + j;
    if (idx < K) out[idx] = run;
    run += v[j];
    if (idx + 1 == K) out[K] = run;
  }
}

// The whole scan by one workgroup, in place, for K <= SCAN_SMALL: three launches
// cost more than one workgroup's walk (12800 counters: 14 us against 9).
static constexpr uint32_t SCAN_SMALL = 16384;
__global__ void __launch_bounds__(1024) k_scan_small(uint32_t *arr, uint32_t K) {
  __shared__ uint32_t wsum[16];
  const uint32_t per = (K + 1023) / 1024, lo = threadIdx.x * per;
  uint32_t v[SCAN_SMALL / 1024], s = 0;
#pragma unroll
  for (uint32_t j = 0; j < SCAN_SMALL / 1024; j++) {
    v[j] = j < per && lo + j < K ? arr[lo + j] : 0u;
    s += v[j];
  }
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63) wsum[wv] = x;
  __syncthreads();
  uint32_t run = x - s, total = 0;
  for (uint32_t k = 0; k < 16; k++) {
    run += k < wv ? wsum[k] : 0u;
    total += wsum[k];
  }
#pragma unroll
  for (uint32_t j = 0; j < SCAN_SMALL / 1024; j++) {
    if (j < per && lo + j < K) arr[lo + j] = run;
    run += v[j];
  }
  if (threadIdx.x == 0) arr[K] = total;
}

// exclusive prefix sums of cnt[0..K) in place, cnt[K] = total; bsum: a word per
// SCAN_TILE counters
static inline void scan_counts(uint32_t *cnt, uint32_t K, uint32_t *bsum, hipStream_t st) {
  if (K <= SCAN_SMALL) {
    k_scan_small<<<1, 1024, 0, st>>>(cnt, K);
    return;
  }
  const uint32_t nb = (K + SCAN_TILE - 1) / SCAN_TILE;
  k_scan_reduce<<<nb, SCAN_THREADS, 0, st>>>(cnt, K, bsum);
  k_scan_blocks<<<1, 1024, 0, st>>>(bsum, nb);
  k_scan_final<<<nb, SCAN_THREADS, 0, st>>>(cnt, K, bsum, cnt);
}

static constexpr int SORT_THREADS = 256;
static constexpr int SORT_TILE = 4096;  // digits of one window per pass-1 workgroup
static constexpr int SORT_IPT = SORT_TILE / SORT_THREADS;

// exclusive scan of arr[0..len) in LDS by one workgroup of THREADS; tmp holds
// THREADS / 64 words (one per wave); returns the total (all threads)
template <int THREADS>
__device__ uint32_t block_exclusive_scan(uint32_t *arr, uint32_t len, uint32_t *tmp) {
  const uint32_t per = (len + THREADS - 1) / THREADS;
  const uint32_t lo = threadIdx.x * per;
  uint32_t s = 0;
  for (uint32_t j = 0; j < per; j++)
    if (lo + j < len) s += arr[lo + j];
  // inclusive scan across the 64 lanes of the wave, then the wave totals
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  uint32_t x = s;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63) tmp[wv] = x;
  __syncthreads();
  uint32_t run = x - s, total = 0;
  for (uint32_t k = 0; k < THREADS / 64; k++) {
    const uint32_t t = tmp[k];
    run += k < wv ? t : 0;
    total += t;
  }
  for (uint32_t j = 0; j < per; j++)
    if (lo + j < len) {
      uint32_t v = arr[lo + j];
      arr[lo + j] = run;
      run += v;
    }
  __syncthreads();
  return total;
}

// ------------------------------------------------------------------ sort pass 1
// Bucket b = hi * 2^s + lo.  Pass 1 groups the entries of every window by hi
// (HB <= 256 bins).  Workgroup x of the group maps to (member j, window w,
// tile) with x = tbase_j + w * NT_j + tile.  k_digits has counted the tile's
// kSortTile digits into cnt[cbase_j + (w*HB + hi)*NT_j + tile]; after an
// exclusive scan of cnt (member-, window-, bin-major), each (bin, tile) owns a
// contiguous output range, and the runs appear in bucket-key order
// j*K + w*B + b.
struct TileRef {
  uint32_t j, w, tile, NT;
  uint64_t n;
  const uint32_t *Dw;
  uint32_t cb;  // counter index of (w, bin 0, tile)
};

__device__ __forceinline__ TileRef tile_ref(const MsmSeg *segs, uint32_t J, uint32_t HB, uint32_t W,
                                            const uint32_t *D) {
  TileRef t;
  t.j = member_of_tile(segs, J, blockIdx.x);
  t.NT = segs[t.j].NT;
  const uint32_t local = blockIdx.x - segs[t.j].tbase;
  t.w = local / t.NT;
  t.tile = local - t.w * t.NT;
  t.n = segs[t.j].n;
  t.Dw = D + W * segs[t.j].pbase + (uint64_t)t.w * t.n;
  t.cb = segs[t.j].cbase + t.w * HB * t.NT + t.tile;
  return t;
}

// Pass 1 placement: the workgroup counting-sorts its entries by hi in LDS and
// writes each bin's run contiguously to the pass-1 arrays: tix (point index |
// sign) and tlo (lo, the low s < 16 bits of the bucket).  The top window of
// every scalar (global window index gw = j * W + w with gw mod Wwin = Wwin - 1:
// w = W - 1 for multiexp members, every Wwin-th member for the one-window
// members of table runs) splits its buckets at ts bits instead; with ts = 0
// its bins are single buckets, the pass-1 ranges are the final ones, and pass 2
// only copies the entries.
// HOIST issues the tile's sixteen digit loads before the counts (unconditional,
// the index clamped into the member's row; the tile's first index is < n);
// otherwise each entry is one guarded load, wait and count.  Measured: HOIST
// is faster for groups below ~2^27 entries (latency-bound), slower above
// (2^24 points x 15 windows: 1.71 vs 1.37 ms), where the loads of the many
// resident workgroups already keep HBM busy.
template <bool HOIST>
__global__ void __launch_bounds__(SORT_THREADS) k_sort_scatter1(const uint32_t *__restrict__ D,
                                                                const MsmSeg *__restrict__ segs, uint32_t J,
                                                                uint32_t s, uint32_t ts, uint32_t HB, uint32_t W,
                                                                uint32_t Wwin, const uint32_t *__restrict__ goff,
                                                                uint32_t *__restrict__ tix,
                                                                uint16_t *__restrict__ tlo) {
  __shared__ uint32_t h[256];
  __shared__ uint32_t base[256];
  __shared__ uint32_t scan_tmp[SORT_THREADS];
  __shared__ uint32_t stage[SORT_TILE];
  __shared__ uint16_t slo[SORT_TILE];
  __shared__ uint16_t sbin[SORT_TILE];
  const TileRef t = tile_ref(segs, J, HB, W, D);
  if ((t.j * W + t.w) % Wwin == Wwin - 1) s = ts;
  const uint32_t lomask = (1u << s) - 1;
  for (uint32_t i = threadIdx.x; i < HB; i += SORT_THREADS) h[i] = 0;
  __syncthreads();
  uint32_t dv[SORT_IPT], rk[SORT_IPT];
  if constexpr (HOIST) {
    for (int j = 0; j < SORT_IPT; j++) {
      const uint64_t idx = (uint64_t)t.tile * SORT_TILE + j * SORT_THREADS + threadIdx.x;
      dv[j] = t.Dw[idx < t.n ? idx : t.n - 1];
    }
    for (int j = 0; j < SORT_IPT; j++) {
      const uint64_t idx = (uint64_t)t.tile * SORT_TILE + j * SORT_THREADS + threadIdx.x;
      if (idx >= t.n) dv[j] = 0xFFFFFFFFu;
      const uint32_t d = dv[j];
      rk[j] = d != 0xFFFFFFFFu ? atomicAdd(&h[(d & 0x7FFFFFFFu) >> s], 1u) : 0u;
    }
  } else {
    for (int j = 0; j < SORT_IPT; j++) {
      const uint64_t idx = (uint64_t)t.tile * SORT_TILE + j * SORT_THREADS + threadIdx.x;
      const uint32_t d = idx < t.n ? t.Dw[idx] : 0xFFFFFFFFu;
      dv[j] = d;
      rk[j] = d != 0xFFFFFFFFu ? atomicAdd(&h[(d & 0x7FFFFFFFu) >> s], 1u) : 0u;
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < HB; i += SORT_THREADS) base[i] = h[i];
  __syncthreads();
  const uint32_t total = block_exclusive_scan<SORT_THREADS>(base, HB, scan_tmp);
  // h (the counts are in base now) takes each bin's output start minus its
  // tile-local start; offsets are < 2^31, the u32 difference wraps back on +p
  for (uint32_t i = threadIdx.x; i < HB; i += SORT_THREADS) h[i] = goff[t.cb + i * t.NT] - base[i];
  for (int j = 0; j < SORT_IPT; j++) {
    uint32_t d = dv[j];
    if (d == 0xFFFFFFFFu) continue;
    uint32_t b = d & 0x7FFFFFFFu, bin = b >> s;
    uint32_t pos = base[bin] + rk[j];
    uint32_t idx = t.tile * SORT_TILE + j * SORT_THREADS + threadIdx.x;
    stage[pos] = idx | (d & 0x80000000u);
    slo[pos] = (uint16_t)(b & lomask);
    sbin[pos] = (uint16_t)bin;
  }
  __syncthreads();
  if (s == 0) {
    for (uint32_t p = threadIdx.x; p < total; p += SORT_THREADS) tix[h[sbin[p]] + p] = stage[p];
    return;
  }
  for (uint32_t p = threadIdx.x; p < total; p += SORT_THREADS) {
    const uint32_t g = h[sbin[p]] + p;
    tix[g] = stage[p];
    tlo[g] = slo[p];
  }
}

// ------------------------------------------------------------------ sort pass 2
// One workgroup per (member, window, hi) segment of the pass-1 arrays, seg = (j*W + w)*HB
// + hi: partition by lo into the 2^s buckets seg*2^s + lo (= j*K + w*B +
// hi*2^s + lo).  The segment is counted once (bucket offsets are written for
// every bucket), then placed TILE entries at a time: each tile is
// counting-sorted by lo in LDS and every bucket's run is written contiguously
// after that bucket's running cursor.  TILE entries per step: 8192 measured
// faster for groups of 2^27 entries and more (2^24 x 15 windows), 4096 below.
// A top window (see pass 1) partitions by its ts low bits into the buckets
// gw*B + hi*2^ts + lo; its last segment also points the buckets it cannot
// reach (from HB*2^ts on) at its end, and with ts = 0 pass 1 has ordered its
// entries already, so they are copied.  `sorted` takes the place of the digits,
// which only pass 1 reads.
// counter[key] += 1 for the live lanes, the count before this lane's: the lanes
// that agree with the first one add once together.  For segments far above the
// average, which hold a bucket of very many entries (the ones among wire
// values): 64 additions to one counter take 64 turns.
__device__ __forceinline__ uint32_t count_hot(uint32_t *counter, uint32_t key, bool live) {
  const uint64_t act = __ballot(live);
  if (act == 0) return 0;
  const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)key, __builtin_ctzll(act));
  const uint64_t same = __ballot(live && key == first);
  const uint32_t lane = threadIdx.x & 63, lead = __builtin_ctzll(same);
  uint32_t r = 0;
  if (live && (key != first || lane == lead)) r = atomicAdd(&counter[key], key == first ? __popcll(same) : 1u);
  const uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)r, lead);
  return key == first ? base + __popcll(same & ((1ull << lane) - 1)) : r;
}

// Segments above `split` entries are left to a launch of their own (LONG), whose
// workgroups have more threads: few segments are long (most of a window's
// entries in one bin: wire values), so one workgroup's time is what they cost
// (300007 scalars, half of them 0 or 1: 249 us without the split, 13 + 70 with).
template <int TILE, int THREADS, bool LONG>
__global__ void __launch_bounds__(THREADS) k_sort_pass2(const uint32_t *__restrict__ tix,
                                                             const uint16_t *__restrict__ tlo,
                                                             const uint32_t *__restrict__ goff,
                                                             const MsmSeg *__restrict__ segs, uint32_t HB,
                                                             uint32_t s, uint32_t ts, uint32_t W, uint32_t Wwin,
                                                             uint32_t Ktot, uint32_t split, uint32_t *__restrict__ offsets,
                                                             uint32_t *__restrict__ sorted) {
  extern __shared__ uint32_t dyn[];  // 3 * 2^s words: counts, cursors, tile bases
  __shared__ uint32_t scan_tmp[THREADS / 64];
  __shared__ uint32_t stage[TILE];
  __shared__ uint16_t sbin[TILE];
  const uint32_t seg = blockIdx.x, per = W * HB, mj = seg / per, rem = seg - mj * per;
  const uint32_t NT = segs[mj].NT, cb = segs[mj].cbase;
  const uint32_t w = rem / HB, hi = rem - w * HB, gw = mj * W + w, B = HB << s;
  if (gw % Wwin == Wwin - 1) s = ts;
  const uint32_t L2 = 1u << s, key0 = gw * B + hi * L2;
  uint32_t *cntv = dyn, *cur = dyn + L2, *tb = dyn + 2 * L2;
  const uint32_t start = goff[cb + rem * NT], end = goff[cb + (rem + 1) * NT];
  if (LONG && end - start <= split) return;
  if (!LONG && seg == gridDim.x - 1 && threadIdx.x == 0) offsets[Ktot] = end;
  if (!LONG && hi == HB - 1)
    for (uint32_t k = key0 + L2 + threadIdx.x; k < (gw + 1) * B; k += THREADS) offsets[k] = end;
  if (s == 0) {
    if (LONG) return;
    if (threadIdx.x == 0) offsets[key0] = start;
    // an equal share of the window's entries each: the bins may be most uneven (c = 14:
    // 126 is 9 * 14, so the top window holds only carries, 2^24 of them in one bin; by
    // one workgroup a 2^24-point multiexp took 29.9 ms, 27.0 so; c = 18 26.0 and 22.6)
    const uint32_t w0 = goff[cb + w * HB * NT], w1 = goff[cb + (w + 1) * HB * NT], share = (w1 - w0 + HB - 1) / HB;
    const uint32_t last = min(w1, w0 + (hi + 1) * share);
    for (uint32_t e0 = w0 + hi * share; e0 < last; e0 += 8 * THREADS) {
      uint32_t v[8];
      for (int k = 0; k < 8; k++) {  // unconditional (clamped) loads, as below
        const uint32_t e = e0 + k * THREADS + threadIdx.x;
        v[k] = tix[e < last ? e : last - 1];
      }
      for (int k = 0; k < 8; k++) {
        const uint32_t e = e0 + k * THREADS + threadIdx.x;
        if (e < last) sorted[e] = v[k];
      }
    }
    return;
  }
  if (!LONG && end - start > split) return;
  for (uint32_t i = threadIdx.x; i < L2; i += THREADS) cntv[i] = 0;
  __syncthreads();
  // eight unconditional (clamped) loads in flight per thread, then their counts
  for (uint32_t e0 = start; e0 < end; e0 += 8 * THREADS) {
    uint32_t l[8];
    for (int k = 0; k < 8; k++) {
      const uint32_t e = e0 + k * THREADS + threadIdx.x;
      l[k] = tlo[e < end ? e : end - 1];
    }
    for (int k = 0; k < 8; k++) {
      const bool live = e0 + k * THREADS + threadIdx.x < end;
      if (LONG) count_hot(cntv, l[k], live);
      else if (live) atomicAdd(&cntv[l[k]], 1u);
    }
  }
  __syncthreads();
  block_exclusive_scan<THREADS>(cntv, L2, scan_tmp);
  for (uint32_t i = threadIdx.x; i < L2; i += THREADS) {
    offsets[key0 + i] = start + cntv[i];
    cur[i] = start + cntv[i];
  }
  __syncthreads();
  for (uint32_t t0 = start; t0 < end; t0 += TILE) {
    const uint32_t tn = min((uint32_t)TILE, end - t0);
    for (uint32_t i = threadIdx.x; i < L2; i += THREADS) tb[i] = 0;
    __syncthreads();
    constexpr int IPT = TILE / THREADS;
    uint32_t v[IPT], vl[IPT], rk[IPT];
    for (int j = 0; j < IPT; j++) {  // unconditional loads (clamped; tn >= 1)
      const uint32_t q = j * THREADS + threadIdx.x, qc = q < tn ? q : tn - 1;
      v[j] = tix[t0 + qc];
      vl[j] = tlo[t0 + qc];
    }
    for (int j = 0; j < IPT; j++) {
      const uint32_t q = j * THREADS + threadIdx.x;
      if (LONG) rk[j] = count_hot(tb, vl[j], q < tn);
      else rk[j] = q < tn ? atomicAdd(&tb[vl[j]], 1u) : 0u;
    }
    __syncthreads();
    // tile-local counts -> tile-local bases; keep the counts for the cursor update
    for (uint32_t i = threadIdx.x; i < L2; i += THREADS) cntv[i] = tb[i];
    __syncthreads();
    block_exclusive_scan<THREADS>(tb, L2, scan_tmp);
    for (int j = 0; j < IPT; j++) {
      uint32_t q = j * THREADS + threadIdx.x;
      if (q < tn) {
        uint32_t lo = vl[j];
        uint32_t pos = tb[lo] + rk[j];
        stage[pos] = v[j];
        sbin[pos] = (uint16_t)lo;
      }
    }
    __syncthreads();
    for (uint32_t p = threadIdx.x; p < tn; p += THREADS) {
      uint32_t lo = sbin[p];
      sorted[cur[lo] + (p - tb[lo])] = stage[p];
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < L2; i += THREADS) cur[i] += cntv[i];
    __syncthreads();
  }
}

// largest key in [0, K) with off[key] <= e (requires off[0] <= e < off[K])
__device__ __forceinline__ uint32_t find_key(const uint32_t *__restrict__ off, uint32_t K, uint32_t e) {
  uint32_t lo = 0, hi = K;
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (off[mid] <= e) lo = mid;
    else hi = mid;
  }
  return lo;
}

// The bucket holding entry e, from a key k with off[k] <= e (requires
// e < off[K]): one load when bucket k holds e.  Runs of empty buckets are
// crossed by doubling steps, then bisection: a top window reaches only
// 2^(254 mod c) of its 2^(c-1) buckets (c = 20: 2^14 of 2^19), and where the
// next member's keys follow, stepping over the rest one key at a time held
// the whole launch on one thread (four 20-bit table runs: +27 ms).
__device__ __forceinline__ uint32_t key_from(const uint32_t *__restrict__ off, uint32_t K, uint32_t k, uint32_t e) {
  if (off[k + 1] > e) return k;
  uint32_t lo = k + 1, hi = K, step = 1;  // off[lo] <= e < off[hi]
  for (;;) {
    const uint64_t nx = (uint64_t)lo + step;
    if (nx >= K) break;
    if (off[nx] > e) {
      hi = (uint32_t)nx;
      break;
    }
    lo = (uint32_t)nx;
    step <<= 1;
  }
  while (hi - lo > 1) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if (off[mid] <= e) lo = mid;
    else hi = mid;
  }
  return lo;
}

}  // namespace

// Sequential reader of one thread's run of the sorted (point index | sign)
// array, four entries per 16-byte load: every lane walks its own run, and
// with random point loads streaming through L2 a line read 4 bytes at a time
// is evicted and fetched again before its 32 entries are used.  The array
// is padded by 4 entries so the last aligned load stays inside it.
struct IndexReader {
  const uint32_t *base;
  uint32_t blk;  // e & ~3 of the loaded quad
  uint4 q;
  __device__ __forceinline__ IndexReader(const uint32_t *sorted, uint32_t e) : base(sorted), blk(e & ~3u) {
    q = *reinterpret_cast<const uint4 *>(base + blk);
  }
  __device__ __forceinline__ uint32_t at(uint32_t e) {
    if ((e & ~3u) != blk) {
      blk = e & ~3u;
      q = *reinterpret_cast<const uint4 *>(base + blk);
    }
    const uint32_t k = e & 3u;
    return k == 0 ? q.x : k == 1 ? q.y : k == 2 ? q.z : q.w;
  }
};

// ------------------------------------------------------------ accumulate
// The bucket loops run on 29-bit limbs (field29.h).  k_digits has written the
// group's points in the 2^261 form (packed words, at concatenated point
// number g) at the head of the sort buffer.
//
// Thread t of k_accumulate29 folds sorted entries [t*L, min((t+1)*L, E)) of
// the group.  Every lane performs exactly one mixed addition per loop trip
// (lane-uniform trip count), and a run is flushed when the entry just added
// closes its bucket or the chunk.  A run whose bucket started in this chunk
// is written to the bucket slot ("owned"); the first run of a chunk whose
// bucket started earlier goes to the chunk's carry slot for k_fixup.  Bucket
// key / Kj names the member whose points the entry indexes; the next entry's
// key is tracked ahead of the flush so its point can be prefetched from the
// right member.  Runs are stored unreduced as 29-bit slots, which the
// carry, fix-up and reduction kernels take as they are; only the window sums
// leave the 29-bit form (a conversion costs a product per component, too
// much for the divergent flush).
template <class F> struct Slot29 {
  static constexpr int NC = FieldIO<F>::NW / 8;  // base-field components per coordinate
  static constexpr int SW = 4 * NC * 9;          // words of one 29-bit XYZZ slot
};

// four 29-bit elements (36 words) as nine 16-byte stores
__device__ __forceinline__ void store4x29(uint32_t *d, const Fq29 &a, const Fq29 &b, const Fq29 &c, const Fq29 &e) {
  uint32_t w[36];
#pragma unroll
  for (int i = 0; i < 9; i++) {
    w[i] = a.l[i];
    w[9 + i] = b.l[i];
    w[18 + i] = c.l[i];
    w[27 + i] = e.l[i];
  }
  uint4 *d4 = reinterpret_cast<uint4 *>(d);
#pragma unroll
  for (int q = 0; q < 9; q++) d4[q] = make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
}
__device__ __forceinline__ void store29(uint32_t *d, const XYZZ29 &a) { store4x29(d, a.X, a.Y, a.ZZ, a.ZZZ); }
// component order X.c0, X.c1, Y.c0, ... as the 2^256-word XYZZ<Fq2> slot
__device__ __forceinline__ void store29(uint32_t *d, const XYZZ2_29 &a) {
  store4x29(d, a.X.c0, a.X.c1, a.Y.c0, a.Y.c1);
  store4x29(d + 36, a.ZZ.c0, a.ZZ.c1, a.ZZZ.c0, a.ZZZ.c1);
}

__device__ __forceinline__ XYZZ29 inf29() { return {Fq29{}, f29_const(Q29::one), Fq29{}, Fq29{}}; }

// It is bound by power: 94% of the cycles issue a vector instruction, and the
// clock falls to 1.97 GHz (2.29 in a loop of multiply-adds alone) under the 1485
// multiply-adds per entry of its 2160 instructions (2^24 points, 2.35 * 10^8
// entries: 16.1 ms, 1.46 * 10^10 entries/s).  A 9% shorter loop gained 1.5%; only
// fewer multiply-adds per entry would gain more.
template <class F>
__global__ void __launch_bounds__(256) k_accumulate29(const MsmSeg *__restrict__ segs, uint32_t Kj,
                                                      const uint32_t *__restrict__ sorted,
                                                      const uint32_t *__restrict__ off, uint32_t K, ChunkLen chunk,
                                                      const uint32_t *__restrict__ pts29,
                                                      uint32_t *__restrict__ buckets29,
                                                      uint32_t *__restrict__ carry29,
                                                      uint32_t *__restrict__ carry_key) {
  static_assert(std::is_same<F, Fq>::value, "29-bit limbs are for the base field");
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t E = off[K], L = chunk(E, K);
  const uint64_t e0l = (uint64_t)t * L;
  if (e0l >= E) return;
  const uint32_t e0 = (uint32_t)e0l;
  const uint32_t e1 = min(e0 + L, E);
  carry_key[t] = 0xFFFFFFFFu;
  uint32_t key = find_key(off, K, e0);
  uint32_t kend = off[key + 1];
  bool owned = off[key] == e0;
  uint32_t mem = key / Kj;
  // table runs pass no pts29: each member reads its own table slice
  const uint32_t *points = pts29 ? pts29 + (uint64_t)segs[mem].qbase * 16 : segs[mem].points;
  uint32_t nkey = key, nkend = kend;  // bucket of the entry being prefetched
  XYZZ29 acc = inf29();
  bool ainf = true;
  IndexReader ir(sorted, e0);
  uint32_t nv = ir.at(e0);
  uint32_t nx[8], ny[8];
  {
    const uint32_t *pp = points + (uint64_t)(nv & 0x7FFFFFFFu) * 16;
    ld8(nx, pp);
    ld8(ny, pp + 8);
  }
  for (uint32_t e = e0; e < e1;) {
    const uint32_t v = nv;
    const Fq29 x = unpack29(nx);
    Fq29 y = unpack29(ny);
    e++;
    if (e < e1) {
      if (e == nkend) {
        nkey = key_from(off, K, nkey + 1, e);
        nkend = off[nkey + 1];
        const uint32_t m2 = nkey / Kj;
        if (m2 != mem) {
          mem = m2;
          points = pts29 ? pts29 + (uint64_t)segs[mem].qbase * 16 : segs[mem].points;
        }
      }
      nv = ir.at(e);
      const uint32_t *pp = points + (uint64_t)(nv & 0x7FFFFFFFu) * 16;
      ld8(nx, pp);
      ld8(ny, pp + 8);
    }
    const Fq29 yn = neg29_loose<2>(y);  // 2q - y for a negative digit
    if (v >> 31) y = yn;
    madd29(acc, ainf, x, y);
    if (e == kend || e == e1) {
      if (owned) {
        store29(buckets29 + (uint64_t)key * Slot29<F>::SW, acc);
      } else {
        store29(carry29 + (uint64_t)t * Slot29<F>::SW, acc);
        carry_key[t] = key;
      }
      acc = inf29();
      ainf = true;
      owned = true;
      key = nkey;
      kend = nkend;
    }
  }
}

__device__ __forceinline__ XYZZ2_29 inf2_29() { return {Fq2_29{}, f2one29(), Fq2_29{}, Fq2_29{}}; }

// signed entry v of a G2 run: the point in the 2^261 form, y negated for a
// negative digit
__device__ __forceinline__ void load2_29(const uint32_t *points, uint32_t v, Fq2_29 &x, Fq2_29 &y) {
  const uint32_t *pp = points + (uint64_t)(v & 0x7FFFFFFFu) * 32;
  uint32_t w[8];
  ld8(w, pp);
  x.c0 = unpack29(w);
  ld8(w, pp + 8);
  x.c1 = unpack29(w);
  ld8(w, pp + 16);
  y.c0 = unpack29(w);
  ld8(w, pp + 24);
  y.c1 = unpack29(w);
  if (v >> 31) {
    y.c0 = sub29<1>(Fq29{}, y.c0);
    y.c1 = sub29<1>(Fq29{}, y.c1);
  }
}

// G2 bucket loop on 29-bit limbs: as k_accumulate29, without the next-point
// prefetch (no registers to spare; the second resident wave hides the
// loads), held to two waves per SIMD.  The rare doubling reloads its point.
template <class F>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
k_accumulate29_g2(const MsmSeg *__restrict__ segs, uint32_t Kj, const uint32_t *__restrict__ sorted,
                  const uint32_t *__restrict__ off, uint32_t K, ChunkLen chunk, const uint32_t *__restrict__ pts29,
                  uint32_t *__restrict__ buckets29, uint32_t *__restrict__ carry29,
                  uint32_t *__restrict__ carry_key) {
  static_assert(std::is_same<F, Fq2>::value, "the G2 loop");
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t E = off[K], L = chunk(E, K);
  const uint64_t e0l = (uint64_t)t * L;
  if (e0l >= E) return;
  const uint32_t e0 = (uint32_t)e0l;
  const uint32_t e1 = min(e0 + L, E);
  carry_key[t] = 0xFFFFFFFFu;
  uint32_t key = find_key(off, K, e0);
  uint32_t kend = off[key + 1];
  bool owned = off[key] == e0;
  uint32_t mem = key / Kj;
  const uint32_t *points = pts29 ? pts29 + (uint64_t)segs[mem].qbase * 32 : segs[mem].points;
  uint32_t nkey = key, nkend = kend;  // bucket of entry e after the increment
  XYZZ2_29 acc = inf2_29();
  bool ainf = true;
  IndexReader ir(sorted, e0);
  for (uint32_t e = e0; e < e1;) {
    const uint32_t v = ir.at(e);
    const uint32_t *cur = points;
    Fq2_29 x, y;
    load2_29(cur, v, x, y);
    e++;
    if (e < e1 && e == nkend) {
      nkey = key_from(off, K, nkey + 1, e);
      nkend = off[nkey + 1];
      const uint32_t m2 = nkey / Kj;
      if (m2 != mem) {
        mem = m2;
        points = pts29 ? pts29 + (uint64_t)segs[mem].qbase * 32 : segs[mem].points;
      }
    }
    if (!madd2_29(acc, ainf, x, y)) {
      Fq2_29 x2, y2;
      load2_29(cur, v, x2, y2);
      acc = dbl2_29_affine(x2, y2);
    }
    if (e == kend || e == e1) {
      if (owned) {
        store29(buckets29 + (uint64_t)key * Slot29<F>::SW, acc);
      } else {
        store29(carry29 + (uint64_t)t * Slot29<F>::SW, acc);
        carry_key[t] = key;
      }
      acc = inf2_29();
      ainf = true;
      owned = true;
      key = nkey;
      kend = nkend;
    }
  }
}

// 29-bit slot access for the carry, fix-up and reduction kernels
__device__ __forceinline__ void load4x29(const uint32_t *s, Fq29 &a, Fq29 &b, Fq29 &c, Fq29 &e) {
  const uint4 *s4 = reinterpret_cast<const uint4 *>(s);
  uint32_t w[36];
#pragma unroll
  for (int q = 0; q < 9; q++) {
    const uint4 v = s4[q];
    w[4 * q] = v.x;
    w[4 * q + 1] = v.y;
    w[4 * q + 2] = v.z;
    w[4 * q + 3] = v.w;
  }
#pragma unroll
  for (int i = 0; i < 9; i++) {
    a.l[i] = w[i];
    b.l[i] = w[9 + i];
    c.l[i] = w[18 + i];
    e.l[i] = w[27 + i];
  }
}
__device__ __forceinline__ void load29(const uint32_t *s, XYZZ29 &a) { load4x29(s, a.X, a.Y, a.ZZ, a.ZZZ); }
__device__ __forceinline__ void load29(const uint32_t *s, XYZZ2_29 &a) {
  load4x29(s, a.X.c0, a.X.c1, a.Y.c0, a.Y.c1);
  load4x29(s + 36, a.ZZ.c0, a.ZZ.c1, a.ZZZ.c0, a.ZZZ.c1);
}
// 256-thread workgroups of `count` groups of lanes
template <class F> static uint32_t grp_blocks(uint64_t count) {
  return (uint32_t)((count * Grp<F>::N + 255) / 256);
}
template <class F> struct Acc29;
template <> struct Acc29<Fq> {
  using T = XYZZ29;
  __device__ __forceinline__ static T inf() { return inf29(); }
};
template <> struct Acc29<Fq2> {
  using T = XYZZ2_29;
  __device__ __forceinline__ static T inf() { return inf2_29(); }
};

// Carries of one bucket occupy the consecutive chunk slots t0+1 .. t1 of a
// bucket [s, e) (t0 = s/L, t1 = (e-1)/L), chain index 0 .. t1-t0-1.  k_fixup adds
// up to `keep` slots of its bucket's chain to the bucket: one with a lane per
// bucket, where a second would keep whole waves for a few lanes (the G1 fix-up of a
// 50000-constraint proof 113 -> 163 us), eight with a group per bucket, where the
// buckets are few and their chains long.  Longer chains are thinned first (a
// bucket far larger than a chunk: skewed digits, small witness values, a narrow top
// window): in the round of step 8^r the slot at chain index i (i % 8^(r+1) == 0) adds the slots at i + k*8^r, k = 1..7, that
// lie in the chain, if the chain has more than keep * 8^r of them.  The slots read
// are never written in the same round.  Slots are 29-bit (SW words).
// A group of lanes per slot (quad29.h): a round is a chain of up to seven
// additions, and few slots of a round head one.
template <class F>
__global__ void __launch_bounds__(256) k_carry_round(const uint32_t *__restrict__ off, uint32_t K, ChunkLen chunk,
                                                     uint32_t *__restrict__ carry,
                                                     const uint32_t *__restrict__ carry_key, uint32_t step,
                                                     uint32_t keep) {
  constexpr int SW = Slot29<F>::SW;
  constexpr uint32_t GN = Grp<F>::N;
  const uint64_t u = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / GN;
  const uint32_t E = off[K], L = chunk(E, K);
  uint32_t i = 0, len = 0;
  if (u * L < E) {
    const uint32_t key = carry_key[u];
    if (key != 0xFFFFFFFFu) {
      const uint32_t t0 = off[key] / L, t1 = (off[key + 1] - 1) / L;
      i = (uint32_t)u - (t0 + 1);
      len = t1 - t0;
    }
  }
  const bool head = ((uint64_t)i & (8ull * step - 1)) == 0 && (uint64_t)i + step < len &&
                    len > (uint64_t)keep * step;
  if (!__any(head)) return;
  Fq29 a = {};
  if (head) grp_load<F>(carry + u * SW, a);
#pragma unroll 1
  for (uint64_t k = 1; k < 8; k++) {
    const bool more = head && i + k * step < len;
    if (!__any(more)) break;
    Fq29 b = {};  // infinity where the chain has ended
    if (more) grp_load<F>(carry + (u + k * step) * SW, b);
    grp_add<F>(a, b);
  }
  if (head) grp_store<F>(carry + u * SW, a);
}

// The slots kCarryTail apart that the rounds of step 1 .. kCarryTail / 8 leave in a
// chain of more than keep * kCarryTail, summed by the wave that finds the chain's
// head: its groups take every NG-th slot each, then join.  Chains this long are
// few, so one launch that looks for them costs less than a launch per round.
static constexpr uint32_t kCarryTail = 64;
template <class F>
__global__ void __launch_bounds__(256) k_carry_tail(const uint32_t *__restrict__ off, uint32_t K, ChunkLen chunk,
                                                    uint32_t *carry, const uint32_t *__restrict__ carry_key, uint32_t keep) {
  constexpr uint32_t SW = Slot29<F>::SW, GN = Grp<F>::N, NG = 64 / GN;
  const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t E = off[K], L = chunk(E, K);
  uint32_t len = 0;
  if ((uint64_t)u * L < E) {
    const uint32_t key = carry_key[u];
    if (key != 0xFFFFFFFFu) {
      const uint32_t t0 = off[key] / L, t1 = (off[key + 1] - 1) / L;
      if (u == t0 + 1) len = t1 - t0;
    }
  }
  uint64_t heads = __ballot(len > keep * kCarryTail);
  const uint32_t lane = threadIdx.x & 63, grp = lane / GN;
  for (; heads; heads &= heads - 1) {
    const uint32_t h = __builtin_ctzll(heads);
    const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)len, h);
    uint32_t *base = carry + (uint64_t)(u - lane + h) * SW;
    const uint32_t count = (n + kCarryTail - 1) / kCarryTail;
    Fq29 a = {};
    if (grp < count) grp_load<F>(base + (uint64_t)grp * kCarryTail * SW, a);
#pragma unroll 1
    for (uint32_t k0 = NG; k0 < count; k0 += NG) {
      Fq29 b = {};
      if (k0 + grp < count) grp_load<F>(base + (uint64_t)(k0 + grp) * kCarryTail * SW, b);
      grp_add<F>(a, b);
    }
#pragma unroll 1
    for (uint32_t d = NG / 2; d > 0; d /= 2) {
      Fq29 b;
#pragma unroll
      for (int i = 0; i < 9; i++) b.l[i] = __shfl_down(a.l[i], d * GN, 64);
      if (grp >= d) b = Fq29{};
      grp_add<F>(a, b);
    }
    if (grp == 0) grp_store<F>(base, a);
  }
}

// the slots apart that the rounds leave of a chain with keep = 8: at most eight, or
// its head
__device__ __forceinline__ uint32_t chain_stride(uint32_t len) {
  return len <= 8 ? 1 : len <= 64 ? 8 : len <= 512 ? 64 : len;
}
static_assert(kCarryTail == 64, "chain_stride");

// every bucket gets its chain: a lane per bucket, or (k_fixup_groups) a group
template <class F>
__global__ void __launch_bounds__(256) k_fixup(const uint32_t *__restrict__ off, uint32_t K, ChunkLen chunk,
                                               uint32_t *__restrict__ buckets,
                                               const uint32_t *__restrict__ carry) {
  constexpr int SW = Slot29<F>::SW;
  using A = typename Acc29<F>::T;
  uint32_t key = blockIdx.x * blockDim.x + threadIdx.x;
  if (key >= K) return;
  const uint32_t s = off[key], e = off[key + 1];
  if (e == s) return;
  const uint32_t L = chunk(off[K], K), t0 = s / L, len = (e - 1) / L - t0;
  if (len == 0) return;
  A acc, c;
  load29(buckets + (uint64_t)key * SW, acc);
  load29(carry + (uint64_t)(t0 + 1) * SW, c);
  xadd29(acc, c);
  store29(buckets + (uint64_t)key * SW, acc);
}
template <class F>
__global__ void __launch_bounds__(256) k_fixup_groups(const uint32_t *__restrict__ off, uint32_t K, ChunkLen chunk,
                                                      uint32_t *__restrict__ buckets,
                                                      const uint32_t *__restrict__ carry) {
  constexpr uint32_t SW = Slot29<F>::SW, GN = Grp<F>::N;
  const uint32_t key = (uint32_t)(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / GN);
  const uint32_t L = chunk(off[K], K);
  uint32_t t0 = 0, len = 0;
  if (key < K) {
    const uint32_t s = off[key], e = off[key + 1];
    if (e != s) {
      t0 = s / L;
      len = (e - 1) / L - t0;
    }
  }
  if (!__any(len != 0)) return;
  const uint32_t stride = chain_stride(len);
  Fq29 acc = {};
  if (len) grp_load<F>(buckets + (uint64_t)key * SW, acc);
#pragma unroll 1
  for (uint32_t k = 0; __any(k < len); k += stride) {
    Fq29 c = {};
    if (k < len) grp_load<F>(carry + (uint64_t)(t0 + 1 + k) * SW, c);
    grp_add<F>(acc, c);
  }
  if (len) grp_store<F>(buckets + (uint64_t)key * SW, acc);
}

// the carries into their buckets
template <class F>
static void carry_chains(const uint32_t *off, uint32_t K, const MsmPlan &pl, uint32_t *buckets, uint32_t *carry,
                         const uint32_t *carry_key, hipStream_t st) {
  // from two waves of buckets per SIMD on a lane each fills the chip, and chains are
  // few or short; below, the chains are what is waited for.  Rounds and fix-up
  // together, keep = 1 with lanes against 8 with groups: 32768 G1 buckets of 49
  // entries 112 against 47 us, 262144 of 52 equal within 2% of the multiexp
  const bool lanes = K >= 1u << 17;
  const uint32_t keep = lanes ? 1 : 8;
  for (uint32_t step = 1; step < kCarryTail && keep * step < pl.max_chunks; step *= 8)
    k_carry_round<F><<<grp_blocks<F>(pl.max_chunks), 256, 0, st>>>(off, K, pl.chunk, carry, carry_key, step, keep);
  if (pl.max_chunks > keep * kCarryTail)
    k_carry_tail<F><<<(uint32_t)((pl.max_chunks + 255) / 256), 256, 0, st>>>(off, K, pl.chunk, carry, carry_key, keep);
  if (lanes)
    k_fixup<F><<<(K + 127) / 128, 128, 0, st>>>(off, K, pl.chunk, buckets, carry);
  else
    k_fixup_groups<F><<<grp_blocks<F>(K), 256, 0, st>>>(off, K, pl.chunk, buckets, carry);
}

// ------------------------------------------------------------ window sums
// sum_b (b + 1) bucket_b of every window, in place in the bucket slots.
//
// A node stands for a run of buckets of one window and holds K points at the
// start of the run's slots: R, the sum of its buckets, A, and C_0 .. C_(K-3),
// where its weighted sum is A + Lr (C_0 + 2 C_1 + 4 C_2 + ...).  The first
// nodes are segments of Lr buckets (k_bucket_reduce: running sums; A weights
// bucket i of the segment i + 1).  Two neighbouring nodes of equal length make
// one of twice the length (k_tree): R, A and every C_j add, and the upper
// node's R becomes the new C, whose weight is the lower one's length.  So a
// window of B buckets takes 2 B additions, about 2 Lr + log2(B / Lr) of them in
// a row, and no doublings before the last step (k_window_horner), log2(B)
// doublings and additions of C's on rows of lanes.  The additions run on groups
// of lanes (quad29.h), as the chain is what costs.
// Measured, 2^20 points (c = 16, 8 x 32768 buckets): 101 + 67 + 38 us; segments
// each multiplied by their offset and summed by lanes, 256 + 118 us.

// a group per (window, segment)
template <class F>
__global__ void __launch_bounds__(256) k_bucket_reduce(const uint32_t *__restrict__ off, uint32_t *buckets,
                                                       uint32_t nseg, uint32_t Lr) {
  constexpr int SW = Slot29<F>::SW;
  constexpr uint32_t GN = Grp<F>::N;
  const uint32_t seg = (uint32_t)(((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / GN);
  const bool live = seg < nseg;
  const uint64_t lo = (uint64_t)seg * Lr;  // windows follow each other: key = w * B + s * Lr
  Fq29 run = {}, acc = {};
#pragma unroll 1
  for (int b = (int)Lr - 1; b >= 0; b--) {
    Fq29 bk = {};
    const uint64_t key = lo + (uint32_t)b;
    if (live && off[key + 1] != off[key]) grp_load<F>(buckets + key * SW, bk);
    grp_add<F>(run, bk);
    grp_add<F>(acc, run);
  }
  if (live) {
    grp_store<F>(buckets + lo * SW, run);
    grp_store<F>(buckets + (lo + 1) * SW, acc);
  }
}

// the same with a lane per segment
template <class F>
__global__ void __launch_bounds__(256) k_bucket_reduce_lanes(const uint32_t *__restrict__ off, uint32_t *buckets,
                                                             uint32_t nseg, uint32_t Lr) {
  constexpr int SW = Slot29<F>::SW;
  using A = typename Acc29<F>::T;
  const uint32_t seg = blockIdx.x * blockDim.x + threadIdx.x;
  if (seg >= nseg) return;
  const uint64_t lo = (uint64_t)seg * Lr;
  A run = Acc29<F>::inf(), acc = Acc29<F>::inf();
#pragma unroll 1
  for (int b = (int)Lr - 1; b >= 0; b--) {
    const uint64_t key = lo + (uint32_t)b;
    if (off[key + 1] != off[key]) {
      A bk;
      load29(buckets + key * SW, bk);
      xadd29(run, bk);
    }
    xadd29(acc, run);
  }
  store29(buckets + lo * SW, run);
  store29(buckets + (lo + 1) * SW, acc);
}

// Threads of the largest k_tree workgroup (the G2 addition takes more than the
// 128 registers a lane of a 1024-thread workgroup has), and its LDS.
template <class F> static constexpr uint32_t kTreeThreads = std::is_same<F, Fq>::value ? 1024 : 512;
static constexpr uint32_t kTreeLds = 65536;

// One workgroup joins n (a power of two) nodes of `span` slots and K points
// each into one of n * span slots.  It has a group for each of the (n / 2) K
// additions and n / 2 copies of its first level; later levels have fewer.
template <class F>
__global__ void __launch_bounds__(kTreeThreads<F>) k_tree(uint32_t *slots, uint32_t span, uint32_t K,
                                                               uint32_t n) {
  constexpr int SW = Slot29<F>::SW;
  constexpr uint32_t GN = Grp<F>::N;
  extern __shared__ uint32_t sh[];  // n * K slots: point k of node i at k * n + i
  uint32_t *base = slots + (uint64_t)blockIdx.x * n * span * SW;
  for (uint32_t w = threadIdx.x; w < n * K * SW; w += blockDim.x) {
    const uint32_t i = w / (K * SW), r = w - i * (K * SW), k = r / SW;
    sh[(k * n + i) * SW + (r - k * SW)] = base[(uint64_t)i * span * SW + r];
  }
  __syncthreads();
  const uint32_t grp = threadIdx.x / GN;
  for (uint32_t m = n; m > 1; m >>= 1, K++) {
    const uint32_t h = m >> 1;
    // point k of the new node i; the quads after the additions' copy the upper R
    const uint32_t k = grp / h, i = grp - k * h;
    Fq29 a = {}, b = {};
    const bool add = k < K, copy = k == K;
    if (add) {
      grp_load<F>(sh + (k * m + 2 * i) * SW, a);
      grp_load<F>(sh + (k * m + 2 * i + 1) * SW, b);
    } else if (copy) {
      grp_load<F>(sh + (2 * i + 1) * SW, a);
    }
    if (__any(add)) grp_add<F>(a, b);
    __syncthreads();
    if (add || copy) grp_store<F>(sh + (k * h + i) * SW, a);
    __syncthreads();
  }
  for (uint32_t w = threadIdx.x; w < K * SW; w += blockDim.x) base[w] = sh[w];
}

// sum_i 2^(step i) v_i over n stored slots, v_i at base + i * stride words, by a
// workgroup of kChainThreads; the result is in sum (G1: of the first wave).
// G1: each of the four waves takes a run of the values, then the runs join
// pairwise: as many doublings in a row, fewer additions.  lds: kChainLds words.
static constexpr uint32_t kChainThreads = 256;
template <class F> static constexpr uint32_t kChainLds = std::is_same<F, Fq>::value ? 4 * 36 : 1;
__device__ __forceinline__ void horner(RowAcc<Fq> &sum, uint32_t *lds, const uint32_t *base, uint32_t stride,
                                       uint32_t n, uint32_t step) {
  // runs of a, b, a and the rest, the last the longest: the waves wait for each
  // other before a join, and with equal even runs no wait adds a doubling
  const uint32_t a = n / 4, b = (n - 2 * a) / 2, wave = threadIdx.x / 64;
  const uint32_t start[5] = {0, a, a + b, 2 * a + b, n};
  const uint32_t lo = wave == 0 ? start[0] : wave == 1 ? start[1] : wave == 2 ? start[2] : start[3];
  const uint32_t hi = wave == 0 ? start[1] : wave == 1 ? start[2] : wave == 2 ? start[3] : start[4];
  sum.clear();
#pragma unroll 1
  for (uint32_t i = hi; i-- > lo;) {
    sum.dbl(step);
    sum.add(base + (uint64_t)i * stride);
  }
#pragma unroll 1
  for (uint32_t d = 1; d < 4; d *= 2) {
    sum.store(lds + wave * 36);
    __syncthreads();
    if (wave % (2 * d) == 0) {
      sum.set(lds + (wave + d) * 36);
      sum.dbl(step * (d == 1 ? a : a + b));
      sum.add(lds + wave * 36);
    }
    __syncthreads();
  }
}
__device__ __forceinline__ void horner(RowAcc<Fq2> &sum, uint32_t *, const uint32_t *base, uint32_t stride,
                                       uint32_t n, uint32_t step) {
#pragma unroll 1
  for (uint32_t i = n - 1; i-- > 0;) {  // sum starts as the last value
    sum.dbl(step);
    sum.add(base + (uint64_t)i * stride);
  }
}

// A + Lr (C_0 + 2 C_1 + ...) of each window's last node (one workgroup per
// window), a 29-bit slot of limbs below 2^29 + 4
template <class F>
__global__ void __launch_bounds__(kChainThreads) k_window_horner(const uint32_t *__restrict__ slots, uint32_t B,
                                                                 uint32_t K, uint32_t lgLr,
                                                                 uint32_t *__restrict__ wsum) {
  constexpr int SW = Slot29<F>::SW;
  const uint32_t *node = slots + (uint64_t)blockIdx.x * B * SW;
  if constexpr (std::is_same<F, Fq>::value) {
    __shared__ uint32_t lds[kChainLds<F>];
    RowAcc<F> acc;
    horner(acc, lds, node + 2 * SW, SW, K - 2, 1);
    if (threadIdx.x >= 64) return;
    acc.dbl(lgLr);
    acc.add(node + SW);
    acc.store(wsum + (uint64_t)blockIdx.x * SW);
  } else {
    __shared__ uint32_t lds[RowAcc<F>::kLds];
    RowAcc<F> acc(lds, node + (uint64_t)(K - 1) * SW);
    if (K > 2) {
      horner(acc, lds, node + 2 * SW, SW, K - 2, 1);
      acc.dbl(lgLr);
      acc.add(node + SW);
    }
    acc.store(wsum + (uint64_t)blockIdx.x * SW);
  }
}

template <class F>
void window_sums(const uint32_t *off, uint32_t *buckets, uint32_t nwin, uint32_t B, uint32_t Lr, uint32_t *wsum,
                 hipStream_t st) {
  const uint32_t nseg = nwin * (B / Lr);
  // From 2^20 buckets (a wave of segments per SIMD) the additions fill the GPU
  // with a lane each, which is the fewest instructions; below, quads shorten
  // the chain (7 x 2^18 buckets: 396 us against 583).
  if ((uint64_t)nwin * B >= 1u << 20)
    k_bucket_reduce_lanes<F><<<(nseg + 255) / 256, 256, 0, st>>>(off, buckets, nseg, Lr);
  else
    k_bucket_reduce<F><<<grp_blocks<F>(nseg), 256, 0, st>>>(off, buckets, nseg, Lr);
  uint32_t N = B / Lr, span = Lr, K = 2;
  while (N > 1) {
    uint32_t n = 2;
    constexpr uint32_t GN = Grp<F>::N;
    while (n < N && n * (K + 1) * GN <= kTreeThreads<F> && 2 * n * K * Slot29<F>::SW * 4 <= kTreeLds) n *= 2;
    const uint32_t th = (n / 2 * (K + 1) * GN + 63) / 64 * 64;  // a group per addition and copy of the first level
    k_tree<F><<<nwin * (N / n), th, n * K * Slot29<F>::SW * 4, st>>>(buckets, span, K, n);
    for (uint32_t m = n; m > 1; m >>= 1) K++;
    span *= n;
    N /= n;
  }
  k_window_horner<F><<<nwin, kChainThreads, 0, st>>>(buckets, B, K, 31 - __builtin_clz(Lr), wsum);
}

// One workgroup per member: Horner over its W window sums (c doublings each),
// written as a canonical affine point to the member's output.  The chain is
// serial and latency bound, so each product is spread over a row of lanes and
// the products of a step run on different rows (row29.h): G1 in waves that
// hold a point in registers each and take a part of the windows, G2 in four
// waves that hold every value in LDS (coop29.h).  Infinity is tracked in a flag every lane holds.
// Measured: 120 doublings 174 us on G1, 273 on G2 (whole scalars' 248 doublings
// with one lane per product: 855 and 1997 us).  One window (table runs: the
// inversion and the conversions): 33 us, 167 with a bit-by-bit Euclid on one lane.
template <class F>
__global__ void __launch_bounds__(kChainThreads) k_final(const MsmSeg *__restrict__ segs,
                                                         const uint32_t *__restrict__ wsum, uint32_t W, uint32_t c) {
  const uint32_t j = blockIdx.x;
  uint32_t *out = segs[j].out;
  if (segs[j].n == 0) {
    if (threadIdx.x == 0) store_affine(out, Affine<F>{F::zero(), F::one()});
    return;
  }
  constexpr int SW = Slot29<F>::SW;
  const uint32_t *ws = wsum + (uint64_t)j * W * SW;
  if constexpr (std::is_same<F, Fq>::value) {
    __shared__ uint32_t lds[kChainLds<F>];
    RowAcc<F> acc;
    horner(acc, lds, ws, SW, W, c);
    if (threadIdx.x < 64) acc.store_affine_to(out);
  } else {
    __shared__ uint32_t lds[RowAcc<F>::kLds];
    RowAcc<F> acc(lds, ws + (uint64_t)(W - 1) * SW);
    horner(acc, lds, ws, SW, W, c);
    acc.store_affine_to(out);
  }
}

// The sort's placement passes over the counted and scanned digits: pass 1
// (bins by hi) and pass 2 (buckets by lo), for a group of J members of pl.W
// windows whose scalars have Wwin windows each (pl.W, or Wt for the one-window
// members of table runs), into offsets (Ktot + 1) and sorted.
static inline void sort_place(const MsmPlan &pl, uint32_t Wwin, const uint32_t *digits, const MsmSeg *segs,
                              const uint32_t *cnt, uint32_t *tix, uint16_t *tlo, uint32_t *offsets,
                              uint32_t *sorted, hipStream_t st) {
  const uint32_t sb = pl.c - 1 - pl.hb, HB = 1u << pl.hb;
  const uint32_t nblk = (uint32_t)(pl.W * pl.tiles), Wtot = pl.J * pl.W, Ktot = pl.J * pl.K;
  if (pl.max_entries < (1ull << 27))
    k_sort_scatter1<true><<<nblk, SORT_THREADS, 0, st>>>(digits, segs, pl.J, sb, pl.st, HB, pl.W, Wwin, cnt, tix,
                                                          tlo);
  else
    k_sort_scatter1<false><<<nblk, SORT_THREADS, 0, st>>>(digits, segs, pl.J, sb, pl.st, HB, pl.W, Wwin, cnt, tix,
                                                           tlo);
  // the 8192-entry tile keeps 49 KB of staging in LDS beside 3 * 2^sb counter
  // words: used up to sb = 10 (61 KB); wider windows take the 4096 tile
  const uint32_t lds = 3 * (1u << sb) * 4;
  // a segment holds at most a member's points; the long ones have eight times
  // the average, and more than four tiles
  const uint64_t longest = std::max<uint64_t>(4 * SORT_TILE, 8 * (pl.most >> pl.hb));
  const uint32_t split = pl.most > longest ? (uint32_t)longest : 0xFFFFFFFFu;
  if (pl.max_entries < (1ull << 27) || sb > 10)
    k_sort_pass2<SORT_TILE, SORT_THREADS, false><<<Wtot * HB, SORT_THREADS, lds, st>>>(
        tix, tlo, cnt, segs, HB, sb, pl.st, pl.W, Wwin, Ktot, split, offsets, sorted);
  else
    k_sort_pass2<2 * SORT_TILE, SORT_THREADS, false><<<Wtot * HB, SORT_THREADS, lds, st>>>(
        tix, tlo, cnt, segs, HB, sb, pl.st, pl.W, Wwin, Ktot, split, offsets, sorted);
  if (split != 0xFFFFFFFFu)
    k_sort_pass2<SORT_TILE, 1024, true><<<Wtot * HB, 1024, lds, st>>>(tix, tlo, cnt, segs, HB, sb, pl.st, pl.W, Wwin,
                                                                      Ktot, split, offsets, sorted);
}

// Enqueue the whole pipeline for one group on stream st.  segs is the
// group's device descriptor table (J + 1 entries); ws is carved in the order
// msm_workspace_bytes assumes.  No allocation, no host synchronisation and no
// memset nodes, so the sequence can be captured into a graph.
template <class F>
int msm_run(void *ws, const MsmPlan &pl, const MsmSeg *segs, hipStream_t st, StageTimer *tm) {
  const bool g2 = FieldIO<F>::NW == 16;
  Carver cv(ws);
  const uint32_t hi_bits = pl.hb;
  const uint32_t sb = pl.c - 1 - hi_bits, HB = 1u << hi_bits;
  const uint32_t nblk = (uint32_t)(pl.W * pl.tiles);
  const uint32_t ncnt = nblk * HB;
  const uint32_t nb = (ncnt + SCAN_TILE - 1) / SCAN_TILE;
  const uint32_t Ktot = pl.J * pl.K, Wtot = pl.J * pl.W;
  uint32_t *digits = cv.take<uint32_t>(pl.max_entries + 4);  // + 4: quad loads
  uint32_t *sorted = digits;  // pass 2 of the sort, which writes it, no longer reads them
  constexpr int PW = 2 * FieldIO<F>::NW, SW = Slot29<F>::SW;
  char *sortbuf = cv.take<char>(msm_sortbuf_bytes(pl, g2));
  Carver cs(sortbuf);
  uint32_t *pts29 = cs.take<uint32_t>((size_t)pl.n * PW);  // written by k_digits
  char *after = sortbuf + Carver::round((size_t)pl.n * PW * 4);
  Carver cs1(after);
  uint32_t *tix = cs1.take<uint32_t>(pl.max_entries);
  uint16_t *tlo = cs1.take<uint16_t>(pl.max_entries);
  uint32_t *cnt = cv.take<uint32_t>((size_t)ncnt + 1);
  uint32_t *bsum = cv.take<uint32_t>(nb);
  uint32_t *offsets = cv.take<uint32_t>((size_t)Ktot + 1);
  uint32_t *carry_key = cv.take<uint32_t>(pl.max_chunks);
  uint32_t *wsum = cv.take<uint32_t>((size_t)Wtot * SW);
  // the pass-1 arrays are free once the sort is done: bucket and carry slots
  Carver c29(after);
  uint32_t *b29 = c29.take<uint32_t>((size_t)Ktot * SW);
  uint32_t *cr29 = c29.take<uint32_t>((size_t)pl.max_chunks * SW);

  if (tm) tm->mark(0, st);
  if (pl.n > 0) {
    // few tiles leave most of the GPU idle: more threads share a tile's points, and
    // below 128 tiles other workgroups convert them: 5003 G2 points (5 tiles) 540 ->
    // 509 us, 20011 G1 points (10) 465 -> 456, 200000 (98) 695 -> 689
    const uint32_t tiles = (uint32_t)pl.tiles, DT = tiles >= 1024 ? 256 : tiles >= 128 ? 1024 : 512;
    const uint32_t conv = tiles >= 128 ? 0 : tiles * (kSortTile / pl.E / DT);
    auto *kd = conv ? digits_kernel<F, true>(pl.E) : digits_kernel<F, false>(pl.E);
    kd<<<tiles + conv, DT, pl.W * HB * 4, st>>>(segs, pl.J, pl.c, pl.W, sb, pl.st, HB, tiles, digits, cnt, pts29);
    CSK_CHECK_LAUNCH();
    scan_counts(cnt, ncnt, bsum, st);
    sort_place(pl, pl.W, digits, segs, cnt, tix, tlo, offsets, sorted, st);
    CSK_CHECK_LAUNCH();
    const uint32_t TB = g2 ? 128 : 256;
    uint32_t ga = (uint32_t)((pl.max_chunks + TB - 1) / TB);
    if (tm) tm->mark(1, st);
    if constexpr (std::is_same<F, Fq>::value)
      k_accumulate29<F><<<ga, TB, 0, st>>>(segs, pl.K, sorted, offsets, Ktot, pl.chunk, pts29, b29, cr29, carry_key);
    else
      k_accumulate29_g2<F><<<ga, TB, 0, st>>>(segs, pl.K, sorted, offsets, Ktot, pl.chunk, pts29, b29, cr29, carry_key);
    CSK_CHECK_LAUNCH();
    if (tm) tm->mark(2, st);
    carry_chains<F>(offsets, Ktot, pl, b29, cr29, carry_key, st);
    CSK_CHECK_LAUNCH();
    window_sums<F>(offsets, b29, Wtot, pl.B, pl.Lr, wsum, st);
    CSK_CHECK_LAUNCH();
  }
  k_final<F><<<pl.J, kChainThreads, 0, st>>>(segs, wsum, pl.W, pl.c);
  CSK_CHECK_LAUNCH();
  if (tm) tm->mark(3, st);
  return CSK_OK;
}


// ------------------------------------------------------------ fixed-base tables
// A table of points P_0 .. P_(n-1) for window width c holds Q[w * n_pad + i] =
// 2^(c w) P_i for w < Wt = floor(254 / c) + 1 (n_pad = n rounded up to the
// sort tile), in the 2^261 form the bucket loops read, and a bit per point,
// 1 unless P_i is at infinity.  With the signed c-bit digits d_(i,w) of k_i,
// sum_i k_i P_i = sum_(w, i) d_(i,w) Q[w * n_pad + i]: the multiexp runs as one
// member of Wt * n_pad points and one window, which sorts, accumulates and
// reduces exactly as a plain one; or, when large, as a group of Wt one-window
// members (member w: digit w of every scalar, points Q[w * n_pad ..]), whose
// buckets b are then summed over w and reduced once.  No doublings are needed
// between windows.

// one thread per point: its Wt table entries (an inversion each) and its bit;
// grid covers n_pad (a multiple of the sort tile) exactly
template <class F>
__global__ void __launch_bounds__(256) k_table_build(const uint32_t *__restrict__ pts, uint64_t n, uint64_t n_pad,
                                                     uint32_t c, uint32_t Wt, uint32_t *__restrict__ table,
                                                     uint32_t *__restrict__ live) {
  constexpr int PW = 2 * FieldIO<F>::NW;
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  Affine<F> p = {F::zero(), F::zero()};
  bool inf = true;
  if (i < n) {
    p = load_affine<F>(pts + i * PW);
    inf = affine_is_inf(p);
  }
  // 32 points per word; i & 31 == threadIdx.x & 31 (blocks of 256)
  const uint64_t m = __ballot(!inf);
  if ((threadIdx.x & 31) == 0 && i < n_pad) live[i >> 5] = (uint32_t)(m >> (threadIdx.x & 32));
  if (inf) return;
  XYZZ<F> acc = XYZZ<F>::from_affine(p);
  store_point29<1>(table + i * PW, p);
  for (uint32_t w = 1; w < Wt; w++) {
    for (uint32_t k = 0; k < c; k++) acc = xyzz_dbl(acc);
    store_point29<1>(table + ((uint64_t)w * n_pad + i) * PW, xyzz_to_affine(acc));
  }
}

namespace {  // curve-independent table kernels: one private copy per translation unit

// Digits of the table group: one workgroup per sort tile of scalars and run
// p (blockIdx.y; tiles past the run's table end return).  Member m = p * Wt +
// w (window w of run p) has digit array D[pbase_m + i], pbase_m = pbase_(p*Wt)
// + w * n_pad (as k_digits writes a one-window member at its concatenated
// points), empty (0xFFFFFFFF) for a zero digit, a point at infinity or i >= n.
// Counts go to cnt[cbase_m + hi * NT + tile], cbase_m = cbase_(p*Wt) + w * HB
// * NT, the member's pass-1 counters.  With a run's windows together (per = 1) it is
// member p, window w's tiles are w * NT + tile of it, and every window splits
// its buckets at s bits.
__global__ void __launch_bounds__(256) k_digits_tab(TabArgs args, const MsmSeg *__restrict__ segs, uint32_t per,
                                                    uint32_t c, uint32_t Wt, uint32_t s, uint32_t ts, uint32_t HB,
                                                    uint32_t *__restrict__ digits, uint32_t *__restrict__ cnt) {
  extern __shared__ uint32_t hist[];  // Wt * HB counters
  const uint32_t tile = blockIdx.x, p = blockIdx.y;
  const MsmSeg &g0 = segs[p * per];
  const uint64_t n = args.n[p];
  const uint32_t NT = (uint32_t)((n + kSortTile - 1) / kSortTile);
  if (tile >= NT) return;  // the whole workgroup: this run's table has fewer tiles
  const uint64_t n_pad = (uint64_t)NT * kSortTile;
  const uint32_t *__restrict__ scalars = args.s[p];
  const uint32_t *__restrict__ live = args.live[p];
  digits += g0.pbase;
  cnt += g0.cbase;
  for (uint32_t i = threadIdx.x; i < Wt * HB; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  for (uint32_t t = threadIdx.x; t < kSortTile; t += blockDim.x) {
    const uint64_t i = (uint64_t)tile * kSortTile + t;
    if (i >= n) {
      for (uint32_t w = 0; w < Wt; w++) digits[(uint64_t)w * n_pad + i] = 0xFFFFFFFFu;
      continue;
    }
    uint32_t k[8];
    ld8(k, scalars + i * 8);
    reduce_mod_r(k);
    const bool zero = ((live[i >> 5] >> (i & 31)) & 1u) == 0;
    Digits<8> d;
    d.set(k, c);
    for (uint32_t w = 0; w < Wt; w++) {
      bool neg;
      const uint32_t b = d.take(neg);
      const bool lv = b != 0xFFFFFFFFu && !zero;
      digits[(uint64_t)w * n_pad + i] = lv ? b | ((uint32_t)neg << 31) : 0xFFFFFFFFu;
      if (lv) atomicAdd(&hist[w * HB + (b >> (w == Wt - 1 ? ts : s))], 1u);
    }
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < Wt * HB; i += blockDim.x) {
    const uint32_t w = i / HB, hi = i - w * HB;
    cnt[per == 1 ? ((uint64_t)hi * Wt + w) * NT + tile : (uint64_t)i * NT + tile] = hist[i];
  }
}

// merged[p * B + b] = sum over the J members of vector p (blockIdx.y) of their
// bucket b (empty buckets skipped)
template <class F>
__global__ void __launch_bounds__(256) k_merge_members(const uint32_t *__restrict__ off,
                                                       const uint32_t *__restrict__ buckets, uint32_t J, uint32_t B,
                                                       uint32_t *__restrict__ merged) {
  constexpr int SW = Slot29<F>::SW;
  using A = typename Acc29<F>::T;
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  const uint64_t p = blockIdx.y;
  off += p * J * B;
  buckets += p * J * B * SW;
  merged += p * B * SW;
  A acc = Acc29<F>::inf();
#pragma unroll 1
  for (uint32_t j = 0; j < J; j++) {
    const uint32_t key = j * B + b;
    if (off[key + 1] != off[key]) {
      A bk;
      load29(buckets + (uint64_t)key * SW, bk);
      xadd29(acc, bk);
    }
  }
  store29(merged + (uint64_t)b * SW, acc);
}

// o[k] = k for k <= B: bucket offsets under which every merged bucket is read
__global__ void __launch_bounds__(256) k_iota(uint32_t *__restrict__ o, uint32_t count) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < count) o[k] = k;
}

// one output descriptor per scalar vector (what k_final reads), and a sentinel
__global__ void k_put_outs(TabArgs args, uint32_t count, MsmSeg *osegs) {
  const uint32_t p = threadIdx.x;
  if (p > count) return;
  MsmSeg g = {};
  if (p < count) {
    g.out = args.o[p];
    g.n = 1;
  }
  osegs[p] = g;
}

}  // namespace

// Workspace of a table run over count scalar vectors, carved in this order
// by msm_run_table.
inline size_t msm_table_workspace_bytes(const MsmPlan &pl, bool g2, uint32_t count) {
  const uint32_t hi_bits = pl.hb;
  const uint64_t ncnt = (uint64_t)pl.W * (1u << hi_bits) * pl.tiles;
  const uint64_t nb = (ncnt + SCAN_TILE - 1) / SCAN_TILE;
  const uint64_t Ktot = (uint64_t)pl.J * pl.K;
  const uint64_t sb = g2 ? 288 : 144;
  const uint64_t sort = Carver::round(pl.max_entries * 4) + pl.max_entries * 2;
  const uint64_t slots = Carver::round(Ktot * sb) + pl.max_chunks * sb;
  size_t b = 0;
  b += Carver::round((pl.max_entries + 4) * 4);  // digits, then sorted
  b += Carver::round(sort > slots ? sort : slots);
  b += Carver::round((ncnt + 1) * 4);
  b += Carver::round(nb * 4);
  b += Carver::round((Ktot + 1) * 4);
  b += Carver::round(pl.max_chunks * 4);
  if (pl.J != count) {
    b += Carver::round((uint64_t)count * pl.B * sb);       // merged buckets
    b += Carver::round(((uint64_t)count * pl.B + 1) * 4);  // iota offsets
  }
  b += Carver::round((uint64_t)count * sb);               // their sums
  b += Carver::round((uint64_t)(count + 1) * sizeof(MsmSeg));  // output descriptors
  b += Carver::round(((uint64_t)pl.J + 1) * sizeof(MsmSeg));   // member descriptors
  return b + 4096;
}

// Enqueue count table multiexps (run p: scalar vector args.s[p] over its
// table -> args.o[p]): pl is the group plan of the runs as count members of all
// their windows, or as count * Wt one-window members m = p * Wt + w (W = 1),
// hsegs their host descriptors (a member reads its table, or the slice of its
// window, through its points pointer), Lrm the buckets of a reduction segment.
template <class F>
int msm_run_table(void *ws, const MsmPlan &pl, const MsmSeg *hsegs, const TabArgs &args, uint32_t count,
                  uint32_t Wt, uint32_t max_nt, uint32_t Lrm, hipStream_t st) {
  const bool g2 = FieldIO<F>::NW == 16;
  constexpr int SW = Slot29<F>::SW;
  Carver cv(ws);
  const uint32_t hi_bits = pl.hb;
  const uint32_t sb = pl.c - 1 - hi_bits, HB = 1u << hi_bits;
  const uint32_t nblk = (uint32_t)(pl.W * pl.tiles);
  const uint32_t ncnt = nblk * HB;
  const uint32_t nb = (ncnt + SCAN_TILE - 1) / SCAN_TILE;
  const uint32_t Ktot = pl.J * pl.K;
  uint32_t *digits = cv.take<uint32_t>(pl.max_entries + 4);
  uint32_t *sorted = digits;  // as in msm_run
  const uint64_t sortb = Carver::round(pl.max_entries * 4) + pl.max_entries * 2;
  const uint64_t slotb = Carver::round((uint64_t)Ktot * SW * 4) + pl.max_chunks * SW * 4;
  char *sortbuf = cv.take<char>(sortb > slotb ? sortb : slotb);
  Carver cs1(sortbuf);
  uint32_t *tix = cs1.take<uint32_t>(pl.max_entries);
  uint16_t *tlo = cs1.take<uint16_t>(pl.max_entries);
  Carver c29(sortbuf);  // the slots reuse the pass-1 arrays once the sort is done
  uint32_t *b29 = c29.take<uint32_t>((size_t)Ktot * SW);
  uint32_t *cr29 = c29.take<uint32_t>((size_t)pl.max_chunks * SW);
  uint32_t *cnt = cv.take<uint32_t>((size_t)ncnt + 1);
  uint32_t *bsum = cv.take<uint32_t>(nb);
  uint32_t *offsets = cv.take<uint32_t>((size_t)Ktot + 1);
  uint32_t *carry_key = cv.take<uint32_t>(pl.max_chunks);
  const uint32_t per = pl.J / count;  // members of a run
  uint32_t *merged = b29, *moff = offsets;
  if (per > 1) {
    merged = cv.take<uint32_t>((size_t)count * pl.B * SW);
    moff = cv.take<uint32_t>((size_t)count * pl.B + 1);
  }
  uint32_t *wsum = cv.take<uint32_t>((size_t)count * SW);
  MsmSeg *osegs = cv.take<MsmSeg>(count + 1);
  MsmSeg *segs = cv.take<MsmSeg>(pl.J + 1);

  CSK_HIP(hipMemcpyAsync(segs, hsegs, ((size_t)pl.J + 1) * sizeof(MsmSeg), hipMemcpyHostToDevice, st));
  k_put_outs<<<1, 128, 0, st>>>(args, count, osegs);
  k_digits_tab<<<dim3(max_nt, count), 256, Wt * HB * 4, st>>>(args, segs, per, pl.c, Wt, sb, per > 1 ? pl.st : sb, HB,
                                                                          digits, cnt);
  CSK_CHECK_LAUNCH();
  scan_counts(cnt, ncnt, bsum, st);
  // no window of a member of all windows is the top one
  sort_place(pl, per > 1 ? Wt : 0xFFFFFFFFu, digits, segs, cnt, tix, tlo, offsets, sorted, st);
  CSK_CHECK_LAUNCH();
  const uint32_t TB = g2 ? 128 : 256;
  const uint32_t ga = (uint32_t)((pl.max_chunks + TB - 1) / TB);
  if constexpr (std::is_same<F, Fq>::value)
    k_accumulate29<F><<<ga, TB, 0, st>>>(segs, pl.K, sorted, offsets, Ktot, pl.chunk, nullptr, b29, cr29, carry_key);
  else
    k_accumulate29_g2<F><<<ga, TB, 0, st>>>(segs, pl.K, sorted, offsets, Ktot, pl.chunk, nullptr, b29, cr29,
                                             carry_key);
  CSK_CHECK_LAUNCH();
  carry_chains<F>(offsets, Ktot, pl, b29, cr29, carry_key, st);
  CSK_CHECK_LAUNCH();
  if (per > 1) {
    k_merge_members<F><<<dim3((pl.B + TB - 1) / TB, count), TB, 0, st>>>(offsets, b29, Wt, pl.B, merged);
    k_iota<<<(uint32_t)(((uint64_t)count * pl.B + 1 + 255) / 256), 256, 0, st>>>(moff, count * pl.B + 1);
  }
  CSK_CHECK_LAUNCH();
  window_sums<F>(moff, merged, count, pl.B, Lrm, wsum, st);
  k_final<F><<<count, kChainThreads, 0, st>>>(osegs, wsum, 1, pl.c);
  CSK_CHECK_LAUNCH();
  return CSK_OK;
}

template <class F>
int msm_table_build(const uint32_t *pts, uint64_t n, uint64_t n_pad, uint32_t c, uint32_t Wt, uint32_t *table,
                    uint32_t *live, hipStream_t st) {
  k_table_build<F><<<(uint32_t)(n_pad / 256), 256, 0, st>>>(pts, n, n_pad, c, Wt, table, live);
  CSK_CHECK_LAUNCH();
  return CSK_OK;
}

}  // namespace csk
