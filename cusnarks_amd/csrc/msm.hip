// Pippenger multi-exponentiation for BN254 G1 / G2 on gfx950.
//
// Replaces the reference's Straus-8 GPU multiexp (cusnarks
// src/cuda/ecbn128_device.cu:508-565, 865-969, 1692-1866) and its CPU twin
// (ec_jacreduce_server_h, src/cuda/ec.cpp:1536-1704).  Both compute the same
// group element sum_i k_i P_i; the output here is the canonical affine point,
// so it is bit-identical to the reference's ec_jac2aff_h of its result.
//
// Pipeline (all on one stream, no host round trip):
//   1. k_digits      one thread per point: k mod r, split in two halves along
//                    the endomorphism (on G2 in four quarters, glv.h), signed
//                    c-bit digits of each for W windows; (window, |digit|)
//                    -> bucket key; histogram.
//   2. scan          exclusive prefix sum of the histogram -> bucket offsets.
//   3. k_scatter     counting-sort placement of (point index | sign) by key.
//   4. k_accumulate  each thread folds a fixed-length chunk of the sorted
//                    array into XYZZ bucket sums with mixed additions; runs
//                    that start in an earlier chunk are handed over as carries.
//   5. k_fixup       the owner of each bucket split over chunks adds the carries.
//   6. k_bucket_reduce  per (window, segment): sum B_b and sum (b+1) B_b by
//                    running sums.
//   7. k_tree, k_window_horner  per window: the segments joined pairwise, then
//                    their weights' powers of two.
//   8. k_final       Horner over the windows (c doublings each) -> affine.
#include <vector>
#include "internal.h"
#include "field.h"
#include "glv.h"
#include "msm.h"

namespace csk {

static constexpr int SCAN_TILE = 256 * 8;  // matches msm_impl.h
static constexpr uint32_t kMultiMembers = 8;         // multiexps of one call run as a group
static constexpr uint64_t kMultiPoints = 1ull << 23;  // points of such a group

static uint32_t floor_log2(uint64_t n) {
  uint32_t lg = 0;
  while ((1ull << (lg + 1)) <= n) lg++;
  return lg;
}

// ------------------------------------------------------------------ host side
uint32_t msm_choose_c(uint64_t n, bool g2, const csk_ctx *ctx, const csk_msm_cfg *cfg) {
  if (cfg && cfg->window_bits) return cfg->window_bits;
  const uint32_t lg = floor_log2(n);
  if (ctx && lg < 64 && ctx->tune[g2][lg].window_bits) return ctx->tune[g2][lg].window_bits;
  // windows whose top window keeps most of its bits (126, on G2 64 for c <= 13, is
  // (W-1) c + t with t close to c): a narrow top window puts every point in a few
  // buckets
  if (g2) return lg <= 7 ? 5 : lg <= 13 ? 11 : lg <= 18 ? 13 : 16;
  return lg <= 11 ? 8 : lg <= 14 ? 13 : lg <= 22 ? 16 : 19;
}

// Bits of the bucket index the sort's first pass bins by: the top 8 (at most
// c - 1), fewer for small members, so a second-pass workgroup (one per member,
// window and first-pass bin) gets about 2048 entries rather than a handful.
// The second pass keeps 3 * 2^(c-1-hb) counters in LDS, so hb >= c - 12.
static uint32_t plan_hi_bits(uint32_t c, uint64_t n_avg) {
  uint32_t hb = c - 1 < 8 ? c - 1 : 8;
  int ideal = (int)floor_log2(n_avg ? n_avg : 1) - 11;
  const int lo = (int)c - 12;
  if (ideal < lo) ideal = lo;
  if (ideal < 0) ideal = 0;
  if (ideal < (int)hb) hb = (uint32_t)ideal;
  return hb;
}

// Low bucket bits the second pass sorts the top window by.  That window
// holds only the top t = bits mod c bits of a scalar or of its half or
// quarter (below 2^bits, bits = 254, 126 or 64), and its digit, at most 2^t <= 2^(c-1), has no
// carry out, so its buckets are below 2^t: its first pass bins by the top hb of those t bits
// (all HB bins filled, as for the other windows) or, when t <= hb, by all of
// them, and each of its first-pass bins is then a single bucket.  Binning it
// like the others instead leaves most of its entries in a few bins, which the
// second pass takes one workgroup each for (c = 18 at 2^24 points: 22 ms).
static uint32_t plan_top_bits(uint32_t bits, uint32_t c, uint32_t hb) {
  const uint32_t t = bits % c;
  return t > hb ? t - hb : 0;
}

static void plan_chunks(MsmPlan &pl, uint32_t fixed) {
  const uint64_t K = (uint64_t)pl.J * pl.K;
  pl.chunk = {fixed, pl.E == 4 ? 4u : 8u};
  if (pl.max_entries >> 31 || K == 0 || K >> 32) return;  // a plan that msm_plan_ok refuses
  pl.L = pl.chunk((uint32_t)pl.max_entries, (uint32_t)K);
  pl.max_chunks = pl.chunk.most((uint32_t)pl.max_entries);
}

MsmPlan msm_group_plan(uint32_t c, uint32_t E, const uint64_t *n, uint32_t J, bool g2, uint32_t chunk,
                       uint32_t reduce_seg) {
  (void)g2;
  MsmPlan pl = {};
  pl.c = c;
  pl.E = E;
  pl.bits = E == 4 ? kGlsBits : E == 2 ? kGlvBits : kScalarBits;
  pl.W = pl.bits / c + 1;
  pl.B = 1u << (c - 1);
  pl.K = pl.W * pl.B;
  pl.J = J;
  for (uint32_t j = 0; j < J; j++) {
    pl.n += E * n[j];
    if (E * n[j] > pl.most) pl.most = E * n[j];
    pl.tiles += (E * n[j] + kSortTile - 1) / kSortTile;
  }
  pl.max_entries = pl.n * pl.W;
  pl.hb = plan_hi_bits(c, J ? pl.n / J : 0);
  pl.st = plan_top_bits(pl.bits, c, pl.hb);
  // buckets per reduction thread: aim for ~2^15 reduction threads
  const uint64_t Ktot = (uint64_t)J * pl.K;
  uint32_t lr = 16;
  if (reduce_seg) lr = reduce_seg < 2 ? 2 : reduce_seg;  // a segment keeps two sums in its slots
  else
    while (lr > 2 && Ktot / lr < (1u << 15)) lr >>= 1;
  if (lr > pl.B) lr = pl.B;
  pl.Lr = lr;
  pl.S = pl.B / pl.Lr;
  plan_chunks(pl, chunk);
  return pl;
}

// At widths where the parts have an entry more per point, whole scalars are the
// fewer additions of a large multiexp: 2^24 G1 points, c = 17, 16 entries a point 22.6
// ms, whole 15 and 21.2; c = 15 26.0 and 23.9; G2 c = 17 65.2 and 55.3.  The parts' fewer
// buckets, and half the doublings, then count 4 entries each and 3.7 million, which is
// where wire values, half of whose digits are 0, tie too: G1 c = 15 at 4.2 million
// points (uniform ones at 1), c = 17 at 6 (3), c = 20 at 17 (12); G2 c = 17 at 4.3 (2.7).
// A whole scalar's narrow top window (c = 14: 254 is 18 * 14 + 2) takes the gain back:
// 27.1 and 27.8 ms.
static bool split_pays(const MsmPlan &split, const MsmPlan &whole) {
  if (split.max_entries <= whole.max_entries || whole.bits % whole.c <= whole.c / 2) return true;
  return split.max_entries - whole.max_entries <= whole.J * (4ull * (whole.K - split.K) + 3700000);
}

// G2 scalars are taken in quarters where these have no more entries at the width
// than halves have: they have half the buckets and half the doublings.  5003 points
// 757 us in halves (c = 13), 538 in quarters (c = 11), 2^18 points 1.88 (c = 16) and
// 1.78 ms (c = 13).  At other widths the top window of a quarter is a waste: c = 16,
// 5 windows of 4 against 8 of 2 per scalar, 5.9 against 5.0 ms at 2^20 points.
MsmPlan msm_split_plan(const MsmPlan &whole, const uint64_t *n, bool g2, uint32_t chunk, uint32_t reduce_seg) {
  MsmPlan split = msm_group_plan(whole.c, 2, n, whole.J, g2, chunk, reduce_seg);
  if (g2) {
    const MsmPlan quarter = msm_group_plan(whole.c, 4, n, whole.J, g2, chunk, reduce_seg);
    if (quarter.max_entries <= split.max_entries && msm_plan_ok(quarter)) split = quarter;
  }
  return msm_plan_ok(split) && split_pays(split, whole) ? split : whole;
}

bool msm_plan_ok(const MsmPlan &pl) {
  if (pl.c < 2 || pl.c > kMaxWindowBits || pl.J == 0) return false;
  if (pl.hb > 8 || pl.hb + 1 > pl.c || pl.c - 1 - pl.hb > 11) return false;
  if (pl.st > pl.c - 1 - pl.hb) return false;
  if (pl.Lr == 0 || (pl.Lr & (pl.Lr - 1)) != 0 || pl.B % pl.Lr) return false;
  if (pl.max_entries >= (1ull << 31)) return false;
  const uint32_t hi_bits = pl.hb;
  if ((uint64_t)pl.W * pl.tiles * (1u << hi_bits) >= (1ull << 32) - 1) return false;
  if ((uint64_t)pl.J * pl.K >= (1ull << 32) - 1) return false;
  if (pl.L == 0 || pl.L > (1u << 20)) return false;
  return true;
}

size_t msm_workspace_bytes(const MsmPlan &pl, bool g2) {
  // must mirror the carve order of msm_run (msm_impl.h)
  const uint32_t hi_bits = pl.hb;
  const uint64_t ncnt = (uint64_t)pl.W * (1u << hi_bits) * pl.tiles;
  const uint64_t nb = (ncnt + SCAN_TILE - 1) / SCAN_TILE;
  const uint64_t Ktot = (uint64_t)pl.J * pl.K, Wtot = (uint64_t)pl.J * pl.W;
  size_t b = 0;
  b += Carver::round((pl.max_entries + 4) * 4); // digits, then sorted (+ 4: quad loads)
  b += Carver::round(msm_sortbuf_bytes(pl, g2)); // pass-1 entries, then 29-bit points and slots
  b += Carver::round((ncnt + 1) * 4);           // tile counts -> offsets
  b += Carver::round(nb * 4);                   // scan block sums
  b += Carver::round((Ktot + 1) * 4);           // bucket offsets
  b += Carver::round(pl.max_chunks * 4);        // carry keys
  b += Carver::round(Wtot * (g2 ? 288 : 144));  // window sums (29-bit slots)
  return b + 4096;
}

void msm_fill_segs(const MsmPlan &pl, const uint64_t *n, const uint32_t *const *scalars,
                   const uint32_t *const *points, uint32_t *const *out, MsmSeg *segs) {
  const uint32_t hi_bits = pl.hb;
  const uint32_t HB = 1u << hi_bits;
  uint64_t pbase = 0, tiles = 0;
  for (uint32_t j = 0; j <= pl.J; j++) {
    MsmSeg &g = segs[j];
    g = MsmSeg{};
    g.pbase = pbase;
    g.tbase = (uint32_t)(pl.W * tiles);
    g.cbase = (uint32_t)(pl.W * HB * tiles);
    if (j == pl.J) break;
    g.scalars = scalars[j];
    g.points = points[j];
    g.out = out[j];
    g.n = pl.E * n[j];
    g.NT = (uint32_t)((g.n + kSortTile - 1) / kSortTile);
    g.qbase = (uint32_t)pbase;
    pbase += g.n;
    tiles += g.NT;
  }
}

MsmPlan msm_least_plan(const MsmPlan &whole, const MsmPlan &split, bool g2) {
  return msm_workspace_bytes(whole, g2) < msm_workspace_bytes(split, g2) ? whole : split;
}

// writes the descriptor table (members + sentinel) of a call on the stream
struct SegArgs {
  MsmSeg s[kMultiMembers + 1];
};
__global__ void k_put_segs(SegArgs a, uint32_t count, MsmSeg *dst) {
  if (threadIdx.x < count) dst[threadIdx.x] = a.s[threadIdx.x];
}
static void put_segs(const MsmPlan &pl, const MsmSeg *segs, MsmSeg *dst, hipStream_t st) {
  SegArgs a;
  for (uint32_t j = 0; j <= pl.J; j++) a.s[j] = segs[j];
  k_put_segs<<<1, 64, 0, st>>>(a, pl.J + 1, dst);
}

// a single call's whole-scalar plan and the settings it was made with
static MsmPlan single_plan(const csk_ctx *ctx, bool g2, uint64_t n, const csk_msm_cfg *cfg, uint32_t &chunk,
                           uint32_t &rseg) {
  const uint32_t lg = floor_log2(n);
  const csk_msm_cfg *tn = lg < 64 && !(cfg && cfg->window_bits) ? &ctx->tune[g2][lg] : nullptr;
  chunk = cfg && cfg->chunk ? cfg->chunk : tn ? tn->chunk : 0;
  rseg = cfg && cfg->reduce_seg ? cfg->reduce_seg : tn ? tn->reduce_seg : 0;
  return msm_group_plan(msm_choose_c(n, g2, ctx, cfg), 1, &n, 1, g2, chunk, rseg);
}

int msm_launch(csk_ctx *ctx, bool g2, const uint32_t *d_scalars, const uint32_t *d_points, uint64_t n,
               uint32_t *d_out, const csk_msm_cfg *cfg, hipStream_t st) {
  if (!d_out) {
    set_error("msm: null output");
    return CSK_ERR_ARG;
  }
  CSK_HIP(hipSetDevice(ctx->device));
  if (n == 0) {
    // empty sum: the point at infinity, (0, 1*R)
    uint32_t inf[32] = {0};
    for (int i = 0; i < 8; i++) inf[(g2 ? 16 : 8) + i] = FieldConst<0>::one[i];
    CSK_HIP(hipMemcpyAsync(d_out, inf, (g2 ? 32 : 16) * 4, hipMemcpyHostToDevice, st));
    CSK_HIP(hipStreamSynchronize(st));
    return CSK_OK;
  }
  if (!d_scalars || !d_points) {
    set_error("msm: null input");
    return CSK_ERR_ARG;
  }
  uint32_t chunk, rseg;
  MsmPlan pl = single_plan(ctx, g2, n, cfg, chunk, rseg);
  if (!msm_plan_ok(pl)) {
    set_error("msm: unsupported configuration (window/chunk/segment or size too large)");
    return CSK_ERR_ARG;
  }
  const size_t seg_bytes = Carver::round(2 * sizeof(MsmSeg));
  const MsmPlan split = msm_split_plan(pl, &n, g2, chunk, rseg), least = msm_least_plan(pl, split, g2);
  int rc = ctx->ws.ensure(seg_bytes + msm_workspace_bytes(split, g2));
  if (rc == CSK_ERR_NOMEM && least.E != split.E) {
    // the split points do not fit: whole scalars need one copy of them
    rc = ctx->ws.ensure(seg_bytes + msm_workspace_bytes(least, g2));
    if (rc == CSK_OK) set_error("");
    pl = least;
  } else {
    pl = split;
  }
  if (rc) return rc;
  StageTimer *tm = nullptr;
  if (ctx->timing) {
    ctx->timer.reset();
    tm = &ctx->timer;
  }
  ctx->last_plan = pl;
  MsmSeg segs[2];
  msm_fill_segs(pl, &n, &d_scalars, &d_points, &d_out, segs);
  MsmSeg *d_segs = (MsmSeg *)ctx->ws.ptr;
  put_segs(pl, segs, d_segs, st);
  CSK_CHECK_LAUNCH();
  void *ws = (char *)ctx->ws.ptr + seg_bytes;
  return g2 ? msm_run_g2(ws, pl, d_segs, st, tm) : msm_run_g1(ws, pl, d_segs, st, tm);
}

// One group of count <= kMultiMembers multiexps in the context's workspace, if its
// plan holds them and the workspace can be had; false: nothing was enqueued.
static bool multi_group(csk_ctx *ctx, bool g2, uint32_t c, uint32_t count, const uint64_t *n,
                        const uint32_t *const *scalars, const uint32_t *const *points, uint32_t *const *out,
                        hipStream_t st, int *rc) {
  MsmPlan pl = msm_group_plan(c, 1, n, count, g2, 0, 0);
  if (!msm_plan_ok(pl)) return false;
  pl = msm_split_plan(pl, n, g2, 0, 0);
  const size_t seg_bytes = Carver::round((count + 1) * sizeof(MsmSeg));
  if (ctx->ws.ensure(seg_bytes + msm_workspace_bytes(pl, g2)) != CSK_OK) {
    set_error("");  // the single calls may fit
    return false;
  }
  StageTimer *tm = nullptr;
  if (ctx->timing) {
    ctx->timer.reset();
    tm = &ctx->timer;
  }
  ctx->last_plan = pl;
  MsmSeg segs[kMultiMembers + 1];
  msm_fill_segs(pl, n, scalars, points, out, segs);
  MsmSeg *d_segs = (MsmSeg *)ctx->ws.ptr;
  put_segs(pl, segs, d_segs, st);
  void *ws = (char *)ctx->ws.ptr + seg_bytes;
  *rc = g2 ? msm_run_g2(ws, pl, d_segs, st, tm) : msm_run_g1(ws, pl, d_segs, st, tm);
  return true;
}

// Width of a group of `count` G1 multiexps of n points in all, which single calls would
// run at width c.  These weigh the buckets' reduction, which waits for chains of
// additions, against launches and chains that a group shares; its cost is the work,
// an addition per entry and about 2.8 per bucket, of 126 / c + 1 windows.  The four of
// a 50000-constraint proof are at 3 entries a bucket by 16 and 25 by 13: 923 -> 791 us;
// from 150000 points each 16 is the least again.
uint32_t multi_width(uint32_t c, uint32_t count, uint64_t n) {
  auto work = [&](uint32_t w) { return (kGlvBits / w + 1) * (20 * n + 14ull * count * (1u << w)); };
  uint32_t best = c;
  for (uint32_t w : {16u, 13u, 8u})
    if (w < c && work(w) < work(best)) best = w;
  return best;
}

// out = (0, 1*R), the affine point at infinity of the empty sum; words 16 (G1), 32 (G2)
__global__ void k_put_inf(uint32_t *out, uint32_t words) {
  const uint32_t i = threadIdx.x, y = words / 2;
  if (i < words) out[i] = i >= y && i < y + 8 ? FieldConst<0>::one[i - y] : 0u;
}

// The members a single call would give the same width run as one group: a stage is
// one launch over all of them, and their window combinations, a chain of 126
// doublings and an inversion that one workgroup each waits for, run side by side.
// Four of 1000 G1 points 1393 -> 357 us, of 50000 2101 -> 923, of 600000 5.17 -> 3.94
// ms, of 2 million 12.6 -> 11.7.  Larger ones gain less than the sum of their
// workspaces, which a group needs, is worth.
int msm_multi(csk_ctx *ctx, bool g2, uint32_t count, const uint32_t *const *scalars, const uint32_t *const *points,
              const uint64_t *n, uint32_t *const *out, hipStream_t st) {
  // what a single call would refuse is refused before anything is enqueued
  uint32_t chunk, rseg;
  for (uint32_t i = 0; i < count; i++) {
    if (!out[i] || (n[i] && (!scalars[i] || !points[i]))) {
      set_error("msm_multi: null pointer for member " + std::to_string(i));
      return CSK_ERR_ARG;
    }
    if (n[i] && !msm_plan_ok(single_plan(ctx, g2, n[i], nullptr, chunk, rseg))) {
      set_error("msm_multi: member " + std::to_string(i) + " too large");
      return CSK_ERR_ARG;
    }
  }
  CSK_HIP(hipSetDevice(ctx->device));
  uint64_t done = 0;  // members enqueued, a bit each
  for (uint32_t i = 0; i < count; i++) {
    if (done >> i & 1) continue;
    if (n[i] == 0) {
      k_put_inf<<<1, 64, 0, st>>>(out[i], g2 ? 32 : 16);
      CSK_CHECK_LAUNCH();
      continue;
    }
    const uint32_t c = msm_choose_c(n[i], g2, ctx, nullptr);
    uint32_t idx[kMultiMembers], k = 0;
    uint64_t gn[kMultiMembers], total = 0;
    const uint32_t *gs[kMultiMembers], *gp[kMultiMembers];
    uint32_t *go[kMultiMembers];
    for (uint32_t j = i; j < count && k < kMultiMembers; j++) {
      if ((done >> j & 1) || n[j] == 0) continue;
      if (n[j] > kMultiPoints || total + n[j] > kMultiPoints || msm_choose_c(n[j], g2, ctx, nullptr) != c) continue;
      total += n[j];
      idx[k] = j;
      gn[k] = n[j];
      gs[k] = scalars[j];
      gp[k] = points[j];
      go[k++] = out[j];
    }
    int rc = CSK_OK;
    if (k > 1 && idx[0] == i && multi_group(ctx, g2, g2 ? c : multi_width(c, k, total), k, gn, gs, gp, go, st, &rc)) {
      for (uint32_t j = 0; j < k; j++) done |= 1ull << idx[j];
    } else {
      done |= 1ull << i;
      rc = msm_launch(ctx, g2, scalars[i], points[i], n[i], out[i], nullptr, st);
    }
    if (rc) return rc;
  }
  return CSK_OK;
}

// ------------------------------------------------- multiexp without allocation
// csk_msm_g1_noalloc runs the same pipeline as csk_msm_g1 in a fixed device
// array instead of the context's growable workspace.  Every GPU that loads
// the library holds one copy of it (kNoAllocBytes) until the process ends;
// host code reaches it only through the address hipGetSymbolAddress gives
// for the current device, looked up once per device at context creation (or
// on the entry point's first call on that device).
static constexpr size_t kNoAllocBytes = 48ull << 20;
static constexpr uint64_t kNoAllocMaxPoints = 1ull << 15;
static constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices] = {};

// with `device` current: look up this device's copy of the array
int msm_noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices) {
    set_error("msm_noalloc: device index beyond the supported 64");
    return CSK_ERR_ARG;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[device]) return CSK_OK;
  void *p = nullptr;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    set_error(std::string("msm_noalloc: hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    return CSK_ERR_HIP;
  }
  g_scratch_ptr[device] = p;
  return CSK_OK;
}

// The bytes that decide which widths the array takes: the workspace of the
// whole-scalar plan, its digits and a slot per reduction segment.  The pipeline
// that runs needs no more, so a width is accepted or refused by n and cfg alone.
static size_t noalloc_bytes(const MsmPlan &pl, uint32_t rseg) {
  const uint32_t seg = rseg && rseg < pl.Lr ? rseg : pl.Lr;
  return msm_workspace_bytes(pl, false) + Carver::round(pl.max_entries * 4) +
         Carver::round((uint64_t)pl.J * pl.W * (pl.B / seg) * 144);
}

}  // namespace csk

using namespace csk;

extern "C" int csk_msm_g1_noalloc(csk_ctx *ctx, const uint32_t *d_scalars, const uint32_t *d_points, uint64_t n,
                                  uint32_t *d_out, const csk_msm_cfg *cfg, void *stream) {
  if (!ctx || !d_out) {
    set_error("msm_g1_noalloc: null context or output");
    return CSK_ERR_ARG;
  }
  if (n > kNoAllocMaxPoints) {
    set_error("msm_g1_noalloc: n = " + std::to_string(n) + " exceeds the no-allocation limit of " +
              std::to_string(kNoAllocMaxPoints) + " points; use csk_msm_g1");
    return CSK_ERR_ARG;
  }
  if (n && (!d_scalars || !d_points)) {
    set_error("msm_g1_noalloc: null input");
    return CSK_ERR_ARG;
  }
  CSK_HIP(hipSetDevice(ctx->device));
  int rc = msm_noalloc_setup(ctx->device);
  if (rc) return rc;
  char *base = (char *)g_scratch_ptr[ctx->device];
  hipStream_t st = (hipStream_t)stream;
  if (n == 0) {
    k_put_inf<<<1, 64, 0, st>>>(d_out, 16);
    CSK_CHECK_LAUNCH();
    return CSK_OK;
  }
  // the tuned window width, narrowed until the workspace fits the array
  // (every width gives the same sum); an explicit width that does not fit is an error
  const bool fixed_c = cfg && cfg->window_bits;
  uint32_t c = msm_choose_c(n, false, ctx, cfg);
  const uint32_t lg = floor_log2(n);
  const csk_msm_cfg *tn = &ctx->tune[0][lg];
  const uint32_t chunk = cfg && cfg->chunk ? cfg->chunk : (!fixed_c ? tn->chunk : 0);
  const uint32_t rseg = cfg && cfg->reduce_seg ? cfg->reduce_seg : (!fixed_c ? tn->reduce_seg : 0);
  const size_t seg_bytes = Carver::round(2 * sizeof(MsmSeg));
  MsmPlan pl = msm_group_plan(c, 1, &n, 1, false, chunk, rseg);
  while (!fixed_c && c > 2 && (!msm_plan_ok(pl) || seg_bytes + noalloc_bytes(pl, rseg) > kNoAllocBytes)) {
    c--;
    pl = msm_group_plan(c, 1, &n, 1, false, chunk, rseg);
  }
  if (!msm_plan_ok(pl)) {
    set_error("msm_g1_noalloc: unsupported configuration (window/chunk/segment)");
    return CSK_ERR_ARG;
  }
  if (seg_bytes + noalloc_bytes(pl, rseg) > kNoAllocBytes) {
    set_error("msm_g1_noalloc: the workspace for window width " + std::to_string(pl.c) + " needs " +
              std::to_string(seg_bytes + noalloc_bytes(pl, rseg)) + " bytes, more than the " +
              std::to_string(kNoAllocBytes) + "-byte scratch array");
    return CSK_ERR_ARG;
  }
  // which widths are taken is settled by the whole scalars' workspace; the
  // split ones run where theirs fits too
  const MsmPlan split = msm_split_plan(pl, &n, false, chunk, rseg);
  if (seg_bytes + msm_workspace_bytes(split, false) <= kNoAllocBytes) pl = split;
  ctx->last_plan = pl;
  MsmSeg segs[2];
  msm_fill_segs(pl, &n, &d_scalars, &d_points, &d_out, segs);
  MsmSeg *d_segs = (MsmSeg *)base;
  put_segs(pl, segs, d_segs, st);
  CSK_CHECK_LAUNCH();
  return msm_run_g1(base + seg_bytes, pl, d_segs, st, nullptr);
}

// ------------------------------------------------------------ fixed-base tables
// csk_msm_table_*: the table multiexp of msm_impl.h (window-shifted copies of
// fixed points, one bucket reduction, no doublings between windows).
struct csk_msm_table {
  csk_ctx *ctx = nullptr;
  int ec2 = 0;
  uint64_t n = 0, n_pad = 0;
  uint32_t c = 0, Wt = 0;
  uint32_t *table = nullptr;  // Wt * n_pad points in the 2^261 form
  uint32_t *live = nullptr;   // one bit per point: not at infinity
  uint32_t Lrm = 0;
  uint64_t table_bytes = 0;
};

namespace csk {

// group plan of the runs over tables of n_pad[0..count) points: count members of
// Wt * n_pad points, or count * Wt one-window members
static MsmPlan table_plan(bool g2, uint32_t c, const uint64_t *n_pad, uint32_t count, uint32_t Wt) {
  MsmPlan pl = {};
  uint64_t most = 0;
  for (uint32_t p = 0; p < count; p++) {
    pl.n += n_pad[p] * Wt;
    if (n_pad[p] > most) most = n_pad[p];
  }
  const bool joint = table_joint(most, c, Wt, g2);
  pl.c = c;
  pl.E = 1;
  pl.bits = kScalarBits;
  pl.W = 1;
  pl.B = 1u << (c - 1);
  pl.K = pl.B;
  pl.J = joint ? count : Wt * count;
  pl.most = joint ? most * Wt : most;
  pl.tiles = pl.n / kSortTile;
  pl.max_entries = pl.n;
  pl.hb = plan_hi_bits(c, pl.n / pl.J);
  pl.st = plan_top_bits(pl.bits, c, pl.hb);
  pl.Lr = pl.B < 16 ? pl.B : 16;
  pl.S = pl.B / pl.Lr;
  plan_chunks(pl, 0);
  return pl;
}

static uint64_t table_point_bytes(int ec2, uint64_t n_pad, uint32_t Wt) {
  return (uint64_t)Wt * n_pad * (ec2 ? 128 : 64) + n_pad / 8;
}

// A table run reduces one set of 2^(c-1) buckets whatever Wt is, so it
// affords wider windows than the plain multiexp: 16 from 2^15 points, 17
// from 2^18 and 20 (13 windows instead of 15) from 3 * 2^22 G1 and 2^24 G2
// points (measured on G1 and G2 at 2^16 .. 2^25: G1 2^24 20.8 against 21.6 ms
// at c = 17, 2^25 38.9 against 41.7, G2 2^24 54.4 against 55.5; G1 2^23 ties,
// G2 2^23 33.4 against 30.5), the plain width below.  A width whose top
// window keeps few scalar bits (t = 254 mod c: 2 at c = 14 and 18) puts that
// window's every entry into 2^t buckets, whose long carry chains cost more
// than the window it saves (2^14 points: 1.09 ms at c = 14, 0.76 ms at 15):
// 14 becomes 15.
static uint32_t table_default_c(uint64_t n, int ec2, const csk_ctx *ctx) {
  const uint32_t lg = floor_log2(n);
  if (n >= (ec2 ? 1ull << 24 : 3ull << 22)) return 20;
  if (lg >= 18) return 17;
  if (lg >= 15) return 16;
  uint32_t c = msm_choose_c(n, ec2 != 0, ctx, nullptr);
  if (c > 16) c = 16;
  if (c == 14) c = 15;
  return c;
}

// count runs in one pipeline, run p over table t[p] (same curve and window
// width), in the workspace of ctx, on stream st
static int table_run(csk_ctx *ctx, uint32_t count, csk_msm_table *const *t, const uint32_t *const *d_scalars,
                     uint32_t *const *d_out, hipStream_t st) {
  const csk_msm_table *t0 = t[0];
  const uint32_t Wt = t0->Wt, c = t0->c;
  uint32_t max_nt = 0;
  uint64_t pads[kTabBatch];
  for (uint32_t p = 0; p < count; p++) {
    if (t[p]->ec2 != t0->ec2 || t[p]->c != c || t[p]->ctx->device != ctx->device) {
      set_error("msm_table_run: the tables of one run must share curve, window width and device");
      return CSK_ERR_ARG;
    }
    pads[p] = t[p]->n_pad;
    const uint32_t nt = (uint32_t)(t[p]->n_pad / kSortTile);
    if (nt > max_nt) max_nt = nt;
  }
  const MsmPlan pl = table_plan(t0->ec2 != 0, c, pads, count, Wt);
  if (!msm_plan_ok(pl)) {
    set_error("msm_table_run: " + std::to_string(count) + " runs of up to " + std::to_string(max_nt * kSortTile) +
              " points exceed the multiexp's index range");
    return CSK_ERR_ARG;
  }
  CSK_HIP(hipSetDevice(ctx->device));
  const uint64_t PW = t0->ec2 ? 32 : 16;
  const uint32_t per = pl.J / count;  // members of a run
  std::vector<uint64_t> ns(pl.J);
  std::vector<const uint32_t *> sc(pl.J, nullptr), pts(pl.J);
  std::vector<uint32_t *> outs(pl.J, nullptr);
  for (uint32_t m = 0; m < pl.J; m++) {
    const csk_msm_table *tp = t[m / per];
    ns[m] = tp->n_pad * (Wt / per);
    pts[m] = tp->table + (uint64_t)(m % per) * tp->n_pad * PW;
  }
  std::vector<MsmSeg> segs(pl.J + 1);
  msm_fill_segs(pl, ns.data(), sc.data(), pts.data(), outs.data(), segs.data());
  int rc = ctx->ws.ensure(msm_table_ws_bytes(pl, t0->ec2 != 0, count));
  if (rc) return rc;
  TabArgs args = {};
  for (uint32_t p = 0; p < count; p++) {
    args.s[p] = d_scalars[p];
    args.o[p] = d_out[p];
    args.live[p] = t[p]->live;
    args.n[p] = t[p]->n;
  }
  return t0->ec2 ? msm_run_table_g2(ctx->ws.ptr, pl, segs.data(), args, count, Wt, max_nt, t0->Lrm, st)
                 : msm_run_table_g1(ctx->ws.ptr, pl, segs.data(), args, count, Wt, max_nt, t0->Lrm, st);
}

}  // namespace csk

extern "C" int csk_msm_table_bytes(int ec2, uint64_t n, uint32_t window_bits, uint64_t *bytes) {
  if (!bytes || n == 0 || window_bits < 2 || window_bits > kMaxWindowBits) {
    set_error("msm_table_bytes: n >= 1 and 2 <= window_bits <= 20 required");
    return CSK_ERR_ARG;
  }
  const uint64_t n_pad = (n + kSortTile - 1) / kSortTile * kSortTile;
  *bytes = table_point_bytes(ec2, n_pad, 254 / window_bits + 1);
  return CSK_OK;
}

extern "C" int csk_msm_table_create(csk_ctx *ctx, int ec2, const uint32_t *d_points, uint64_t n, uint32_t window_bits,
                                    csk_msm_table **out, void *stream) {
  if (!ctx || !out || !d_points || n == 0) {
    set_error("msm_table_create: null argument or n == 0");
    return CSK_ERR_ARG;
  }
  *out = nullptr;
  const uint32_t c = window_bits ? window_bits : table_default_c(n, ec2, ctx);
  if (c < 2 || c > kMaxWindowBits) {
    set_error("msm_table_create: window_bits must be 2..20");
    return CSK_ERR_ARG;
  }
  const uint32_t Wt = 254 / c + 1;
  const uint64_t n_pad = (n + kSortTile - 1) / kSortTile * kSortTile;
  MsmPlan pl = table_plan(ec2 != 0, c, &n_pad, 1, Wt);
  if (!msm_plan_ok(pl)) {
    set_error("msm_table_create: " + std::to_string(n) + " points x " + std::to_string(Wt) +
              " windows exceed the multiexp's index range");
    return CSK_ERR_ARG;
  }
  CSK_HIP(hipSetDevice(ctx->device));
  hipStream_t st = (hipStream_t)stream;
  csk_msm_table *t = new csk_msm_table();
  t->ctx = ctx;
  t->ec2 = ec2 ? 1 : 0;
  t->n = n;
  t->n_pad = n_pad;
  t->c = c;
  t->Wt = Wt;
  uint32_t lr = 16;
  while (lr > 2 && pl.B / lr < (1u << 15)) lr >>= 1;
  if (lr > pl.B) lr = pl.B;
  t->Lrm = lr;
  const uint64_t PW = ec2 ? 32 : 16;
  t->table_bytes = table_point_bytes(t->ec2, n_pad, Wt);
  hipError_t e = hipMalloc(&t->table, (size_t)Wt * n_pad * PW * 4);
  if (e == hipSuccess) e = hipMalloc(&t->live, (size_t)(n_pad / 32) * 4);
  if (e != hipSuccess) {
    set_error(std::string("msm_table_create: allocation: ") + hipGetErrorString(e));
    csk_msm_table_destroy(t);
    return CSK_ERR_NOMEM;
  }
  int rc = t->ec2 ? msm_table_build_g2(d_points, n, n_pad, c, Wt, t->table, t->live, st)
                  : msm_table_build_g1(d_points, n, n_pad, c, Wt, t->table, t->live, st);
  if (rc == CSK_OK) {
    e = hipStreamSynchronize(st);
    if (e != hipSuccess) {
      set_error(std::string("msm_table_create: ") + hipGetErrorString(e));
      rc = CSK_ERR_HIP;
    }
  }
  if (rc) {
    csk_msm_table_destroy(t);
    return rc;
  }
  *out = t;
  return CSK_OK;
}

extern "C" int csk_msm_table_run(csk_msm_table *t, const uint32_t *d_scalars, uint32_t *d_out, void *stream) {
  if (!t || !d_scalars || !d_out) {
    set_error("msm_table_run: null argument");
    return CSK_ERR_ARG;
  }
  return table_run(t->ctx, 1, &t, &d_scalars, &d_out, (hipStream_t)stream);
}

extern "C" int csk_msm_table_run_batch(csk_ctx *ctx, csk_msm_table *t, uint32_t count,
                                       const uint32_t *const *d_scalars, uint32_t *const *d_out, void *stream) {
  if (!t || (count && (!d_scalars || !d_out)) || count > kTabBatch) {
    set_error("msm_table_run_batch: null argument or more than 64 scalar vectors");
    return CSK_ERR_ARG;
  }
  if (!ctx) ctx = t->ctx;
  if (ctx->device != t->ctx->device) {
    set_error("msm_table_run_batch: the context's device is not the table's");
    return CSK_ERR_ARG;
  }
  for (uint32_t p = 0; p < count; p++)
    if (!d_scalars[p] || !d_out[p]) {
      set_error("msm_table_run_batch: null buffer for scalar vector " + std::to_string(p));
      return CSK_ERR_ARG;
    }
  if (count == 0) return CSK_OK;
  std::vector<csk_msm_table *> ts(count, t);
  return table_run(ctx, count, ts.data(), d_scalars, d_out, (hipStream_t)stream);
}

extern "C" int csk_msm_table_run_multi(csk_ctx *ctx, uint32_t count, csk_msm_table *const *tables,
                                       const uint32_t *const *d_scalars, uint32_t *const *d_out, void *stream) {
  if (!ctx || (count && (!tables || !d_scalars || !d_out)) || count > kTabBatch) {
    set_error("msm_table_run_multi: null argument or more than 64 runs");
    return CSK_ERR_ARG;
  }
  for (uint32_t p = 0; p < count; p++)
    if (!tables[p] || !d_scalars[p] || !d_out[p]) {
      set_error("msm_table_run_multi: null table or buffer for run " + std::to_string(p));
      return CSK_ERR_ARG;
    }
  if (count == 0) return CSK_OK;
  return table_run(ctx, count, tables, d_scalars, d_out, (hipStream_t)stream);
}

extern "C" int csk_msm_table_info(const csk_msm_table *t, uint64_t *out, int n) {
  if (!t || !out || n < 1) return CSK_ERR_ARG;
  const MsmPlan pl = table_plan(t->ec2 != 0, t->c, &t->n_pad, 1, t->Wt);
  const uint64_t v[5] = {t->n, t->c, t->Wt, t->table_bytes, msm_table_ws_bytes(pl, t->ec2 != 0, 1)};
  for (int i = 0; i < n && i < 5; i++) out[i] = v[i];
  return CSK_OK;
}

extern "C" void csk_msm_table_destroy(csk_msm_table *t) {
  if (!t) return;
  if (t->ctx) (void)hipSetDevice(t->ctx->device);
  if (t->table || t->live) (void)hipDeviceSynchronize();
  if (t->table) (void)hipFree(t->table);
  if (t->live) (void)hipFree(t->live);
  delete t;
}
