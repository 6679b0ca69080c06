// Index maps, per-thread operand loaders and launch plan of the implicit-GEMM
// convolutions (k_conv_gemm.hip). Host + device code, so that the exact loaders the
// kernel runs can also be exercised on the CPU.
//
// GEMM view, per group g (images are folded into the spatial dimension):
//   conv2d             Y[co][(b,p)]  = sum_{k=(cl,kh,kw)}  W[co][k] * x[b, cl, ho*sH+kh-pH, wo*sW+kw-pW]
//   conv2d_input_grad  dX[cl][(b,q)] = sum_{k=(col,kh,kw)} W[col][cl][kh,kw] * dy[b, col, ho, wo],
//                                      (ho, wo) with ho*sH+kh-pH = hi, wo*sW+kw-pW = wi
//   conv2d_weight_grad dW[co][n=(cl,kh,kw)] = sum_{k=(b,p)} dy[b, co, p] * x[b, cl, ho*sH+kh-pH, wo*sW+kw-pW]
// with p = (ho, wo), q = (hi, wi). Out-of-image taps read as zero.
//
// The gathers are separable: an operand element's offset is a term of its row (an output position, a weight row) plus a
// term of its reduction index, and whether a tap falls outside the image is a bit of the position's row mask or column
// mask, picked by the tap. Row terms are found once per block. The reduction index' terms (KTerm) are found once per
// block and stage and read from LDS by all, so an element costs one add and, where taps can fall outside, three more
// operations. Offsets are bytes modulo 2^32: every tensor has fewer than 2^29 elements, row terms are not
// negative, so a valid sum is exact and an element that reads as zero gets bit 31 set, which the buffer unit returns 0 for.
//
// The input gradient of a strided convolution is one stride-1 problem per phase (hi mod sH, wi mod sW): the positions
// of a phase meet the same taps, kh = kh0 + j * sH, and ho = hi' + dh - j, so no products with zeros are made. Its
// reduction runs tap by tap, k = tap * CoutPG + col.
#pragma once
#include <algorithm>
#include <cstdint>

#include "kernels.h"

namespace tgk {
namespace cg {

using gd::f32x4;

#define CG_HD __host__ __device__ __forceinline__

constexpr int kCT = 256;    // threads per block
constexpr int kCBK = 16;    // k per LDS stage

enum { CV_FWD = 0, CV_DGRAD = 1, CV_WGRAD = 2 };
// Loader variants, chosen per launch (template flags, so the k loop has no runtime tests):
// F_AVEC: 4 consecutive k of A are consecutive in memory (one 16-byte load). F_PAD: some tap falls outside the image.
// F_WIDE: a kernel of more than 32 rows or columns, whose taps do not fit the masks: coordinates are compared. F_TAP: a
// thread's consecutive k share a tap (the input gradient over a multiple of 8 channels): one test for all.
// F_BVEC: the weight gradient's 4 consecutive k of B are consecutive in memory (stride 1, no padding, Wo % 4 == 0).
enum { F_AVEC = 1, F_PAD = 2, F_WIDE = 4, F_TAP = 8, F_BVEC = 16 };

struct ConvGemmArgs {
  int B, Cin, H, W, Cout, CinPG, CoutPG, kH, kW, Ho, Wo, G, sH, sW, pH, pW;
  int M, N, K;                  // GEMM sizes per group
  int tiles_m, tiles_n, splits, k_per_split;
  int pad;                      // some tap can fall outside the image: bounds checks needed
  int phases;                   // input gradient: min(sH, H) * min(sW, W)
  int ipb;                      // few-taps weight gradient: images per block
  FastDiv dKHW, dKW, dWo, dHoWo;
  FastDiv dCpg;                 // CoutPG
  FastDiv dTn, dPh, dPhW;       // tiles_n; the input gradient's phases, and those of a row
  const float* x;
  const float* w;
  const float* dy;
  float* out;                   // y / dx / dw
  float* work;                  // weight-gradient partials [split][G][M][N] (splits > 1)
  // A pointwise group applied at the store: kConvEpiBiasRelu on the forward's
  // output channel ch, kConvEpiReluMask on the input gradient's element.
  int epi;
  const float* ebias;           // [Cout]
  const float* emask;           // laid out as the output
};

// kConvEpiBiasRelu: relu(v + bias[ch]) as the fused group computes it (f32 add; relu keeps
// NaN as the canonical NaN and maps -0 to +0). kConvEpiReluMask: relu_grad(mask, v) =
// mask > 0 ? v : +0, the mask at the output element's offset.
constexpr int kConvEpiNone = 0, kConvEpiBiasRelu = 1, kConvEpiReluMask = 2;

// x / d for 0 <= x < 2^31 (FastDiv, kernels.h), on the host or the device.
CG_HD int fdiv(int x, const FastDiv& f) {
  return (int)((((uint32_t)(((uint64_t)(uint32_t)x * f.m) >> 32)) + (uint32_t)x) >> f.s);
}

CG_HD bool inside(int a, int lim) { return (uint32_t)a < (uint32_t)lim; }

// An operand tensor read through the buffer unit (raw buffer loads: 32-bit byte offsets
// from a uniform base, and offsets at or past the tensor's size read as 0 without a
// memory access). Elements that read as zero are loaded from an offset with bit 31 set, past
// every tensor (fewer than 2^29 elements each), so the loads need no branches. The host build (used to exercise the loaders on the CPU) reads the
// array directly with the same rule.
constexpr uint32_t kMasked = 0x80000000u;
struct Src {
#if defined(__HIP_DEVICE_COMPILE__)
  __amdgpu_buffer_rsrc_t r;
#else
  const float* p;
  uint32_t bytes;
#endif
};
CG_HD Src make_src(const float* p, int64_t elems) {
  Src s;
#if defined(__HIP_DEVICE_COMPILE__)
  // word 3 = 0x00020000: 32-bit data format, the setting for untyped loads on gfx9 parts
  s.r = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)(elems * 4), 0x00020000);
#else
  s.p = p;
  s.bytes = (uint32_t)(elems * 4);
#endif
  return s;
}
CG_HD float ldb(const Src& s, uint32_t off) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(s.r, (int)off, 0, 0));
#else
  return off < s.bytes ? s.p[off >> 2] : 0.0f;
#endif
}
CG_HD uint32_t boff(bool ok, uint32_t idx) { return ok ? idx << 2 : kMasked; }
CG_HD f32x4 ldb4(const Src& s, uint32_t off) {   // off 4-byte aligned; all four elements inside or off >= kMasked
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(s.r, (int)off, 0, 0));
#else
  f32x4 v;
  for (int u = 0; u < 4; ++u) v[u] = off + 4 * u < s.bytes ? s.p[(off >> 2) + u] : 0.0f;
  return v;
#endif
}

// Bits [lo, hi) of the taps 0 .. n-1 at coordinates first + t (step > 0) or first - t (step < 0) that lie inside
// 0 .. lim-1 are clear, the others set (n <= 32).
CG_HD uint32_t outside_bits(int first, int step, int n, int lim) {
  const int lo = std::max(0, step > 0 ? -first : first - lim + 1);
  const int hi = std::min(n, step > 0 ? lim - first : first + 1);
  return hi <= lo ? ~0u : ~((~0u >> (32 - (hi - lo))) << lo);
}

// The term of reduction index k: byte offsets into A and B, and the two numbers that the in-image test takes from the
// reduction side. conv2d and the input gradient: shifts 31 - tap row / column, which bring the row term's mask bits to
// bit 31 (F_WIDE: the tap's row / column shift). Weight gradient: the position's masks (F_WIDE: its coordinates).
struct KTerm { uint32_t a, b, t0, t1; };
// The term of a row of B (conv2d, input gradient: an output position; weight gradient: a tap of a channel).
struct BTerm { uint32_t off, t0, t1; };

// One output tile's place and the maps of one launch's operands.
template <int MODE, int F>
struct ConvMap {
  int m0, n0, z, split, kbeg, kend;   // tile origin, group, k range
  int N;                              // columns (input gradient: of the phase)
  // input gradient's phase: first position, position grid, first tap, taps, output row of (hi' = 0, tap 0)
  int rh, rw, Hr, Wr, kh0, kw0, nh, nw, dh, dw;
  int rnw;                            // 65536 / nw, rounded up
  Src sa, sb;

  template <int BM, int BN>
  CG_HD void init(const ConvGemmArgs& c, uint32_t blk, uint32_t nblk) {
    // Tiles are numbered so each XCD (the chip's 8 L2 domains take blocks round robin) receives a contiguous run, n
    // fastest (input gradient: phase fastest, so that a run holds as many blocks of each).
    uint32_t bid = blk;
    if (nblk % gd::kXcds == 0) bid = (bid % gd::kXcds) * (nblk / gd::kXcds) + bid / gd::kXcds;
    const int rest = fdiv((int)bid, c.dTn);
    int tn = (int)bid - rest * c.tiles_n;
    const int tm = rest % c.tiles_m, zs = rest / c.tiles_m;
    m0 = tm * BM;
    z = MODE == CV_WGRAD ? zs / c.splits : zs;
    split = MODE == CV_WGRAD ? zs % c.splits : 0;
    kbeg = split * c.k_per_split;
    kend = std::min(c.K, kbeg + c.k_per_split);
    N = c.N;
    if (MODE == CV_DGRAD) {
      const int t = fdiv(tn, c.dPh), ph = tn - t * c.phases;
      tn = t;
      rh = fdiv(ph, c.dPhW);
      rw = ph - rh * (int)c.dPhW.d;
      Hr = (c.H - rh + c.sH - 1) / c.sH;
      Wr = (c.W - rw + c.sW - 1) / c.sW;
      kh0 = (rh + c.pH) % c.sH;
      kw0 = (rw + c.pW) % c.sW;
      nh = (c.kH - kh0 + c.sH - 1) / c.sH;   // (kh0 < sH: not negative)
      nw = (c.kW - kw0 + c.sW - 1) / c.sW;
      rnw = 65536 / std::max(nw, 1) + 1;
      dh = (rh + c.pH - kh0) / c.sH;
      dw = (rw + c.pW - kw0) / c.sW;
      N = c.B * Hr * Wr;
      kend = nh * nw * c.CoutPG;
    }
    n0 = tn * BN;
    const int64_t xs = (int64_t)c.B * c.Cin * c.H * c.W, ws = (int64_t)c.Cout * c.CinPG * c.kH * c.kW,
                  ys = (int64_t)c.B * c.Cout * c.Ho * c.Wo;
    if (MODE == CV_FWD) { sa = make_src(c.w, ws); sb = make_src(c.x, xs); }
    else if (MODE == CV_DGRAD) { sa = make_src(c.w, ws); sb = make_src(c.dy, ys); }
    else { sa = make_src(c.dy, ys); sb = make_src(c.x, xs); }
  }

  // Position of column n: image, row, column of the output (input gradient: in the phase's grid).
  CG_HD void position(const ConvGemmArgs& c, int n, int& b, int& i, int& j) const {
    if (MODE == CV_DGRAD) {
      const int hw = Hr * Wr;
      b = n / hw;
      const int q = n - b * hw;
      i = q / Wr;
      j = q - i * Wr;
    } else {
      b = fdiv(n, c.dHoWo);
      const int q = n - b * c.Ho * c.Wo;
      i = fdiv(q, c.dWo);
      j = q - i * c.Wo;
    }
  }

  // Byte offset term of row m of A (past the last row: the last).
  CG_HD uint32_t a_row(const ConvGemmArgs& c, int m) const {
    const int mm = std::min(m, c.M - 1);
    if (MODE == CV_FWD) return (uint32_t)((z * c.CoutPG + mm) * c.K) << 2;
    if (MODE == CV_DGRAD) return (uint32_t)((z * c.CoutPG * c.CinPG + mm) * c.kH * c.kW) << 2;
    return (uint32_t)((z * c.CoutPG + mm) * c.Ho * c.Wo) << 2;
  }

  // The term of row n of B (past the last: the last; its products are not stored).
  CG_HD BTerm b_row(const ConvGemmArgs& c, int n) const {
    BTerm t;
    const int nn = std::min(n, N - 1);
    if (MODE == CV_WGRAD) {
      const int cl = fdiv(nn, c.dKHW), r = nn - cl * c.kH * c.kW;
      const int kh = fdiv(r, c.dKW), kw = r - kh * c.kW;
      t.off = (uint32_t)(((z * c.CinPG + cl) * c.H + kh) * c.W + kw) << 2;
      t.t0 = (F & F_WIDE) ? kh : 31 - kh;
      t.t1 = (F & F_WIDE) ? kw : 31 - kw;
      return t;
    }
    int b, i, j;
    position(c, nn, b, i, j);
    if (MODE == CV_FWD) {
      t.off = (uint32_t)(((b * c.Cin + z * c.CinPG) * c.H + i * c.sH) * c.W + j * c.sW) << 2;
      t.t0 = (F & F_WIDE) ? i * c.sH - c.pH : outside_bits(i * c.sH - c.pH, 1, c.kH, c.H);
      t.t1 = (F & F_WIDE) ? j * c.sW - c.pW : outside_bits(j * c.sW - c.pW, 1, c.kW, c.W);
    } else {
      t.off = (uint32_t)(((b * c.Cout + z * c.CoutPG) * c.Ho + i + dh) * c.Wo + j + dw) << 2;
      t.t0 = (F & F_WIDE) ? i + dh : outside_bits(i + dh, -1, nh, c.Ho);
      t.t1 = (F & F_WIDE) ? j + dw : outside_bits(j + dw, -1, nw, c.Wo);
    }
    return t;
  }

  CG_HD KTerm k_term(const ConvGemmArgs& c, int k) const {
    KTerm t;
    if (k >= kend) {   // both operands read as zero
      t.a = t.b = kMasked;
      t.t0 = t.t1 = 0;
      return t;
    }
    if (MODE == CV_FWD) {
      const int cl = fdiv(k, c.dKHW), r = k - cl * c.kH * c.kW;
      const int kh = fdiv(r, c.dKW), kw = r - kh * c.kW;
      t.a = (uint32_t)k << 2;
      t.b = (uint32_t)((cl * c.H + kh - c.pH) * c.W + kw - c.pW) << 2;
      t.t0 = (F & F_WIDE) ? kh : 31 - kh;
      t.t1 = (F & F_WIDE) ? kw : 31 - kw;
    } else if (MODE == CV_DGRAD) {
      const int tap = fdiv(k, c.dCpg), col = k - tap * c.CoutPG;
      // (fewer than 1024 taps, nw <= 32: rnw * nw - 65536 < 32, so the quotient is exact)
      const int jh = (F & F_WIDE) ? tap / nw : (int)((uint32_t)(tap * rnw) >> 16), jw = tap - jh * nw;
      t.a = (uint32_t)((col * c.CinPG * c.kH + kh0 + jh * c.sH) * c.kW + kw0 + jw * c.sW) << 2;
      t.b = (uint32_t)((col * c.Ho - jh) * c.Wo - jw) << 2;
      t.t0 = (F & F_WIDE) ? -jh : 31 - jh;
      t.t1 = (F & F_WIDE) ? -jw : 31 - jw;
    } else {
      const int b = fdiv(k, c.dHoWo), p = k - b * c.Ho * c.Wo;
      const int ho = fdiv(p, c.dWo), wo = p - ho * c.Wo;
      const int h = ho * c.sH - c.pH, w = wo * c.sW - c.pW;
      t.a = (uint32_t)(b * c.Cout * c.Ho * c.Wo + p) << 2;
      t.b = (uint32_t)((b * c.Cin * c.H + h) * c.W + w) << 2;
      t.t0 = (F & F_WIDE) ? h : outside_bits(h, 1, c.kH, c.H);
      t.t1 = (F & F_WIDE) ? w : outside_bits(w, 1, c.kW, c.W);
    }
    return t;
  }

  // Bit 31: the element of B at (row, k) lies outside the image.
  CG_HD uint32_t outside(const ConvGemmArgs& c, uint32_t r0, uint32_t r1, uint32_t k0, uint32_t k1) const {
    if (MODE != CV_DGRAD && !(F & F_PAD)) return 0;
    if (F & F_WIDE) {
      const int lh = MODE == CV_DGRAD ? c.Ho : c.H, lw = MODE == CV_DGRAD ? c.Wo : c.W;
      return inside((int)(r0 + k0), lh) && inside((int)(r1 + k1), lw) ? 0u : kMasked;
    }
    if (MODE == CV_WGRAD) return ((k0 << (r0 & 31)) | (k1 << (r1 & 31))) & kMasked;
    return ((r0 << (k0 & 31)) | (r1 << (k1 & 31))) & kMasked;
  }

  // Output offset of GEMM element (0, n) and the stride between rows m (for split weight gradients, the offset inside
  // the split's partial tile array).
  CG_HD int64_t out_col(const ConvGemmArgs& c, int n) const {
    if (MODE == CV_WGRAD) return ((int64_t)(c.splits > 1 ? split * c.G : 0) + z) * c.M * c.N + n;
    int b, i, j;
    position(c, n, b, i, j);
    if (MODE == CV_FWD) return (((int64_t)b * c.Cout + z * c.CoutPG) * c.Ho + i) * c.Wo + j;
    return (((int64_t)b * c.Cin + z * c.CinPG) * c.H + i * c.sH + rh) * c.W + j * c.sW + rw;
  }
  CG_HD int64_t out_rs(const ConvGemmArgs& c) const {
    return MODE == CV_FWD ? (int64_t)c.Ho * c.Wo : MODE == CV_DGRAD ? (int64_t)c.H * c.W : (int64_t)c.N;
  }
};

// The 16 terms of a stage in LDS.
struct KTab { uint32_t a[kCBK], b[kCBK], t0[kCBK], t1[kCBK]; };

// What one thread loads of a stage. A: 4 k of a row (a tile of 32 rows: the first two wavefronts); in the input gradient
// lanes take consecutive rows, kH * kW elements apart, since its consecutive k lie further apart. B, conv2d and
// input gradient: PB consecutive k of row tid % BN, so a wavefront's loads take consecutive output positions. Weight
// gradient: 4 k of rows tid / 4 + 64 e, whose consecutive k are consecutive positions.
template <int MODE, int BM, int BN, int F>
struct ConvLoader {
  static constexpr bool ROWS = MODE != CV_WGRAD;
  static constexpr int PB = BN * kCBK / kCT;          // elements of B per thread: 8 or 4
  static constexpr int NR = ROWS ? 1 : PB / 4;        // its rows
  uint32_t arow;
  BTerm brow[NR];
  int ka, kb;                                         // first k in the stage

  CG_HD static int a_row(int tid) { return MODE == CV_DGRAD ? tid % BM : tid >> 2; }
  CG_HD static int b_row(int tid, int e) { return ROWS ? tid % BN : (tid >> 2) + 64 * e; }

  CG_HD void init(const ConvMap<MODE, F>& map, const ConvGemmArgs& c, int tid) {
    arow = map.a_row(c, map.m0 + a_row(tid));
    for (int e = 0; e < NR; ++e) brow[e] = map.b_row(c, map.n0 + b_row(tid, e));
    ka = MODE == CV_DGRAD ? tid / BM * 4 & 12 : (tid & 3) * 4;
    kb = ROWS ? tid / BN * PB : (tid & 3) * 4;
  }
  CG_HD void load(const ConvMap<MODE, F>& map, const ConvGemmArgs& c, const KTab& t, bool has_a, float* qa,
                  float* qb) const {
    if (has_a) {
      if (F & F_AVEC) {
        const f32x4 v = ldb4(map.sa, arow + t.a[ka]);
#pragma unroll
        for (int u = 0; u < 4; ++u) qa[u] = v[u];
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) qa[u] = ldb(map.sa, arow + t.a[ka + u]);
      }
    }
#pragma unroll
    for (int e = 0; e < NR; ++e) {
      const BTerm& r = brow[e];
      if (F & F_BVEC) {
        const f32x4 v = ldb4(map.sb, r.off + t.b[kb]);
#pragma unroll
        for (int u = 0; u < 4; ++u) qb[e * 4 + u] = v[u];
        continue;
      }
      if (F & F_TAP) {
        // lanes outside the image take no part: as out-of-range loads they cost more (48 us in place of 44)
#pragma unroll
        for (int u = 0; u < PB; ++u) qb[u] = 0.0f;
        if (map.outside(c, r.t0, r.t1, t.t0[kb], t.t1[kb]) == 0) {
#pragma unroll
          for (int u = 0; u < PB; ++u) qb[u] = ldb(map.sb, r.off + t.b[kb + u]);
        }
        continue;
      }
#pragma unroll
      for (int u = 0; u < PB / NR; ++u) {
        const int k = kb + u;
        const uint32_t out = map.outside(c, r.t0, r.t1, t.t0[k], t.t1[k]);
        qb[e * (PB / NR) + u] = ldb(map.sb, (r.off + t.b[k]) | out);
      }
    }
  }
};

// (the tiles: see k_conv_gemm)
struct ConvPlan { int mode, bm, bn, splits, k_per_split, tiles_m, tiles_n; int64_t blocks; };

inline ConvPlan conv_plan(int mode, const ConvDesc& d) {
  ConvPlan p{};
  p.mode = mode;
  const int64_t CoutPG = d.Cout / d.G, khw = d.kH * d.kW;
  const int64_t M = mode == CV_DGRAD ? d.CinPG : CoutPG;
  // (input gradient: the columns of phase 0, the largest)
  const int64_t N = mode == CV_FWD     ? d.B * d.Ho * d.Wo
                    : mode == CV_DGRAD ? d.B * ((d.H + d.sH - 1) / d.sH) * ((d.W + d.sW - 1) / d.sW)
                                       : d.CinPG * khw;
  const int64_t K = mode == CV_FWD ? d.CinPG * khw : mode == CV_DGRAD ? CoutPG * khw : d.B * d.Ho * d.Wo;
  const int64_t Z = d.G, phases = mode == CV_DGRAD ? std::min(d.sH, d.H) * std::min(d.sW, d.W) : 1;
  p.bm = M <= 32 ? 32 : 64;
  p.bn = p.bm == 32 ? 128 : 64;
  p.tiles_m = (int)((M + p.bm - 1) / p.bm);
  p.tiles_n = (int)((N + p.bn - 1) / p.bn * phases);
  p.splits = 1;
  p.k_per_split = (int)K;
  if (mode == CV_WGRAD) {
    // Enough blocks to fill the chip twice over, each split at least 256 k, and the
    // partials within kConvWorkBytes.
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n * Z;
    int64_t s = (512 + tiles - 1) / tiles;
    s = std::min<int64_t>(s, std::max<int64_t>(1, K / 256));
    const int64_t per = Z * M * N * 4;
    s = std::min<int64_t>(s, std::max<int64_t>(1, kConvWorkBytes / per));
    if (s > 1) {
      int64_t kps = (K + s - 1) / s;
      kps = (kps + 31) / 32 * 32;
      s = (K + kps - 1) / kps;
      p.k_per_split = (int)kps;
    }
    p.splits = (int)s;
  }
  p.blocks = (int64_t)p.tiles_m * p.tiles_n * Z * p.splits;
  return p;
}

inline ConvGemmArgs make_args(const ConvDesc& d, const ConvPlan& p) {
  ConvGemmArgs a{};
  a.B = (int)d.B; a.Cin = (int)d.Cin; a.H = (int)d.H; a.W = (int)d.W; a.Cout = (int)d.Cout;
  a.CinPG = (int)d.CinPG; a.CoutPG = (int)(d.Cout / d.G); a.kH = (int)d.kH; a.kW = (int)d.kW;
  a.Ho = (int)d.Ho; a.Wo = (int)d.Wo; a.G = (int)d.G; a.sH = (int)d.sH; a.sW = (int)d.sW;
  a.pH = (int)d.pH; a.pW = (int)d.pW;
  const int khw = a.kH * a.kW;
  if (p.mode == CV_FWD) { a.M = a.CoutPG; a.N = a.B * a.Ho * a.Wo; a.K = a.CinPG * khw; }
  else if (p.mode == CV_DGRAD) { a.M = a.CinPG; a.N = a.B * a.H * a.W; a.K = a.CoutPG * khw; }
  else { a.M = a.CoutPG; a.N = a.CinPG * khw; a.K = a.B * a.Ho * a.Wo; }
  a.tiles_m = p.tiles_m; a.tiles_n = p.tiles_n; a.splits = p.splits; a.k_per_split = p.k_per_split;
  a.phases = p.mode == CV_DGRAD ? std::min(a.sH, a.H) * std::min(a.sW, a.W) : 1;
  // A tap outside the image exists iff padding is used or the last window overhangs.
  a.pad = (a.pH > 0 || a.pW > 0 || (a.Ho - 1) * a.sH + a.kH > a.H || (a.Wo - 1) * a.sW + a.kW > a.W) ? 1 : 0;
  a.dKHW = make_fastdiv((uint32_t)khw);
  a.dKW = make_fastdiv((uint32_t)a.kW);
  a.dWo = make_fastdiv((uint32_t)a.Wo);
  a.dHoWo = make_fastdiv((uint32_t)(a.Ho * a.Wo));
  a.dPhW = make_fastdiv((uint32_t)std::min(a.sW, a.W));
  a.dCpg = make_fastdiv((uint32_t)std::max(1, a.CoutPG));
  a.dTn = make_fastdiv((uint32_t)std::max(1, a.tiles_n));
  a.dPh = make_fastdiv((uint32_t)a.phases);
  return a;
}

// Loader flags of a launch.
inline int conv_flags(const ConvGemmArgs& a, int mode) {
  if (a.kH > 32 || a.kW > 32) return F_WIDE | (mode == CV_DGRAD ? 0 : F_PAD);
  if (mode == CV_DGRAD) return a.CoutPG % 8 == 0 ? F_TAP : 0;
  int f = a.pad ? F_PAD : 0;
  if (mode == CV_FWD) return f | (a.K % 4 == 0 ? F_AVEC : 0);
  if (a.Ho * a.Wo % 4 == 0) f |= F_AVEC;
  if (!a.pad && a.sW == 1 && a.Wo % 4 == 0) f |= F_BVEC;
  return f;
}

// Every tensor, offset and launch indexable in 32 bits, and a geometry the maps assume.
inline bool conv_ok(const ConvDesc& d) {
  const int64_t lim = int64_t(1) << 29;
  if (d.B <= 0 || d.G <= 0 || d.Cout % d.G != 0 || d.sH <= 0 || d.sW <= 0 || d.Ho <= 0 || d.Wo <= 0 || d.kH <= 0 ||
      d.kW <= 0 || d.pH < 0 || d.pW < 0 || d.H <= 0 || d.W <= 0)
    return false;
  // the position terms of the input gradient reach (b, g*CoutPG, Ho + pH, Wo + pW)
  const int64_t big = std::max({d.B * d.Cin * d.H * d.W, d.B * d.Cout * d.Ho * d.Wo, d.Cout * d.CinPG * d.kH * d.kW,
                                d.B * d.Cout * (d.Ho + d.H + d.pH + 1) * (d.Wo + d.W + d.pW + 1),
                                (d.H + d.pH + d.kH) * (d.W + d.pW + d.kW)});
  if (big >= lim) return false;
  for (int mode : {CV_FWD, CV_DGRAD, CV_WGRAD})
    if (conv_plan(mode, d).blocks >= lim) return false;
  return true;
}

#undef CG_HD

}  // namespace cg
}  // namespace tgk
