// Implicit-GEMM convolution (NCHW, f32) on the gfx950 matrix cores (f32 products from
// bf16 MFMAs, as x3_tile in gemm_dev.h). Nothing is materialised: each operand tile is gathered from
// the activations with the convolution's index map while it is staged into LDS.
//
// Per image b and group g (z = b * G + g), the three IR kinds are GEMMs
//   conv2d            Y[co][p]   = sum_k W[co][k]        * X^[k][p]    k = (cl, kh, kw), p = (ho, wo)
//   conv2d_input_grad dX[cl][q]  = sum_k W^T[cl][k]      * dY^[k][q]   k = (col, kh, kw), q = (hi, wi)
//   conv2d_weight_grad dW[co][n] = sum_k dY[co][k]       * X~[k][n]    k = (b, ho, wo), n = (cl, kh, kw)
// with X^[k][p] = x[b, g*CinPG+cl, ho*sH+kh-pH, wo*sW+kw-pW] (zero outside the image),
// dY^[k][q] = dy[b, g*CoutPG+col, ho, wo] for the (ho, wo) with ho*sH+kh-pH = hi and
// wo*sW+kw-pW = wi (zero when there is none), and X~ the same gather as X^ with the roles
// of k and n exchanged. The weight gradient reduces over the whole batch, so its k range
// is split across blocks (deterministic: each split writes its own partial tile, a second
// kernel adds the partials in split order).
//
// 256 threads make a 64 x 64 or 32 x 128 output tile in 32 x 32 wavefront tiles. Every
// index is 32-bit (the host checks the sizes) and divisions by the geometry use precomputed
// multiplicative inverses (FastDiv).
#include "conv_gemm_dev.h"
#include "gemm_dev.h"

#include <algorithm>
#include <stdexcept>

namespace tgk {
namespace {

using namespace gd;
using namespace cg;


// An operand's ROWS x 16 stage in LDS: three planes of bf16, a row of 32 bytes each (XTile's layout).
template <int ROWS>
struct ConvStage {
  static constexpr int PLANE = ROWS * 32, SIZE = 3 * PLANE;
  template <int N>   // N k of a row, from k on: 4 or 8
  __device__ __forceinline__ static void store(const float* q, char* L, int row, int k) {
    uint32_t h[N / 2], m[N / 2], l[N / 2];
#pragma unroll
    for (int u = 0; u < N / 2; ++u) split3(q[2 * u], q[2 * u + 1], h[u], m[u], l[u]);
    char* p = L + XTile<64, true>::at(row, k >> 3) + (k & 7) * 2;
    put<N>(p, h);
    put<N>(p + PLANE, m);
    put<N>(p + 2 * PLANE, l);
  }
  template <int N>
  __device__ __forceinline__ static void put(char* p, const uint32_t* v) {
    if constexpr (N == 8) *reinterpret_cast<u32x4*>(p) = (u32x4){v[0], v[1], v[2], v[3]};
    else *reinterpret_cast<u32x2*>(p) = (u32x2){v[0], v[1]};
  }
  __device__ __forceinline__ static bf16x8 frag(const char* L, int plane, int row, int h) {
    return *reinterpret_cast<const bf16x8*>(L + plane * PLANE + XTile<64, true>::at(row, h));
  }
};

// f32 products from six bf16 MFMAs, as x3_tile (gemm_dev.h, which gives the arithmetic and its error): the stage in one
// half of the LDS is multiplied while the next is split into the other half and the third from here loaded. The terms of
// four stages (KTab) are found at once by one wavefront.
//
// What bounds it: the vector port, and then the gathers. Per stage a wavefront of a 64 x 64 tile issues 6 MFMAs (which
// keep the port for half their time) and about 95 vector instructions: 8 elements split (5.5 each), their offsets, the
// running sum. An element is split once for each tap it meets. Tile: 4 blocks a CU hide each other's latencies; 64 x 128
// was slower everywhere (its registers admit 3), and 32-row outputs take 128 columns so that A's share stays small.
// [128, 32, 26, 26] * [64, 32, 3, 3]: forward 45 -> 32 us, input gradient 64 -> 44 us, weight gradient 50 -> 33 us
// against f32 MFMAs; [32, 64, 33, 33] * [64, 64, 3, 3] with stride 2: 32 -> 23, 74 -> 23, 30 -> 25 us.
template <int MODE, int BM, int BN, int F>
__global__ __launch_bounds__(kCT, 4) void k_conv_gemm(ConvGemmArgs c) {
  constexpr int WGM = BM >= 64 ? 2 : 1, WGN = 4 / WGM;   // wave grid
  constexpr int TN = BN / WGN / 32;                      // a wavefront's tiles: 32 x (TN * 32)
  static_assert(BM / WGM == 32 && TN >= 1, "bad conv tile");
  using LD = ConvLoader<MODE, BM, BN, F>;
  using SA = ConvStage<BM>;
  using SB = ConvStage<BN>;
  __shared__ __attribute__((aligned(16))) char lds[2][SA::SIZE + SB::SIZE];
  __shared__ __attribute__((aligned(16))) KTab tab[8];   // of stage s in tab[s % 8]

  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm0 = (wave / WGN) * 32, wn0 = (wave % WGN) * TN * 32;
  const int lrow = lane % 32, h = lane / 32;
  const bool has_a = BM == 64 || wave < 2;
  ConvMap<MODE, F> map;
  map.template init<BM, BN>(c, blockIdx.x, gridDim.x);
  if (MODE == CV_DGRAD && map.n0 >= map.N) return;       // a smaller phase than the first
  auto put_terms = [&](int st) {   // of four stages
    const int s = st + lane / kCBK, l = lane % kCBK;
    const KTerm t = map.k_term(c, map.kbeg + s * kCBK + l);
    KTab& k = tab[s & 7];
    k.a[l] = t.a;
    k.b[l] = t.b;
    k.t0[l] = t.t0;
    k.t1[l] = t.t1;
  };
  if (wave == 0) put_terms(0);
  LD ld;
  ld.init(map, c, tid);
  __syncthreads();

  float qa[2][4], qb[2][LD::PB];
  f32x16 acc[TN], part[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = part[j][r] = 0.0f;
  auto load = [&](int st, int set) { ld.load(map, c, tab[st & 7], has_a, qa[set], qb[set]); };
  auto store = [&](int set, float sign) {
    if (has_a) {
      float q[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) q[u] = sign * qa[set][u];
      SA::template store<4>(q, lds[set], LD::a_row(tid), ld.ka);
    }
#pragma unroll
    for (int e = 0; e < LD::NR; ++e)
      SB::template store<LD::PB / LD::NR>(qb[set] + e * (LD::PB / LD::NR), lds[set] + SA::SIZE, LD::b_row(tid, e), ld.kb);
  };
  auto meet = [&]() {   // LDS traffic only: the loads of later stages stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  const int nst = map.kbeg < map.kend ? (map.kend - map.kbeg + kCBK - 1) / kCBK : 0;
  // Stages past the last read as zeros (their terms are masked), so nothing here tests for the end.
  // Every two stages begin a new part, and the running sums take the last. The bf16 MFMAs round towards one side by a
  // little (2^-27 of a part), which over many parts of either sign would be all of the error; so every other part is
  // made of negated A, and the running sums change sign each time: the weight gradient's error over K = 73728 is 1.5e-7 so, 3.9e-7 without.
  auto sign = [](int st) { return (st & 2) ? -1.0f : 1.0f; };
  auto body = [&](int st, auto ptag) {
    constexpr int P = decltype(ptag)::value;
    constexpr bool FRESH = P == 0;
    if (P == 0 && (st & 15) == (wave << 2)) put_terms(st + 4);
    const char *La = lds[P], *Lb = La + SA::SIZE;
    constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};   // small terms first
    bf16x8 a[3], b[TN][3];
#pragma unroll
    for (int o = 0; o < 3; ++o) {
      a[o] = SA::frag(La, o, wm0 + lrow, h);
#pragma unroll
      for (int j = 0; j < TN; ++j) b[j][o] = SB::frag(Lb, o, wn0 + j * 32 + lrow, h);
    }
    store(P ^ 1, sign(st + 1));
    load(st + 3, P ^ 1);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if (FRESH) acc[j] = part[j] - acc[j];
#pragma unroll
      for (int t = 0; t < 6; ++t) {
        const f32x16 p = FRESH && t == 0 ? (f32x16)(0.0f) : part[j];
        part[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[PA[t]], b[j][PB[t]], p, 0, 0, 0);
      }
    }
    meet();
  };
  if (nst > 0) {
    load(0, 0);
    load(1, 1);
    store(0, 1.0f);
    load(2, 0);
  }
  meet();
  for (int st = 0; st < nst; st += 2) {
    body(st, IntTag<0>{});
    if (st + 1 < nst) body(st + 1, IntTag<1>{});
  }
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = sign(nst - 1) * (part[j][r] - acc[j][r]);

  // Values that are not finite do not split (x3_tile): such a wavefront multiplies its tile again with f32 MFMAs.
  float bad = 0.0f;   // 0 * v is 0 for a finite v and NaN otherwise
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) bad = fmaf(acc[j][r], 0.0f, bad);
  if (__builtin_amdgcn_ballot_w64(bad != 0.0f) != 0) {
    const uint32_t ar = map.a_row(c, map.m0 + wm0 + lrow);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const BTerm br = map.b_row(c, map.n0 + wn0 + j * 32 + lrow);
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][r] = 0.0f;
      for (int kb = map.kbeg; kb < map.kend; kb += 32) {
        f32x16 sum = (f32x16)(0.0f);
#pragma unroll 1
        for (int u = 0; u < 32; u += 2) {
          const KTerm t = map.k_term(c, kb + u + h);
          const float av = ldb(map.sa, ar + t.a);
          const float bv = ldb(map.sb, (br.off + t.b) | map.outside(c, br.t0, br.t1, t.t0, t.t1));
          sum = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, sum, 0, 0, 0);
        }
        acc[j] += sum;
      }
    }
  }

  // Register r of lane l holds row (r/4)*8 + (l/32)*4 + r%4, column l%32.
  float* O = (MODE == CV_WGRAD && c.splits > 1) ? c.work : c.out;
  const int64_t rs = map.out_rs(c);
  const bool epi = MODE != CV_WGRAD && c.epi != kConvEpiNone;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int gn = map.n0 + wn0 + j * 32 + lrow;
    const int64_t cofs = map.out_col(c, min(gn, map.N - 1));
    float e[16];
    if (epi) {
      // The layer's pointwise step at the store (one group, G = 1: channel gm). Every bias / mask value is loaded first
      // (clamped in range): loaded between the stores, each would wait for the stores before it.
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gm = min(map.m0 + wm0 + (r / 4) * 8 + h * 4 + (r % 4), c.M - 1);
        e[r] = c.epi == kConvEpiBiasRelu ? c.ebias[gm] : c.emask[cofs + gm * rs];
      }
    }
    if (gn >= map.N) continue;
    float* col = O + cofs;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int gm = map.m0 + wm0 + (r / 4) * 8 + h * 4 + (r % 4);
      if (gm >= c.M) continue;
      float v = acc[j][r];
      if (epi) {
        if (c.epi == kConvEpiBiasRelu) {
          const float a = v + e[r];
          v = a != a ? __uint_as_float(0x7fc00000u) : (a > 0.0f ? a : 0.0f);
        } else {
          v = e[r] > 0.0f ? v : 0.0f;
        }
      }
      col[gm * rs] = v;
    }
  }
}

// dW = sum of the split partials, deterministic. Many outputs: a block of four wavefronts
// takes 64 consecutive outputs (coalesced), wavefront w adds splits w, w + 4, ... in order
// (8 loads in flight, clamped to split 0 past the end), and the four sums are added in
// order through LDS. Few outputs and many splits (small weights reducing over a large
// batch): one wavefront per output, lane l adding splits l, l + 64, ... in order, then a
// fixed butterfly across the lanes.
__global__ __launch_bounds__(256) void k_conv_wgrad_reduce(const float* __restrict__ work, int splits,
                                                           int64_t per_split, float* __restrict__ dw) {
  __shared__ float ws[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t i = (int64_t)blockIdx.x * 64 + lane;
  const int64_t ii = i < per_split ? i : per_split - 1;
  float s = 0.0f;
  for (int sp0 = w; sp0 < splits; sp0 += 4 * 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int sp = sp0 + 4 * u;
      v[u] = work[(int64_t)(sp < splits ? sp : 0) * per_split + ii];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (sp0 + 4 * u < splits) s += v[u];
  }
  ws[w][lane] = s;
  __syncthreads();
  if (w == 0 && i < per_split) dw[i] = ((ws[0][lane] + ws[1][lane]) + ws[2][lane]) + ws[3][lane];
}

__global__ __launch_bounds__(256) void k_conv_wgrad_reduce_wave(const float* __restrict__ work, int splits,
                                                                int64_t per_split, float* __restrict__ dw) {
  const int lane = threadIdx.x % 64;
  const int64_t i = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;   // one output per wavefront
  if (i >= per_split) return;                                      // uniform across the wavefront
  float s = 0.0f;
  for (int sp = lane; sp < splits; sp += 64) s += work[sp * per_split + i];
  s = wave_allsum(s);
  if (lane == 0) dw[i] = s;
}

// ---- convolutions with few taps ------------------------------------------------------------
// A first layer over 1-3 channel images has CinPG * kH * kW <= 16 taps per output: as a
// GEMM its forward has K <= 16 and its weight gradient N <= 16, so most of every 32-wide
// MFMA stage or tile would multiply padding. Both run on the vector ALU instead (f32 FMAs,
// GEMM tolerance like the MFMA path).
constexpr int kSmallTaps = 16;
constexpr int kSmallCo = 4;      // output channels per weight-gradient block
constexpr int kSmallW = 2048;    // forward: a group's weights staged in LDS, CoutPG * kSmallTaps floats

// Tap q = (cl, kh, kw) of an output position: its row and column shift and its channel
// plane offset, decoded once per thread.
struct SmallTaps {
  int dh[kSmallTaps], dw[kSmallTaps];
  uint32_t off[kSmallTaps];
  __device__ __forceinline__ void init(const ConvGemmArgs& c) {
#pragma unroll
    for (int q = 0; q < kSmallTaps; ++q) {
      const int qq = q < c.K ? q : 0;
      const int cl = fdiv(qq, c.dKHW), r = qq - cl * c.kH * c.kW;
      const int kh = fdiv(r, c.dKW), kw = r - kh * c.kW;
      dh[q] = kh - c.pH;
      dw[q] = kw - c.pW;
      off[q] = (uint32_t)(cl * c.H * c.W);
    }
  }
  // The taps of output position (ho, wo) of image plane base `base` (x's (b, g * CinPG)
  // offset), zero outside the image: raw buffer loads, masked ones at an out-of-range
  // offset, so all of them are in flight together.
  __device__ __forceinline__ void gather(const ConvGemmArgs& c, const Src& sx, uint32_t base, int ho, int wo,
                                         float* xv) const {
#pragma unroll
    for (int q = 0; q < kSmallTaps; ++q) {
      const int hi = ho * c.sH + dh[q], wi = wo * c.sW + dw[q];
      const bool ok = q < c.K && inside(hi, c.H) && inside(wi, c.W);
      xv[q] = ldb(sx, boff(ok, base + off[q] + (uint32_t)(hi * c.W + wi)));
    }
  }
};

// Forward: block (image b, group g, 256 positions), one thread per position, every output
// channel of the group from the group's weights in LDS, each row padded with zeros to
// kSmallTaps (the masked taps are zero too), so the product loop has no branches and reads
// each row as four 128-bit broadcasts.
__global__ __launch_bounds__(256) void k_conv_small_fwd(const ConvGemmArgs c) {
  __shared__ __attribute__((aligned(16))) float ws[kSmallW];
  __shared__ float bs[kSmallW / kSmallTaps];   // the group's biases (kConvEpiBiasRelu)
  const int hw = c.Ho * c.Wo;
  const int nchunk = (hw + 255) / 256;
  const int z = blockIdx.x / nchunk, chunk = blockIdx.x - z * nchunk;
  const int b = z / c.G, g = z - b * c.G;
  for (int i = threadIdx.x; i < c.CoutPG * kSmallTaps; i += 256) {
    const int co = i / kSmallTaps, q = i - co * kSmallTaps;
    ws[i] = q < c.K ? c.w[(int64_t)(g * c.CoutPG + co) * c.K + q] : 0.0f;
  }
  if (c.epi == kConvEpiBiasRelu)
    for (int i = threadIdx.x; i < c.CoutPG; i += 256) bs[i] = c.ebias[g * c.CoutPG + i];
  SmallTaps tp;
  tp.init(c);
  __syncthreads();
  const int p = chunk * 256 + threadIdx.x;
  if (p >= hw) return;
  const int ho = fdiv(p, c.dWo), wo = p - ho * c.Wo;
  const Src sx = make_src(c.x, (int64_t)c.B * c.Cin * c.H * c.W);
  float xv[kSmallTaps];
  tp.gather(c, sx, (uint32_t)((b * c.Cin + g * c.CinPG) * c.H * c.W), ho, wo, xv);
  float* y = c.out + (int64_t)(b * c.Cout + g * c.CoutPG) * hw + p;
  for (int co = 0; co < c.CoutPG; ++co) {
    const f32x4* wr = reinterpret_cast<const f32x4*>(ws + co * kSmallTaps);
    float s = 0.0f;
#pragma unroll
    for (int u = 0; u < kSmallTaps / 4; ++u) {
      const f32x4 w4 = wr[u];
#pragma unroll
      for (int e = 0; e < 4; ++e) s = fmaf(w4[e], xv[u * 4 + e], s);
    }
    if (c.epi == kConvEpiBiasRelu) {   // the bias from LDS
      const float a = s + bs[co];
      s = a != a ? __uint_as_float(0x7fc00000u) : (a > 0.0f ? a : 0.0f);
    }
    y[(int64_t)co * hw] = s;
  }
}

// Weight gradient: block (ipb consecutive images, group g, kSmallCo output channels) sums
// dy * tap over the images' positions (threads take positions t, t + 256, ... of each image
// in turn), then across the block in a fixed order: every thread stores its sums in LDS,
// four threads per sum add 64 threads' values each in thread order, and the four quarters
// are added in order, giving the image group's partial dW rows work[ig][g * CoutPG + co][q].
// The partials are added in image-group order. Several images per block spread the fixed
// cost of the block sum over more positions.
__global__ __launch_bounds__(256) void k_conv_small_wgrad(const ConvGemmArgs c) {
  constexpr int NV = kSmallCo * kSmallTaps;
  static_assert(NV * 4 == 256, "four threads per sum");
  __shared__ float red[256][NV + 1];
  const int hw = c.Ho * c.Wo;
  const int nch = (c.CoutPG + kSmallCo - 1) / kSmallCo;
  const int blk = blockIdx.x, cc = blk % nch, z = blk / nch;
  const int ig = z / c.G, g = z - ig * c.G;
  const int tid = threadIdx.x;
  SmallTaps tp;
  tp.init(c);
  const Src sx = make_src(c.x, (int64_t)c.B * c.Cin * c.H * c.W);
  const Src sdy = make_src(c.dy, (int64_t)c.B * c.Cout * hw);
  float acc[kSmallCo][kSmallTaps];
#pragma unroll
  for (int j = 0; j < kSmallCo; ++j)
#pragma unroll
    for (int q = 0; q < kSmallTaps; ++q) acc[j][q] = 0.0f;
  const int bend = min(c.B, (ig + 1) * c.ipb);
  for (int b = ig * c.ipb; b < bend; ++b) {
    const uint32_t xbase = (uint32_t)((b * c.Cin + g * c.CinPG) * c.H * c.W);
    const uint32_t dbase = (uint32_t)((b * c.Cout + g * c.CoutPG + cc * kSmallCo) * hw);
    for (int p = tid; p < hw; p += 256) {
      const int ho = fdiv(p, c.dWo), wo = p - ho * c.Wo;
      float xv[kSmallTaps], d[kSmallCo];
      tp.gather(c, sx, xbase, ho, wo, xv);
#pragma unroll
      for (int j = 0; j < kSmallCo; ++j)
        d[j] = ldb(sdy, boff(cc * kSmallCo + j < c.CoutPG, dbase + (uint32_t)(j * hw + p)));
#pragma unroll
      for (int j = 0; j < kSmallCo; ++j)
#pragma unroll
        for (int q = 0; q < kSmallTaps; ++q) acc[j][q] = fmaf(d[j], xv[q], acc[j][q]);
    }
  }
#pragma unroll
  for (int j = 0; j < kSmallCo; ++j)
#pragma unroll
    for (int q = 0; q < kSmallTaps; ++q) red[tid][j * kSmallTaps + q] = acc[j][q];
  __syncthreads();
  const int v = tid % NV, quarter = tid / NV;   // 256 threads = 4 quarters of the NV sums
  float s = 0.0f;
  for (int i = 0; i < 64; ++i) s += red[quarter * 64 + i][v];
  __syncthreads();
  red[quarter][v] = s;
  __syncthreads();
  if (tid < NV) {
    const int j = tid / kSmallTaps, q = tid % kSmallTaps, co = cc * kSmallCo + j;
    if (co < c.CoutPG && q < c.K) {
      const float t = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
      c.work[(int64_t)ig * c.G * c.CoutPG * c.K + (int64_t)(g * c.CoutPG + co) * c.K + q] = t;
    }
  }
}

// The few-taps weight gradient applies when its per-image partials fit the workspace.
bool small_wgrad_ok(const ConvDesc& d) {
  const int64_t taps = d.CinPG * d.kH * d.kW;
  return taps <= kSmallTaps && d.B * d.Cout * taps * 4 <= kConvWorkBytes;
}

template <int MODE, int F>
void launch_tile(const ConvPlan& p, const ConvGemmArgs& a, hipStream_t st) {
  const dim3 grid((unsigned)p.blocks);
  if (p.bm == 32) klaunch(k_conv_gemm<MODE, 32, 128, F>, grid, kCT, 0, st, a);
  else klaunch(k_conv_gemm<MODE, 64, 64, F>, grid, kCT, 0, st, a);
}

// The loader variant (conv_flags) of a launch picks the instantiation.
template <int MODE>
void launch_mode(const ConvPlan& p, const ConvGemmArgs& a, hipStream_t st) {
  const int f = conv_flags(a, MODE);
  if constexpr (MODE == CV_DGRAD) {
    switch (f) {
      case F_WIDE: return launch_tile<MODE, F_WIDE>(p, a, st);
      case F_TAP: return launch_tile<MODE, F_TAP>(p, a, st);
      default: return launch_tile<MODE, 0>(p, a, st);
    }
  } else {
    switch (f) {
      case F_WIDE | F_PAD: return launch_tile<MODE, F_WIDE | F_PAD>(p, a, st);
      case F_AVEC: return launch_tile<MODE, F_AVEC>(p, a, st);
      case F_PAD: return launch_tile<MODE, F_PAD>(p, a, st);
      case F_AVEC | F_PAD: return launch_tile<MODE, F_AVEC | F_PAD>(p, a, st);
      case F_AVEC | F_BVEC:
        if constexpr (MODE == CV_WGRAD) return launch_tile<MODE, F_AVEC | F_BVEC>(p, a, st);
      default: return launch_tile<MODE, 0>(p, a, st);
    }
  }
}

}  // namespace

bool conv_gemm_ok(const ConvDesc& d) { return conv_ok(d); }

int64_t conv_gemm_workspace_bytes(const ConvDesc& d) {
  if (small_wgrad_ok(d)) return d.B * d.Cout * d.CinPG * d.kH * d.kW * 4;
  const ConvPlan p = conv_plan(CV_WGRAD, d);
  if (p.splits <= 1) return 0;
  return (int64_t)p.splits * d.G * (d.Cout / d.G) * d.CinPG * d.kH * d.kW * 4;
}

void conv2d_gemm(const float* x, const float* w, float* y, const ConvDesc& d, hipStream_t st, const float* bias) {
  const ConvPlan p = conv_plan(CV_FWD, d);
  ConvGemmArgs a = make_args(d, p);
  a.x = x; a.w = w; a.out = y;
  if (bias) {
    if (d.G != 1) throw std::runtime_error("conv2d: a bias epilogue needs one group");
    a.epi = kConvEpiBiasRelu;
    a.ebias = bias;
  }
  if (d.CinPG * d.kH * d.kW <= kSmallTaps && (d.Cout / d.G) * kSmallTaps <= kSmallW) {
    // the K taps of a row of W are contiguous: W[co][cl][kh][kw] = w[co * K + q]
    const int64_t n = d.B * d.G * ((d.Ho * d.Wo + 255) / 256);
    if (n > 0) klaunch(k_conv_small_fwd, (unsigned)n, 256, 0, st, a);
    return;
  }
  if (p.blocks > 0) launch_mode<CV_FWD>(p, a, st);
}

void conv2d_input_grad_gemm(const float* w, const float* dy, float* dx, const ConvDesc& d, hipStream_t st,
                            const float* mask) {
  const ConvPlan p = conv_plan(CV_DGRAD, d);
  ConvGemmArgs a = make_args(d, p);
  a.w = w; a.dy = dy; a.out = dx;
  if (mask) {
    a.epi = kConvEpiReluMask;
    a.emask = mask;
  }
  if (p.blocks > 0) launch_mode<CV_DGRAD>(p, a, st);
}

void conv2d_weight_grad_gemm(const float* x, const float* dy, float* dw, const ConvDesc& d, float* work,
                             hipStream_t st) {
  const ConvPlan p = conv_plan(CV_WGRAD, d);
  ConvGemmArgs a = make_args(d, p);
  a.x = x; a.dy = dy; a.out = dw; a.work = work;
  if (small_wgrad_ok(d)) {
    if (!work) throw std::runtime_error("conv2d_weight_grad: missing workspace");
    if (d.B <= 0 || d.Cout <= 0) return;
    ConvGemmArgs sa = a;   // K: the taps per output (the GEMM view's N)
    sa.K = (int)(d.CinPG * d.kH * d.kW);
    const int64_t per = d.Cout * sa.K;
    const int64_t nch = (a.CoutPG + kSmallCo - 1) / kSmallCo;
    // images per block: about two blocks per CU (the block sum's LDS admits two)
    sa.ipb = (int)std::max<int64_t>(1, d.B * d.G * nch / 512);
    const int64_t ngroups = (d.B + sa.ipb - 1) / sa.ipb;
    klaunch(k_conv_small_wgrad, (unsigned)(ngroups * d.G * nch), 256, 0, st, sa);
    if (per < 16384 && ngroups > 16) {
      klaunch(k_conv_wgrad_reduce_wave, (unsigned)((per + 3) / 4), 256, 0, st, work, (int)ngroups, per, dw);
    } else {
      klaunch(k_conv_wgrad_reduce, (unsigned)((per + 63) / 64), 256, 0, st, work, (int)ngroups, per, dw);
    }
    return;
  }
  if (p.blocks <= 0) return;
  if (p.splits > 1 && !work) throw std::runtime_error("conv2d_weight_grad: missing workspace");
  launch_mode<CV_WGRAD>(p, a, st);
  if (p.splits > 1) {
    const int64_t per = (int64_t)a.G * a.M * a.N;
    if (per < 16384 && p.splits > 16) {
      klaunch(k_conv_wgrad_reduce_wave, (unsigned)((per + 3) / 4), 256, 0, st, work, p.splits, per, dw);
    } else {
      klaunch(k_conv_wgrad_reduce, (unsigned)((per + 63) / 64), 256, 0, st, work, p.splits, per, dw);
    }
  }
}

}  // namespace tgk
