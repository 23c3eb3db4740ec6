// The filter MLP as a function of the pair distance alone.
//
// PaiNNMessage's filter W(d) = W2 silu(W1 e(d) + b1) + b2 (student_model.py:
// 313-322, 350-355) has one scalar input, the distance d in [0, rc], and 3H
// smooth outputs, and the force adjoint needs it only through W'(d):
//   dE/dd = sum_c (dE/dW_c) W'_c(d).
// So W and W' are tabulated once per weight blob, in float64, and each pair
// interpolates them instead of running 2 (RH + 3H^2) flops forward and as many
// again in the adjoint.  256 molecules of 10-100 atoms at H = 128 (337,000
// pairs): 2560 intervals against 337,000 MLP rows.
//
// Interpolation: cubic Hermite between knots.  The knot spacing h is a power
// of two, so x = d / h, the interval k = floor(x) and t = x - k are exact in
// float32: reading the table adds no rounding to d.  h is at most 1/100 of
// the default basis width rc / R (table_shape); W is read at twice that
// spacing.  For the initialisation of the full student the truncation is then
// 0.02 (W) and 0.15 (W') float32 rounding units of the sum of magnitudes that
// the direct product adds up, and the stored values are rounded once from
// float64, where the direct product rounds every term.
//
// The width of features in d depends on the weights (narrow learned basis
// widths, a steep first layer), so the table checks itself: table_guard_kernel
// compares it with the float64 MLP between the knots, and the flag it raises
// sends the pair kernels back to the direct MFMA path (painn.hip).
//
// Layout per block, float32: W part [Kc + 1][2][3H] = {W, 2h W'} at the knots
// 2h k, then W' part [K + 1][2][3H] = {W', h W''} at the knots h k.

#include <math.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"

namespace mlff {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kTabBlock = 256;
constexpr int kTabWaves = kTabBlock / 64;
constexpr int kTabRows = 16;         // knots (or samples) per block: one MFMA row tile
constexpr int kTabMaxRbf = 32;
constexpr int kGuardStride = 16;     // one sample in every 16 intervals

// Rows of the first layer at one position x[m] per tile row, in float64, left
// in LDS as hs[stream][m][c]:
//   build : h, h', h''  (silu of the pre-activation a and its derivatives in d)
//   GUARD : h, h', |h|, |silu'(a)| sum_j |W1_cj e'_j|
// Raises `bad` when a' moves by more than 1/8 per interval or a basis width
// is under 16 intervals: features that the guard's samples could miss.
template <int H, bool GUARD>
__device__ void table_hidden(const float* __restrict__ w, const LayerW& lw,
                             const float* __restrict__ centers, const float* __restrict__ widths,
                             int R, double rc, double h, double x0, double dx,
                             double (&es)[3][kTabRows][kTabMaxRbf],
                             double* __restrict__ hs, int32_t* __restrict__ bad) {
  constexpr int LDS = H + 2, PL = kTabRows * LDS;
  const double q = M_PI / rc;
  bool steep = false;
  for (int idx = threadIdx.x; idx < kTabRows * R; idx += kTabBlock) {
    const int m = idx / R, j = idx - m * R;
    const double d = x0 + m * dx;
    const double wd = (double)widths[j], g = 1.0 / (wd * wd), u = d - (double)centers[j];
    const double phi = exp(-g * u * u);
    const double p1 = -2.0 * g * u * phi, p2 = (4.0 * g * g * u * u - 2.0 * g) * phi;
    const double c0 = 0.5 * (cos(q * d) + 1.0), c1 = -0.5 * q * sin(q * d),
                 c2 = -0.5 * q * q * cos(q * d);
    es[0][m][j] = phi * c0;
    es[1][m][j] = p1 * c0 + phi * c1;
    es[2][m][j] = p2 * c0 + 2.0 * p1 * c1 + phi * c2;
    steep |= !(fabs(wd) >= 16.0 * h);
  }
  __syncthreads();
  const float* w1t = w + lw.f1t;   // [RP][H]
  for (int idx = threadIdx.x; idx < kTabRows * H; idx += kTabBlock) {
    const int m = idx / H, c = idx - m * H;
    double a = (double)w[lw.f1b + c], a1 = 0.0, a2 = 0.0, s1 = 0.0;
    for (int j = 0; j < R; ++j) {
      const double wj = (double)w1t[j * H + c];
      a += wj * es[0][m][j];
      a1 += wj * es[1][m][j];
      if (GUARD) s1 += fabs(wj * es[1][m][j]);
      else a2 += wj * es[2][m][j];
    }
    const double sg = 1.0 / (1.0 + exp(-a)), sm = 1.0 / (1.0 + exp(a));
    const double f1 = sg * (1.0 + a * sm);                        // silu'
    const double f2 = sg * sm * (2.0 + a * (sm - sg));            // silu''
    double* o = hs + m * LDS + c;
    o[0] = a * sg;
    o[PL] = f1 * a1;
    if (GUARD) {
      o[2 * PL] = fabs(a * sg);
      o[3 * PL] = fabs(f1) * s1;
    } else {
      o[2 * PL] = f2 * a1 * a1 + f1 * a2;
    }
    steep |= !(fabs(a1) * h <= 0.125);
  }
  if (steep) *bad = 1;
  __syncthreads();
}

// acc[s] = hs[s] W2^T for the 16 output columns cb.., on the FP64 matrix
// cores.  As in mma_tile, lane group g feeds k = 16 q + 4 g + s in sub-step s
// of slab q for both operands.  acc[s][i] is row 4 i + lane / 16, column
// cb + lane % 16 (ABS: of |W2| for the streams from ABS on).
template <int H, int NS, int ABS>
__device__ __forceinline__ void table_product(const double* __restrict__ hs,
                                              const float* __restrict__ w2, int cb,
                                              d4 (&acc)[NS]) {
  constexpr int LDS = H + 2, PL = kTabRows * LDS, S = H / 16;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const float* brow = w2 + (size_t)(cb + r) * H + 4 * g;
  f4 b[S];
#pragma unroll
  for (int q = 0; q < S; ++q) b[q] = *reinterpret_cast<const f4*>(brow + 16 * q);
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = d4{0.0, 0.0, 0.0, 0.0};
  const double* arow = hs + r * LDS + 4 * g;
#pragma unroll
  for (int q = 0; q < S; ++q)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const double bv = (double)b[q][s];
#pragma unroll
      for (int t = 0; t < NS; ++t)
        acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(arow[t * PL + 16 * q + s],
                                                      t < ABS ? bv : fabs(bv), acc[t], 0, 0, 0);
    }
}

// Block (k / 16, l): sixteen knots of block l.  FP64 matrix work, 3 x 3H x H
// multiply-adds per knot (0.75 GFLOP per block at H = 128, rc = 5, R = 20).
template <int H>
__global__ __launch_bounds__(kTabBlock) void table_build_kernel(
    const float* __restrict__ w, ModelW mw, TableShape ts, float rc, float* __restrict__ tab,
    int32_t* __restrict__ bad) {
  constexpr int LDS = H + 2, CT = 3 * H / 16;
  __shared__ double es[3][kTabRows][kTabMaxRbf];
  __shared__ __align__(16) double hs[3 * kTabRows * LDS];
  const LayerW& lw = mw.layer[blockIdx.y];
  const double h = ts.h;
  const int k0 = blockIdx.x * kTabRows;
  table_hidden<H, false>(w, lw, w + mw.centers, w + mw.widths, mw.R, (double)rc, h, k0 * h, h, es,
                         hs, bad);
  float* wt = tab + blockIdx.y * ts.layer_floats;
  float* dt = wt + ts.d_off;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  for (int ct = wave; ct < CT; ct += kTabWaves) {
    d4 acc[3];
    table_product<H, 3, 3>(hs, w + lw.f2w, 16 * ct, acc);
    const int c = 16 * ct + r;
    const double b2 = (double)w[lw.f2b + c];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + 4 * i + g;
      if (k <= ts.K) {
        float* o = dt + (size_t)k * 2 * 3 * H + c;
        o[0] = (float)acc[1][i];
        o[3 * H] = (float)(h * acc[2][i]);
      }
      if (k % 2 == 0 && k / 2 <= ts.Kc) {
        float* o = wt + (size_t)(k / 2) * 2 * 3 * H + c;
        o[0] = (float)(acc[0][i] + b2);
        o[3 * H] = (float)(2.0 * h * acc[1][i]);
      }
    }
  }
}

__device__ __forceinline__ double hermite64(const float* __restrict__ part, int C, double x,
                                            int K) {
  const int k = min((int)x, K - 1);
  const double t = x - k, u = 1.0 - t;
  const float* p = part + (size_t)k * 2 * C;
  return p[0] + t * t * (3.0 - 2.0 * t) * ((double)p[2 * C] - p[0]) + t * u * u * p[C] -
         t * t * u * p[3 * C];
}

// Sample s sits in the middle of fine interval 16 s + 8, a quarter into a W
// interval.  The interpolants of the stored values, evaluated in float64, must
// be within one float32 rounding unit of the sum of magnitudes behind them: the
// truncation and the one rounding of each knot (half a unit of the value at
// most).  Where the filter vanishes (towards the cutoff, with zero biases) the
// sum at the point is no measure: a sixteenth of the largest one within 256
// intervals is added.  A NaN fails too.
template <int H>
__global__ __launch_bounds__(kTabBlock) void table_guard_kernel(
    const float* __restrict__ w, ModelW mw, TableShape ts, float rc,
    const float* __restrict__ tab, int32_t* __restrict__ bad) {
  constexpr int LDS = H + 2, CT = 3 * H / 16;
  __shared__ double es[3][kTabRows][kTabMaxRbf];
  __shared__ __align__(16) double hs[4 * kTabRows * LDS];
  const LayerW& lw = mw.layer[blockIdx.z];
  const double h = ts.h;
  const int s0 = blockIdx.x * kTabRows;
  const double dx = kGuardStride * h, x0 = s0 * dx + (kGuardStride / 2 + 0.5) * h;
  table_hidden<H, true>(w, lw, w + mw.centers, w + mw.widths, mw.R, (double)rc, h, x0, dx, es, hs,
                        bad);
  const TableView tv = table_view(ts, tab, blockIdx.z, 3 * H);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int ct = blockIdx.y * kTabWaves + wave;
  if (ct >= CT) return;
  d4 acc[4];
  table_product<H, 4, 2>(hs, w + lw.f2w, 16 * ct, acc);
  const int c = 16 * ct + r;
  const double b2 = (double)w[lw.f2b + c];
  constexpr double kUnit = 1.0 / (1 << 24), kFloor = 1.0 / 16;
  // largest sums of the block's samples (256 intervals)
  double top = 0.0, top1 = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    top = fmax(top, acc[2][i]);
    top1 = fmax(top1, acc[3][i]);
  }
#pragma unroll
  for (int off = 16; off < 64; off <<= 1) {
    top = fmax(top, __shfl_xor(top, off, 64));
    top1 = fmax(top1, __shfl_xor(top1, off, 64));
  }
  bool off = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const double d = x0 + (4 * i + g) * dx;
    if (d > (double)rc) continue;
    const double W = hermite64(tv.w + c, 3 * H, d * tv.inv_c, tv.Kc);
    const double D = hermite64(tv.d + c, 3 * H, d * tv.inv, tv.K);
    off |= !(fabs(W - (acc[0][i] + b2)) <= kUnit * (acc[2][i] + fabs(b2) + kFloor * top));
    off |= !(fabs(D - acc[1][i]) <= kUnit * (acc[3][i] + kFloor * top1));
  }
  if (off) *bad = 1;
}

// ---------------------------------------------------------------------------
// W_p of every pair, four columns per thread.  Bound by the 3H floats written
// per pair (HBM) and the 4 x 3H read from the table (L2); kTabUnroll pairs'
// table rows are in flight per thread.  One launch takes all blocks
// (blockIdx.y): with few pairs a launch is mostly its own latency (60 atoms, three
// blocks: 7.7 us against 3 x 4.8 us), and the embedding rides along (blockIdx.y
// == L; 3.9 us by itself).
// ---------------------------------------------------------------------------
constexpr int kTabUnroll = 4;

template <int H>
__global__ __launch_bounds__(kTabBlock) void filter_table_fwd_kernel(
    const float4* __restrict__ geom, const int32_t* __restrict__ counts, int32_t pcap,
    TableView tv, int64_t layer_floats, const int32_t* __restrict__ gate, float* __restrict__ Wf,
    int L, int N, const int64_t* __restrict__ Z, const float* __restrict__ emb,
    float* __restrict__ S0, float* __restrict__ V0, bool skip) {
  if ((int)blockIdx.y == L) {
    for (int idx = blockIdx.x * kTabBlock + threadIdx.x; idx < N * (H / 4);
         idx += gridDim.x * kTabBlock)
      embed_item<H>(idx, Z, emb, S0, V0);
    return;
  }
  if (gate != nullptr && *gate != 0) return;
  const float* tab = tv.w + blockIdx.y * layer_floats;
  float* Wout = Wf + blockIdx.y * (size_t)pcap * 3 * H;
  const int P = min(counts[MLFF_COUNT_PAIRS], pcap);
  // Q items of four columns per pair: all of W, or (zero_vectors) without Wv1
  auto fill = [&](auto items) {
    constexpr int Q = decltype(items)::value;
    const int64_t total = (int64_t)P * Q;
    constexpr int kItems = kTabBlock * kTabUnroll;
    auto column = [](int q) { return 4 * q + (Q < 3 * H / 4 && q >= H / 4 ? H : 0); };
    for (int64_t base = (int64_t)blockIdx.x * kItems; base < total;
         base += (int64_t)gridDim.x * kItems) {
      TableAt at[kTabUnroll];
      f4 v[kTabUnroll][4];
      // items past the end read the last pair and are not stored
#pragma unroll
      for (int u = 0; u < kTabUnroll; ++u) {
        const int64_t it = min(base + u * kTabBlock + threadIdx.x, total - 1);
        const int p = (int)(it / Q), c = column((int)(it - (int64_t)p * Q));
        at[u] = table_at(geom[p].w, tv.inv_c, tv.Kc);
        const float* row = tab + (size_t)at[u].k * 2 * 3 * H + c;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[u][k] = *reinterpret_cast<const f4*>(row + k * 3 * H);
      }
#pragma unroll
      for (int u = 0; u < kTabUnroll; ++u) {
        const int64_t it = base + u * kTabBlock + threadIdx.x;
        if (it < total) {
          const f4 o = hermite(at[u], v[u][0], v[u][1], v[u][2], v[u][3]);
          const int64_t p = it / Q;
          __builtin_nontemporal_store(
              o, reinterpret_cast<f4*>(Wout + p * 3 * H + column((int)(it - p * Q))));
        }
      }
    }
  };
  if (skip && blockIdx.y == 0) fill(std::integral_constant<int, 2 * H / 4>{});
  else fill(std::integral_constant<int, 3 * H / 4>{});
}

// ---------------------------------------------------------------------------
// Filter adjoint of pair p = (a < b) from the table (see filter_bwd_kernel for
// the terms): H/4 lanes per pair, four channels each, gather both endpoints'
// features and gradients (the lower atom's once for a run of consecutive pairs,
// see pair_run), form dL/dW_p in registers and contract it with
// W'(d_p) to dL/dd, and (gv_a - gv_b) with Wv2 to dL/du.  Bound by the gathers
// (16H floats per pair) and the 12H floats of the W' rows, all from L2.  The
// blocks' terms meet in force_gather_kernel, so all blocks (blockIdx.y) run in
// one launch once the last gradients are there (60 atoms, three blocks: 7.6 us
// against 3 x 4.9 us one by one).  A split into 32-channel slices, one slice's
// table per XCD's L2, was slower: 282 us a block against 234 us for 256
// molecules at H = 128, although a block's W' table (7.9 MB) exceeds an L2.
// ---------------------------------------------------------------------------
template <int H>
__global__ __launch_bounds__(kTabBlock) void filter_table_bwd_kernel(
    const int32_t* __restrict__ counts, int32_t pcap, const int32_t* __restrict__ pair_lo,
    const int32_t* __restrict__ pair_hi, const float4* __restrict__ geom, TableView tv,
    int64_t layer_floats, const int32_t* __restrict__ gate, const float* __restrict__ Wf, int N,
    const float* __restrict__ s_in, const float* __restrict__ v_in,
    const float* __restrict__ gs1, const float* __restrict__ gv1, float4* __restrict__ pacc,
    bool skip, int run) {
  constexpr int G = H / 4, PPB = kTabBlock / G;
  if (gate != nullptr && *gate != 0) return;
  const int l = blockIdx.y;
  const bool vectors = !(skip && l == 0);
  const size_t nh = (size_t)l * N * H;
  const float* tab = tv.d + l * layer_floats;
  Wf += (size_t)l * pcap * 3 * H;
  s_in += nh;
  v_in += 3 * nh;
  gs1 += nh;
  gv1 += 3 * nh;
  pacc += (size_t)l * pcap;
  const int P = min(counts[MLFF_COUNT_PAIRS], pcap);
  int t0, t1, tstep;
  persistent_range((P + PPB * run - 1) / (PPB * run), t0, t1, tstep);
  const int c = 4 * (threadIdx.x % G);
  auto ld = [&](const float* q) { return *reinterpret_cast<const f4*>(q); };
  for (int tile = t0; tile < t1; tile += tstep) {
    const int first = (tile * PPB + threadIdx.x / G) * run;
    int a = -1;
    f4 sa = {}, ga = {}, va0 = {}, va1 = {}, va2 = {}, qa0 = {}, qa1 = {}, qa2 = {};
    for (int r = 0; r < run; ++r) {
      const int p = min(first + r, P - 1);   // past the end: the last pair, not stored
      const int lo = pair_lo[p], b = pair_hi[p];
      const float4 gm = geom[p];
      const float* vb = v_in + (size_t)b * 3 * H + c;
      const float* qb = gv1 + (size_t)b * 3 * H + c;
      const TableAt at = table_at(gm.w, tv.inv, tv.K);
      const float* row = tab + (size_t)at.k * 2 * 3 * H + c;
      if (lo != a) {
        a = lo;
        const float* va = v_in + (size_t)a * 3 * H + c;
        const float* qa = gv1 + (size_t)a * 3 * H + c;
        sa = ld(s_in + (size_t)a * H + c);
        ga = ld(gs1 + (size_t)a * H + c);
        qa0 = ld(qa), qa1 = ld(qa + H), qa2 = ld(qa + 2 * H);
        if (vectors) va0 = ld(va), va1 = ld(va + H), va2 = ld(va + 2 * H);
      }
      const f4 sb = ld(s_in + (size_t)b * H + c);
      const f4 gb = ld(gs1 + (size_t)b * H + c);
      const f4 wv2 = ld(Wf + (size_t)p * 3 * H + 2 * H + c);
      f4 acc = (ga * sb + gb * sa) *
               hermite(at, ld(row), ld(row + 3 * H), ld(row + 6 * H), ld(row + 9 * H));
      const f4 qb0 = ld(qb), qb1 = ld(qb + H), qb2 = ld(qb + 2 * H);
      if (vectors) {
        const f4 g1 = qa0 * ld(vb) + qa1 * ld(vb + H) + qa2 * ld(vb + 2 * H) + qb0 * va0 +
                      qb1 * va1 + qb2 * va2;
        const float* r1 = row + H;
        acc += g1 * hermite(at, ld(r1), ld(r1 + 3 * H), ld(r1 + 6 * H), ld(r1 + 9 * H));
      }
      const float den = gm.w + kEdgeEps;
      const float ux = gm.x / den, uy = gm.y / den, uz = gm.z / den;
      const f4 d0 = qa0 - qb0, d1 = qa1 - qb1, d2 = qa2 - qb2;
      {
        const float* r2 = row + 2 * H;
        acc += (ux * d0 + uy * d1 + uz * d2) *
               hermite(at, ld(r2), ld(r2 + 3 * H), ld(r2 + 6 * H), ld(r2 + 9 * H));
      }
      const f4 w0 = wv2 * d0, w1 = wv2 * d1, w2 = wv2 * d2;
      const float gd = group_sum<G>((acc[0] + acc[1]) + (acc[2] + acc[3]));
      const float gx = group_sum<G>((w0[0] + w0[1]) + (w0[2] + w0[3]));
      const float gy = group_sum<G>((w1[0] + w1[1]) + (w1[2] + w1[3]));
      const float gz = group_sum<G>((w2[0] + w2[1]) + (w2[2] + w2[3]));
      if (c == 0 && first + r < P) pacc[p] = make_float4(gx, gy, gz, gd);
    }
  }
}

template <int H>
hipError_t build_impl(const Buffers& b, hipStream_t s) {
  const TableShape& ts = b.ts;
  const int rows = 2 * ts.Kc + 1;
  table_build_kernel<H><<<dim3((rows + kTabRows - 1) / kTabRows, b.L), kTabBlock, 0, s>>>(
      b.w, *b.mw, ts, b.rc, b.tab, b.tab_bad);
  const int ns = (ts.K + kGuardStride - 1) / kGuardStride;
  table_guard_kernel<H><<<dim3((ns + kTabRows - 1) / kTabRows,
                               (3 * H / 16 + kTabWaves - 1) / kTabWaves, b.L),
                          kTabBlock, 0, s>>>(b.w, *b.mw, ts, b.rc, b.tab, b.tab_bad);
  return hipGetLastError();
}

// Workgroups of a pair kernel of `work` units over the pair capacity: the
// plan's persistent grid at most, a multiple of 8 for the XCD-interleaved order
int table_grid(const Buffers& b, int64_t units) {
  const int64_t n = (units + 7) / 8 * 8;
  return (int)(n < 8 ? 8 : (n < b.blocks ? n : b.blocks));
}

// Consecutive pairs that one group of lanes of the filter adjoint takes, so that
// the features of their common lower atom are read once: four from 64 rounds of
// resident wavefronts (256 CUs x 16) on, two from 16 on, one below.  Runs of
// 1 / 2 / 4 / 8 took 621 / 583 / 575 / 607 us for 256 molecules at H = 128 (100
// rounds), 150 / 143 / 146 / 168 us for 1000 periodic waters (24 rounds), 7.5 / 8.0
// / 10.4 / 17.3 us for 60 atoms.  Indices read one pair ahead: 1-2 % slower.
// Whole evaluations of 50-atom molecules at H = 128, runs of 1 / 2 / 4: 230 / 232 / 242 us
// at 9 rounds, 346 / 345 / 357 at 18, 603 / 599 / 606 at 36, 1043 / 1029 / 1038 at 71,
// 1804 / 1778 / 1777 at 125; at H = 32 224 / 222 / 224 at 12, 353 / 350 / 354 at 21.
int pair_run(int H, int64_t pcap, int blocks) {
  const int64_t rounds = pcap * (H / 4) * blocks / (256 * 16 * 64);
  return rounds >= 64 ? 4 : rounds >= 16 ? 2 : 1;
}

}  // namespace

// The finest spacing wanted is 1/100 of the default basis width rc / R; below
// 2.56 intervals per basis function (R = 1, 2) at least 256 intervals.
TableShape table_shape(int H, int R, int L, float rc) {
  TableShape t = {};
  if (!(rc >= 1e-3f && rc <= 1e4f)) return t;   // no such model; keeps the exponent small
  const double want = R > 2 ? 100.0 * R : 256.0;
  int e = 0;
  while (ldexp((double)rc, e) < want) ++e;
  while (ldexp((double)rc, e - 1) >= want) --e;
  t.h = ldexp(1.0, -e);
  t.K = (int)ceil(ldexp((double)rc, e));
  t.Kc = (t.K + 1) / 2;
  t.d_off = (int64_t)(t.Kc + 1) * 2 * 3 * H;
  t.layer_floats = t.d_off + (int64_t)(t.K + 1) * 2 * 3 * H;
  t.bytes = 4 * t.layer_floats * L;
  // a plan keeps at most this much for its tables; past it (more than five
  // blocks at H = 128, R = 20) the pair kernels stay on the direct product
  if (t.bytes > kTableMaxBytes) t.bytes = 0;
  return t;
}

hipError_t build_tables(const Buffers& b, hipStream_t s) {
  switch (b.H) {
    case 32: return build_impl<32>(b, s);
    case 64: return build_impl<64>(b, s);
    case 128: return build_impl<128>(b, s);
    default: return hipErrorInvalidValue;
  }
}

template <int H>
void launch_filter_table_fwd(const Buffers& b, hipStream_t s, int l0, int l1, bool embed,
                             bool all) {
  constexpr int Q = 3 * H / 4;
  int64_t units = ((int64_t)b.pcap * Q + kTabBlock * kTabUnroll - 1) / (kTabBlock * kTabUnroll);
  if (embed) units = std::max(units, ((int64_t)b.N * (H / 4) + kTabBlock - 1) / kTabBlock);
  filter_table_fwd_kernel<H><<<dim3(table_grid(b, units), l1 - l0 + embed), kTabBlock, 0, s>>>(
      b.geom, b.counts, b.pcap, table_view(b.ts, b.tab, l0, 3 * H), b.ts.layer_floats, b.gate,
      b.Wf + (size_t)l0 * b.pcap * 3 * H, l1 - l0, b.N, b.numbers, b.w + b.mw->emb, b.S, b.V,
      l0 == 0 && zero_vectors(b) && !all);
}

template <int H>
void launch_filter_table_bwd(const Buffers& b, hipStream_t s, int l0, int l1) {
  constexpr int PPB = kTabBlock / (H / 4);
  const size_t nh = (size_t)l0 * b.N * H;
  const int run = pair_run(H, b.pcap, l1 - l0), per = PPB * run;
  filter_table_bwd_kernel<H><<<dim3(table_grid(b, ((int64_t)b.pcap + per - 1) / per), l1 - l0),
                               kTabBlock, 0, s>>>(
      b.counts, b.pcap, b.pair_lo, b.pair_hi, b.geom, table_view(b.ts, b.tab, l0, 3 * H),
      b.ts.layer_floats, b.gate, b.Wf + (size_t)l0 * b.pcap * 3 * H, b.N, b.S + nh, b.V + 3 * nh,
      b.gS1 + nh, b.gV1 + 3 * nh, b.pacc + (size_t)l0 * b.pcap, l0 == 0 && zero_vectors(b), run);
}

#define MLFF_TABLE_INST(HH)                                                         \
  template void launch_filter_table_fwd<HH>(const Buffers&, hipStream_t, int, int, bool, bool); \
  template void launch_filter_table_bwd<HH>(const Buffers&, hipStream_t, int, int);
MLFF_TABLE_INST(32)
MLFF_TABLE_INST(64)
MLFF_TABLE_INST(128)
#undef MLFF_TABLE_INST

}  // namespace mlff
