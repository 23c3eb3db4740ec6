// The filter MLP of PaiNNMessage (student_model.py:313-322, 350-355) in the
// force-matching training pass, one fused pair-tile kernel for the forward
// and one for its tangent along a position direction:
//
//   forward:  a = e W1^T + b1,    h = silu(a),          W = h W2^T + b2
//   tangent:  da = de W1^T,       dh = silu'(a) da,     dW = dh W2^T
//
// e (or de) is [P][R] per pair; a, h (da, dh) are [P][H] and W (dW) is
// [P][3H], all row-major float32.
//
// A third kernel runs the reverse of the first layer's product and SiLU for
// the reverse pass (student_model.py:318-322 under autograd), given the
// filter-output adjoint gW [P][3H] and its tangent dgW:
//
//   gh = gW W2,   ga = silu'(a) gh,
//   dgh = dgW W2, dga = silu'(a) dgh + silu''(a) da gh
//
// on the FP32 matrix cores (W2 comes transposed, [H][3H]) or, for H >= 64, the
// bf16 ones.  In the forward and the tangent the first product runs on the FP32
// matrix cores; the second, the large one, on the bf16 matrix cores with both
// operands split into three bf16 parts (six part products, float32
// accuracy), as in the evaluation's filter kernel.  W1 comes padded to RP
// columns (16 or 32, zeros beyond R) and W2 and its transpose as three bf16
// planes, which mlff_filter_planes makes once per weight update.

#include <stdint.h>

#include "common.hpp"
#include "internal.hpp"

namespace mlff {
namespace {

constexpr int kTfBlock = 512;
constexpr int kTfWaves = kTfBlock / 64;
constexpr int kTfMaxRbf = 32;
// pairs per tile: 128 for the compact hidden size, 64 above (LDS: three bf16
// planes of the tile's hidden activations)
template <int H>
constexpr int kTfPairs = H <= 32 ? 128 : 64;

// One block's filters: weights and outputs of the forward (a, h, w) and of its
// tangent (da, dh, dw).
struct FilterRow {
  const float *w1p, *b1;
  const uint16_t* w2;
  const float *b2;
  float *a, *h, *w, *da, *dh, *dw;
};
constexpr int kTfMaxLayers = 8;
struct FilterRows {
  FilterRow row[kTfMaxLayers];
};

// One pair tile's forward (or tangent, TAN) of the filter MLP.
template <int H, int TM, bool TAN>
__device__ __forceinline__ void train_filter_tile(int pbase, int P, int R, int RP, const float* x,
                                                  const FilterRow& q, float* e_lds,
                                                  uint16_t* h_bf) {
  constexpr int RT = TM / 16;
  constexpr int LDE = kTfMaxRbf + 4;
  constexpr int LDHB = H + 8;          // bf16 row stride of the split hidden activations
  constexpr int PHB = TM * LDHB;       // plane stride
  constexpr int CT1 = H / 16, NT1 = (CT1 + kTfWaves - 1) / kTfWaves;
  constexpr int CT2 = 3 * H / 16, NT2 = (CT2 + kTfWaves - 1) / kTfWaves;
  static_assert(CT1 % NT1 == 0 && CT2 % NT2 == 0, "tile split");
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const float* a_in = q.a;
  float* a_out = TAN ? q.da : q.a;
  float* h_out = TAN ? q.dh : q.h;
  float* w_out = TAN ? q.dw : q.w;
  // the tile's basis rows, zero past R and past the last pair
  for (int idx = threadIdx.x; idx < TM * RP; idx += kTfBlock) {
    const int m = idx / RP, k = idx - m * RP, p = pbase + m;
    e_lds[m * LDE + k] = (p < P && k < R) ? x[(size_t)p * R + k] : 0.f;
  }
  __syncthreads();
  if (wave < CT1 / NT1) {
    int cb[NT1];
    f4 acc[RT][NT1];
#pragma unroll
    for (int ct = 0; ct < NT1; ++ct) cb[ct] = (wave * NT1 + ct) * 16;
    zero_acc(acc);
    mma_tile<RT, NT1>(e_lds, LDE, q.w1p, RP, RP, cb, acc);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < NT1; ++ct) {
        const int c = cb[ct] + r;
        const float bias = TAN ? 0.f : q.b1[c];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = rt * 16 + 4 * g + i, p = pbase + m;
          const size_t o = (size_t)p * H + c;
          float a = acc[rt][ct][i] + bias, hv = 0.f;
          if (p < P) {
            hv = TAN ? silu_grad(a_in[o]) * a : silu(a);
            a_out[o] = a;
            h_out[o] = hv;
          }
          uint16_t hh, hm, hl;
          split3_bf16(hv, hh, hm, hl);
          h_bf[m * LDHB + c] = hh;
          h_bf[PHB + m * LDHB + c] = hm;
          h_bf[2 * PHB + m * LDHB + c] = hl;
        }
      }
  }
  __syncthreads();
  if (wave < CT2 / NT2) {
    int cb[NT2];
    f4 acc[RT][NT2];
#pragma unroll
    for (int ct = 0; ct < NT2; ++ct) cb[ct] = (wave * NT2 + ct) * 16;
    zero_acc(acc);
    mma_tile_x6<RT, NT2, H>(h_bf, LDHB, PHB, q.w2, H, 3 * H * H, cb, acc);
    float bias[NT2];
#pragma unroll
    for (int ct = 0; ct < NT2; ++ct) bias[ct] = TAN ? 0.f : q.b2[cb[ct] + r];
    // lane (r, g) holds rows rt*16 + 4g + i, columns cb[ct] + r
    float* out = w_out + (size_t)(pbase + 4 * g) * 3 * H + r;
    if (pbase + TM <= P) {   // full tile: no per-element bounds checks
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int ct = 0; ct < NT2; ++ct)
            out[(size_t)(rt * 16 + i) * 3 * H + cb[ct]] = acc[rt][ct][i] + bias[ct];
    } else {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (pbase + rt * 16 + 4 * g + i >= P) continue;
#pragma unroll
          for (int ct = 0; ct < NT2; ++ct)
            out[(size_t)(rt * 16 + i) * 3 * H + cb[ct]] = acc[rt][ct][i] + bias[ct];
        }
    }
  }
  __syncthreads();
}

// The filters of several blocks (blockIdx.y) in one launch, the forward from e, its
// tangent from de, or (WHAT = 2) both, the tangent of a tile behind its forward: the
// activations it needs are still in the L2, and a launch of all blocks leaves one
// last round of part-filled CUs instead of two per block (50000 pairs: 1.5 rounds of
// two blocks per CU).  64 molecules, three blocks at H = 128: 368 us in six launches,
// 287 us in one; two blocks at H = 32: 147 and 111 us.  The messages then read the
// filters from further away (70 -> 77 us a block).  Bound by the matrix cores and
// the stores by turns: 2 blocks per CU do not fully overlap a tile's phases.
template <int H, int TM, int WHAT>
__global__ __launch_bounds__(kTfBlock, 4) void train_filter_kernel(int P, int R, int RP,
                                                                   const float* e,
                                                                   const float* de,
                                                                   FilterRows rows) {
  __shared__ __align__(16) float e_lds[TM * (kTfMaxRbf + 4)];
  __shared__ __align__(16) uint16_t h_bf[3 * TM * (H + 8)];
  const FilterRow& q = rows.row[blockIdx.y];
  const int ntiles = (P + TM - 1) / TM;
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    if (WHAT != 1) train_filter_tile<H, TM, false>(tile * TM, P, R, RP, e, q, e_lds, h_bf);
    if (WHAT != 0) train_filter_tile<H, TM, true>(tile * TM, P, R, RP, de, q, e_lds, h_bf);
  }
}

// The filter adjoint kernel: 256-thread blocks (four per CU, so one block's
// staging overlaps the others' products), TM pairs per tile, the K = 3H sum
// of the product in three chunks of H columns staged in LDS (for TAN both gW
// and dgW).  The 4 waves split the CT = H/16 output column tiles (NTW each)
// and, when there are fewer than 4, the tile's row tiles (RG groups).
constexpr int kTaBlock = 256;

// mma_tile_k over one or (PAIR) two A operands (the adjoint and its tangent,
// same rows) with one B operand: each B fetch, PF slabs ahead, feeds both
// products.  hook() runs right after the first PF slabs' B fetches are
// issued: loads it issues then complete behind those slabs' MFMAs instead of
// delaying the first B wait (memory loads complete in issue order).
template <int RT, int NT, int K, bool PAIR, typename Hook, int PF = 2>
__device__ __forceinline__ void mma_tile_k_pair(const float* __restrict__ A0,
                                                const float* __restrict__ A1, int lda,
                                                const float* __restrict__ B, int ldb,
                                                const int (&cb)[NT], f4 (&acc0)[RT][NT],
                                                f4 (&acc1)[RT][NT], Hook&& hook) {
  static_assert(K % 16 == 0, "K must be a multiple of 16");
  constexpr int S = K / 16;
  const int lane = threadIdx.x & 63;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int aoff = r * lda + 4 * g;
  int boff[NT];
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) boff[ct] = (cb[ct] + r) * ldb + 4 * g;
  f4 b[PF + 1][NT];
#pragma unroll
  for (int q = 0; q < PF; ++q)
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
      if (q < S) b[q][ct] = *reinterpret_cast<const f4*>(B + boff[ct] + 16 * q);
  hook();
#pragma unroll
  for (int sl = 0; sl < S; ++sl) {
    if (sl + PF < S) {
#pragma unroll
      for (int ct = 0; ct < NT; ++ct)
        b[(sl + PF) % (PF + 1)][ct] = *reinterpret_cast<const f4*>(B + boff[ct] + 16 * (sl + PF));
    }
    f4 a0[RT], a1[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      a0[rt] = *reinterpret_cast<const f4*>(A0 + aoff + rt * 16 * lda + 16 * sl);
      if (PAIR) a1[rt] = *reinterpret_cast<const f4*>(A1 + aoff + rt * 16 * lda + 16 * sl);
    }
    const int cur = sl % (PF + 1);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) {
          acc0[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[rt][s], b[cur][ct][s],
                                                              acc0[rt][ct], 0, 0, 0);
          if (PAIR)
            acc1[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[rt][s], b[cur][ct][s],
                                                                acc1[rt][ct], 0, 0, 0);
        }
  }
}
constexpr int kTaWaves = kTaBlock / 64;
template <int H>
constexpr int kTaPairs = H >= 128 ? 32 : 64;

template <int H, int TM, bool TAN>
__global__ __launch_bounds__(kTaBlock, 4) void train_filter_adjoint_kernel(
    int P, const float* __restrict__ gw, const float* __restrict__ dgw,
    const float* __restrict__ w2t, const float* __restrict__ a, const float* __restrict__ da,
    float* __restrict__ ga, float* __restrict__ dga) {
  constexpr int KC = H;                 // columns per chunk
  constexpr int LDA = KC + 4;
  constexpr int CT = H / 16;
  constexpr int NTW = CT >= kTaWaves ? CT / kTaWaves : 1;
  constexpr int RG = CT >= kTaWaves ? 1 : kTaWaves / CT;
  constexpr int RTW = TM / 16 / RG;
  static_assert(NTW * kTaWaves == CT * RG && (TM / 16) % RG == 0, "wave split");
  constexpr int NSTAGE = TAN ? 2 : 1;
  __shared__ __align__(16) float a_lds[NSTAGE][TM * LDA];
  const int ntiles = (P + TM - 1) / TM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int cw = wave % (CT / NTW), rg = wave / (CT / NTW);
  int cb[NTW];
#pragma unroll
  for (int ct = 0; ct < NTW; ++ct) cb[ct] = (cw * NTW + ct) * 16;
  // Each thread's share of a chunk (NV float4s per operand) is fetched into
  // registers while the previous chunk's products run, then stored to LDS
  // (PRE, the tangent kernels; 136 -> 132 µs at H = 128 on 50,132 pairs).  The
  // tangent kernel at H = 64 would spill with those registers live across the
  // products, and the forward-only kernels (one operand, half the products)
  // gain nothing: those stage each chunk straight from memory.
  constexpr bool PRE = TAN && H != 64;
  constexpr int NV = TM * (KC / 4) / kTaBlock;
  static_assert(NV * kTaBlock == TM * (KC / 4), "chunk split");
  f4 st_g[NV], st_dg[TAN ? NV : 1];
  auto fetch = [&](int t, int ch) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int idx = threadIdx.x + v * kTaBlock;
      const int m = idx / (KC / 4), k4 = idx - m * (KC / 4), p = t * TM + m;
      const f4 zero = {0.f, 0.f, 0.f, 0.f};
      const bool on = t < ntiles && p < P;
      const size_t o = on ? (size_t)p * 3 * H + ch * KC + 4 * k4 : 0;
      st_g[v] = on ? *reinterpret_cast<const f4*>(gw + o) : zero;
      if (TAN) st_dg[v] = on ? *reinterpret_cast<const f4*>(dgw + o) : zero;
    }
  };
  if (PRE) fetch(blockIdx.x, 0);
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int pbase = tile * TM;
    f4 acc[RTW][NTW], dacc[RTW][NTW];
    zero_acc(acc);
    if (TAN) zero_acc(dacc);
#pragma unroll 1
    for (int ch = 0; ch < 3; ++ch) {
      __syncthreads();   // the previous chunk's products are done with the LDS
      if (PRE) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const int idx = threadIdx.x + v * kTaBlock;
          const int m = idx / (KC / 4), k4 = idx - m * (KC / 4);
          *reinterpret_cast<f4*>(&a_lds[0][m * LDA + 4 * k4]) = st_g[v];
          if (TAN) *reinterpret_cast<f4*>(&a_lds[NSTAGE - 1][m * LDA + 4 * k4]) = st_dg[v];
        }
      } else {
        for (int idx = threadIdx.x; idx < TM * (KC / 4); idx += kTaBlock) {
          const int m = idx / (KC / 4), k4 = idx - m * (KC / 4), p = pbase + m;
          const size_t o = (size_t)p * 3 * H + ch * KC + 4 * k4;
          const f4 zero = {0.f, 0.f, 0.f, 0.f};
          *reinterpret_cast<f4*>(&a_lds[0][m * LDA + 4 * k4]) =
              p < P ? *reinterpret_cast<const f4*>(gw + o) : zero;
          if (TAN)
            *reinterpret_cast<f4*>(&a_lds[NSTAGE - 1][m * LDA + 4 * k4]) =
                p < P ? *reinterpret_cast<const f4*>(dgw + o) : zero;
        }
      }
      __syncthreads();
      if (TAN) {
        // the next chunk (this tile's, or the next tile's first), in flight
        // during this chunk's products
        const int nt = ch < 2 ? tile : tile + gridDim.x, nch = ch < 2 ? ch + 1 : 0;
        mma_tile_k_pair<RTW, NTW, KC, true>(&a_lds[0][rg * RTW * 16 * LDA],
                                            &a_lds[NSTAGE - 1][rg * RTW * 16 * LDA], LDA,
                                            w2t + ch * KC, 3 * H, cb, acc, dacc,
                                            [&] {
                                              if (PRE) fetch(nt, nch);
                                            });
      } else {
        mma_tile_k<RTW, NTW, KC>(&a_lds[0][rg * RTW * 16 * LDA], LDA, w2t + ch * KC, 3 * H,
                                 cb, acc);
      }
    }
    // lane (r, g) holds rows (rg RTW + rt) 16 + 4g + i of columns cb[ct] + r
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = pbase + (rg * RTW + rt) * 16 + 4 * g + i;
        if (p >= P) continue;
#pragma unroll
        for (int ct = 0; ct < NTW; ++ct) {
          const size_t o = (size_t)p * H + cb[ct] + r;
          const float x = a[o];
          // s = sigmoid(x); 1 - s as 1 / (1 + exp(x)) (exact for large x)
          const float sg = 1.0f / (1.0f + expf(-x));
          const float sm = 1.0f / (1.0f + expf(x));
          const float d1 = sg * (1.0f + x * sm);
          const float gh = acc[rt][ct][i];
          ga[o] = gh * d1;
          if (TAN) {
            const float d2 = sg * sm * (2.0f + x * (sm - sg));
            dga[o] = dacc[rt][ct][i] * d1 + gh * d2 * da[o];
          }
        }
      }
  }
}

// ---------------------------------------------------------------------------
// The filter adjoint on the bf16 matrix cores (H >= 64): each K chunk of gW and
// dgW is split into three bf16 parts on its way to LDS and multiplied with the
// split W2^T (six part products, float32 accuracy).  Bound by the 10H floats per
// pair read and written and the splitting.  64 molecules, H = 128: 90 us per
// block against 117 us of the FP32 form above, which its products bound (121
// TFLOP/s).  At H = 32 that form's products are short enough (29 us).
// ---------------------------------------------------------------------------
template <int H, int TM, bool TAN>
__global__ __launch_bounds__(kTfBlock, 4) void train_filter_adjoint_x6_kernel(
    int P, const float* __restrict__ gw, const float* __restrict__ dgw,
    const uint16_t* __restrict__ w2t, const float* __restrict__ a, const float* __restrict__ da,
    float* __restrict__ ga, float* __restrict__ dga) {
  constexpr int LDA = H + 8, PA = TM * LDA, NS = TAN ? 2 : 1;
  constexpr int CT = H / 16, RG = kTfWaves / CT, RTW = TM / 16 / RG;
  constexpr int PB = 3 * H * H;                // plane stride of W2^T
  static_assert(RG * CT == kTfWaves && RTW * RG * 16 == TM, "wave split");
  constexpr int NV = TM * (H / 4) / kTfBlock;
  static_assert(NV * kTfBlock == TM * (H / 4), "chunk split");
  __shared__ __align__(16) uint16_t a_bf[NS][3 * PA];
  const int ntiles = (P + TM - 1) / TM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int cw = 16 * (wave % CT), rg = wave / CT;
  // a thread's share of the next chunk is in flight during the products
  f4 st[NS][NV];
  auto fetch = [&](int t, int ch) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int idx = threadIdx.x + v * kTfBlock;
      const int m = idx / (H / 4), c = 4 * (idx % (H / 4));
      const size_t o = (size_t)min(t * TM + m, P - 1) * 3 * H + ch * H + c;
      st[0][v] = *reinterpret_cast<const f4*>(gw + o);
      if (TAN) st[NS - 1][v] = *reinterpret_cast<const f4*>(dgw + o);
    }
  };
  if ((int)blockIdx.x < ntiles) fetch(blockIdx.x, 0);
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int pbase = tile * TM;
    f4 acc[RTW][1], dacc[RTW][1];
    zero_acc(acc);
    zero_acc(dacc);
#pragma unroll 1
    for (int ch = 0; ch < 3; ++ch) {
      __syncthreads();   // the products before are done with the LDS
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int j = 0; j < NS; ++j) {
          const int idx = threadIdx.x + v * kTfBlock;
          uint16_t* o = a_bf[j] + (idx / (H / 4)) * LDA + 4 * (idx % (H / 4));
          ushort4 h, md, l;
          split3_bf16(st[j][v][0], h.x, md.x, l.x);
          split3_bf16(st[j][v][1], h.y, md.y, l.y);
          split3_bf16(st[j][v][2], h.z, md.z, l.z);
          split3_bf16(st[j][v][3], h.w, md.w, l.w);
          *reinterpret_cast<ushort4*>(o) = h;
          *reinterpret_cast<ushort4*>(o + PA) = md;
          *reinterpret_cast<ushort4*>(o + 2 * PA) = l;
        }
      __syncthreads();
      const int nt = ch < 2 ? tile : tile + gridDim.x;
      if (nt < ntiles) fetch(nt, ch < 2 ? ch + 1 : 0);
      const uint16_t* B = w2t + (size_t)(cw + r) * 3 * H + ch * H + 8 * g;
      const int ao = (rg * RTW * 16 + r) * LDA + 8 * g;
#pragma unroll
      for (int k0 = 0; k0 < H; k0 += 32) {
        auto b8 = [&](const uint16_t* q) { return *reinterpret_cast<const bf8*>(q); };
        const bf8 bh = b8(B + k0), bm = b8(B + PB + k0), bl = b8(B + 2 * PB + k0);
        auto six = [&](const uint16_t* A, f4& c) {
          const bf8 ah = b8(A), am = b8(A + PA), al = b8(A + 2 * PA);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm, c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bh, c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bm, c, 0, 0, 0);
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
        };
#pragma unroll
        for (int rt = 0; rt < RTW; ++rt) {
          six(a_bf[0] + ao + rt * 16 * LDA + k0, acc[rt][0]);
          if (TAN) six(a_bf[NS - 1] + ao + rt * 16 * LDA + k0, dacc[rt][0]);
        }
      }
    }
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int p = pbase + (rg * RTW + rt) * 16 + 4 * g + i;
        if (p >= P) continue;
        const size_t o = (size_t)p * H + cw + r;
        const float x = a[o];
        // s = sigmoid(x); 1 - s as 1 / (1 + exp(x)) (exact for large x)
        const float sg = 1.0f / (1.0f + expf(-x)), sm = 1.0f / (1.0f + expf(x));
        const float d1 = sg * (1.0f + x * sm), gh = acc[rt][0][i];
        ga[o] = gh * d1;
        if (TAN) dga[o] = dacc[rt][0][i] * d1 + gh * (sg * sm * (2.0f + x * (sm - sg))) * da[o];
      }
  }
}

// What the pair kernels read of a filter MLP, remade for new weights in one
// launch: W1 [H][R] padded with zeros to RP columns, the bf16 planes of W2 [3H][H]
// and of its transpose, and the transpose.
__global__ void filter_planes_kernel(int H, int R, int RP, const float* __restrict__ w1,
                                     const float* __restrict__ w2, float* __restrict__ w1p,
                                     uint16_t* __restrict__ planes,
                                     uint16_t* __restrict__ planes_t, float* __restrict__ w2t) {
  const int n = 3 * H * H;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    uint16_t h, m, l;
    split3_bf16(w2[i], h, m, l);
    planes[i] = h;
    planes[n + i] = m;
    planes[2 * n + i] = l;
    const int t = (i % H) * 3 * H + i / H;
    planes_t[t] = h;
    planes_t[n + t] = m;
    planes_t[2 * n + t] = l;
    w2t[t] = w2[i];
    if (i < H * RP) w1p[i] = i % RP < R ? w1[(i / RP) * R + i % RP] : 0.f;
  }
}

__global__ void split_bf16x3_kernel(int64_t n, const float* __restrict__ src,
                                    uint16_t* __restrict__ dst) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    uint16_t h, m, l;
    split3_bf16(src[i], h, m, l);
    dst[i] = h;
    dst[n + i] = m;
    dst[2 * n + i] = l;
  }
}

template <int H, int WHAT>
hipError_t launch_train_filter(hipStream_t s, int P, int R, int RP, const float* e,
                               const float* de, int layers, const FilterRows& rows) {
  constexpr int TM = kTfPairs<H>;
  const int tiles = (P + TM - 1) / TM;
  // two blocks per CU fit the LDS; a few rounds of them
  const int grid = tiles < 2048 ? tiles : 2048;
  train_filter_kernel<H, TM, WHAT><<<dim3(grid, layers), kTfBlock, 0, s>>>(P, R, RP, e, de,
                                                                           rows);
  return hipGetLastError();
}

hipError_t dispatch_train_filter(hipStream_t s, int hidden, int what, int P, int R,
                                 const float* e, const float* de, int layers,
                                 const FilterRows& rows) {
  const int RP = R <= 16 ? 16 : 32;
  switch (hidden * 4 + what) {
#define MLFF_TF(HH, WW) \
  case HH * 4 + WW: return launch_train_filter<HH, WW>(s, P, R, RP, e, de, layers, rows);
#define MLFF_TF3(HH) MLFF_TF(HH, 0) MLFF_TF(HH, 1) MLFF_TF(HH, 2)
    MLFF_TF3(32)
    MLFF_TF3(64)
    MLFF_TF3(128)
#undef MLFF_TF3
#undef MLFF_TF
    default: return hipErrorInvalidValue;
  }
}

template <int H, bool TAN>
hipError_t launch_train_filter_adjoint(hipStream_t s, int P, const float* gw, const float* dgw,
                                       const float* w2t, const float* a, const float* da,
                                       float* ga, float* dga) {
  constexpr int TM = kTaPairs<H>;
  const int tiles = (P + TM - 1) / TM;
  // one tile per block (the dispatcher balances the CUs), strided past 8192
  const int grid = tiles < 8192 ? tiles : 8192;
  train_filter_adjoint_kernel<H, TM, TAN><<<grid, kTaBlock, 0, s>>>(P, gw, dgw, w2t, a, da, ga,
                                                                    dga);
  return hipGetLastError();
}

template <int H>
hipError_t launch_adjoint_x6(hipStream_t st, int P, const float* gw, const float* dgw,
                             const uint16_t* w2t, const float* a, const float* da, float* ga,
                             float* dga) {
  constexpr int TM = H >= 128 ? 32 : 64;
  const int tiles = (P + TM - 1) / TM, grid = tiles < 8192 ? tiles : 8192;
  if (dgw) train_filter_adjoint_x6_kernel<H, TM, true><<<grid, kTfBlock, 0, st>>>(P, gw, dgw, w2t, a, da, ga, dga);
  else train_filter_adjoint_x6_kernel<H, TM, false><<<grid, kTfBlock, 0, st>>>(P, gw, dgw, w2t, a, da, ga, dga);
  return hipGetLastError();
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace mlff

using namespace mlff;

extern "C" {

int mlff_filter_planes(void* stream, int hidden_dim, int R, const float* w1_dev,
                       const float* w2_dev, float* w1p_dev, uint16_t* planes_dev,
                       uint16_t* planes_t_dev, float* w2t_dev) {
  if (hidden_dim < 32 || hidden_dim > 4096 || R < 1 || R > kTfMaxRbf || !w1_dev || !w2_dev ||
      !w1p_dev || !planes_dev || !planes_t_dev || !w2t_dev) {
    set_error("mlff_filter_planes: need 32 <= hidden_dim <= 4096, 1 <= R <= %d and non-null "
              "buffers", kTfMaxRbf);
    return MLFF_ERR_INVALID;
  }
  const int n = 3 * hidden_dim * hidden_dim;
  filter_planes_kernel<<<(n + 255) / 256, 256, 0, static_cast<hipStream_t>(stream)>>>(
      hidden_dim, R, R <= 16 ? 16 : 32, w1_dev, w2_dev, w1p_dev, planes_dev, planes_t_dev,
      w2t_dev);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("mlff_filter_planes: %s", hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

int mlff_train_filter_adjoint_x6(void* stream, int hidden_dim, int n_pairs, const float* gw_dev,
                                 const float* dgw_dev, const uint16_t* planes_t_dev,
                                 const float* a_dev, const float* da_dev, float* ga_dev,
                                 float* dga_dev) {
  const char* nm = "mlff_train_filter_adjoint_x6";
  if (n_pairs < 0) { set_error("%s: negative size", nm); return MLFF_ERR_INVALID; }
  if (n_pairs == 0) return MLFF_OK;
  if (!gw_dev || !planes_t_dev || !a_dev || !ga_dev || (dgw_dev && (!da_dev || !dga_dev))) {
    set_error("%s: null pointer", nm);
    return MLFF_ERR_INVALID;
  }
  if (!aligned16(gw_dev) || !aligned16(dgw_dev) || !aligned16(planes_t_dev)) {
    set_error("%s: buffers must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (hidden_dim) {
    case 64: e = launch_adjoint_x6<64>(st, n_pairs, gw_dev, dgw_dev, planes_t_dev, a_dev, da_dev, ga_dev, dga_dev); break;
    case 128: e = launch_adjoint_x6<128>(st, n_pairs, gw_dev, dgw_dev, planes_t_dev, a_dev, da_dev, ga_dev, dga_dev); break;
    default:
      set_error("%s: hidden_dim %d not supported (64, 128)", nm, hidden_dim);
      return MLFF_ERR_UNSUPPORTED;
  }
  if (e != hipSuccess) {
    set_error("%s: %s", nm, hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

int mlff_split_bf16x3(void* stream, int64_t n, const float* src_dev, uint16_t* planes_dev) {
  if (n < 0 || (n > 0 && (!src_dev || !planes_dev))) {
    set_error("mlff_split_bf16x3: need n >= 0 and non-null buffers");
    return MLFF_ERR_INVALID;
  }
  if (n == 0) return MLFF_OK;
  const int64_t blocks = (n + 255) / 256;
  split_bf16x3_kernel<<<(unsigned)(blocks < 1024 ? blocks : 1024), 256, 0,
                        static_cast<hipStream_t>(stream)>>>(n, src_dev, planes_dev);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("mlff_split_bf16x3: %s", hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

int mlff_train_filter(void* stream, int tangent, int hidden, int n_pairs, int num_rbf,
                      const float* x_dev, const float* w1_padded_dev, const float* b1_dev,
                      const uint16_t* w2_planes_dev, const float* b2_dev, const float* a_dev,
                      float* a_out_dev, float* h_out_dev, float* w_out_dev) {
  const char* nm = "mlff_train_filter";
  if (hidden != 32 && hidden != 64 && hidden != 128) {
    set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden);
    return MLFF_ERR_UNSUPPORTED;
  }
  if (n_pairs < 0 || num_rbf < 1 || num_rbf > 32) {
    set_error("%s: need n_pairs >= 0 and 1 <= num_rbf <= 32", nm);
    return MLFF_ERR_INVALID;
  }
  const bool tan = tangent != 0;
  if (!x_dev || !w1_padded_dev || !w2_planes_dev || !a_out_dev || !h_out_dev || !w_out_dev ||
      (tan ? !a_dev : (!b1_dev || !b2_dev))) {
    set_error("%s: null buffer (the tangent needs a, the forward b1 and b2)", nm);
    return MLFF_ERR_INVALID;
  }
  if (!aligned16(w1_padded_dev) || !aligned16(w2_planes_dev)) {
    set_error("%s: padded W1 and the W2 planes must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_pairs == 0) return MLFF_OK;
  FilterRows rows = {};
  FilterRow& q = rows.row[0];
  q.w1p = w1_padded_dev; q.b1 = b1_dev; q.w2 = w2_planes_dev; q.b2 = b2_dev;
  if (tan) {
    q.a = const_cast<float*>(a_dev);   // read only
    q.da = a_out_dev; q.dh = h_out_dev; q.dw = w_out_dev;
  } else {
    q.a = a_out_dev; q.h = h_out_dev; q.w = w_out_dev;
  }
  hipError_t e = dispatch_train_filter(static_cast<hipStream_t>(stream), hidden, tan, n_pairs,
                                       num_rbf, x_dev, x_dev, 1, rows);
  if (e != hipSuccess) {
    set_error("%s: %s", nm, hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

int mlff_train_filters(void* stream, int hidden, int n_blocks, int n_pairs, int num_rbf,
                       const float* e_dev, const float* de_dev, const void* const* rows) {
  const char* nm = "mlff_train_filters";
  if (hidden != 32 && hidden != 64 && hidden != 128) {
    set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden);
    return MLFF_ERR_UNSUPPORTED;
  }
  if (n_blocks < 0 || n_blocks > kTfMaxLayers || n_pairs < 0 || num_rbf < 1 || num_rbf > 32) {
    set_error("%s: need 0 <= n_blocks <= %d, n_pairs >= 0 and 1 <= num_rbf <= 32", nm,
              kTfMaxLayers);
    return MLFF_ERR_INVALID;
  }
  if (n_blocks == 0) return MLFF_OK;
  const int what = de_dev ? 2 : 0;
  FilterRows t = {};
  bool null = !e_dev || !rows, odd = false;
  for (int k = 0; k < n_blocks && !null; ++k) {
    const void* const* r = rows + 10 * k;
    for (int i = 0; i < (what ? 10 : 7); ++i) null = null || !r[i];
    odd = odd || !aligned16(r[0]) || !aligned16(r[2]);
    auto out = [&](int i) { return static_cast<float*>(const_cast<void*>(r[i])); };
    t.row[k] = {static_cast<const float*>(r[0]), static_cast<const float*>(r[1]),
                static_cast<const uint16_t*>(r[2]), static_cast<const float*>(r[3]),
                out(4), out(5), out(6), out(7), out(8), out(9)};
  }
  if (null) {
    set_error("%s: null buffer", nm);
    return MLFF_ERR_INVALID;
  }
  if (odd) {
    set_error("%s: padded W1 and the W2 planes must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_pairs == 0) return MLFF_OK;
  hipError_t e = dispatch_train_filter(static_cast<hipStream_t>(stream), hidden, what, n_pairs,
                                       num_rbf, e_dev, de_dev, n_blocks, t);
  if (e != hipSuccess) {
    set_error("%s: %s", nm, hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

int mlff_train_filter_adjoint(void* stream, int tangent, int hidden, int n_pairs,
                              const float* gw_dev, const float* dgw_dev, const float* w2t_dev,
                              const float* a_dev, const float* da_dev, float* ga_out_dev,
                              float* dga_out_dev) {
  const char* nm = "mlff_train_filter_adjoint";
  if (hidden != 32 && hidden != 64 && hidden != 128) {
    set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden);
    return MLFF_ERR_UNSUPPORTED;
  }
  if (n_pairs < 0) {
    set_error("%s: need n_pairs >= 0", nm);
    return MLFF_ERR_INVALID;
  }
  const bool tan = tangent != 0;
  if (!gw_dev || !w2t_dev || !a_dev || !ga_out_dev ||
      (tan && (!dgw_dev || !da_dev || !dga_out_dev))) {
    set_error("%s: null buffer (the tangent needs dgw, da and dga_out)", nm);
    return MLFF_ERR_INVALID;
  }
  if (!aligned16(gw_dev) || !aligned16(w2t_dev) || (tan && !aligned16(dgw_dev))) {
    set_error("%s: gw, dgw and w2t must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_pairs == 0) return MLFF_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e;
  switch (hidden * 2 + (tan ? 1 : 0)) {
#define MLFF_TA(HH, TT)                                                                    \
  case HH * 2 + TT:                                                                        \
    e = launch_train_filter_adjoint<HH, TT>(s, n_pairs, gw_dev, dgw_dev, w2t_dev, a_dev,   \
                                            da_dev, ga_out_dev, dga_out_dev);              \
    break;
    MLFF_TA(32, false)
    MLFF_TA(32, true)
    MLFF_TA(64, false)
    MLFF_TA(64, true)
    MLFF_TA(128, false)
    MLFF_TA(128, true)
#undef MLFF_TA
    default:
      e = hipErrorInvalidValue;
  }
  if (e != hipSuccess) {
    set_error("%s: %s", nm, hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

}  // extern "C"
