// The update block of the training pass (PaiNNUpdate, student_model.py:430-470)
// with its tangent along a position direction, one launch per block and
// direction (the readout's kernels follow):
//   forward:  n = |v|_xyz, xin = (s, n), a = xin W1^T + b1, h = silu(a),
//             y = (ds, g1, g2) = h W2^T + b2, Mv = M v,
//             s' = s + ds, v' = v g1 + Mv g2, and/or the tangent of all of it;
//   adjoint:  gy = (gs, gv.v, gv.Mv), ga = silu'(a) (gy W2), gx = ga W1 = (gsx, gn),
//             gvg2 = gv g2, gs_m = gs + gsx, gv_m = gv g1 + M^T gvg2 + gn v / n,
//             and with it the tangent of all of it.
// What the weight gradients and the other pass read (xin, a, h, y, Mv, gy, ga,
// gvg2 and their tangents) goes to memory; the rest stays in the workgroup.
//
// A workgroup takes 16 atoms; the tangent's 16 rows share the tile, so every
// weight fetched feeds both.  Wave w owns the 16-channel column tile w of each
// H-wide plane, and the epilogues work on the accumulators in place.  Bound by
// the weights' way from L2 and the two products' latency (one round of the CUs
// up to 4096 atoms).  As separate kernels (elementwise, two library products,
// SiLU), 64 molecules of 2,400 atoms at H = 128 took 52 us per block forward and
// 36 us adjoint, 15 launches; the step's host side took longer than that where
// the batch is small.

#include <stdint.h>

#include <initializer_list>

#include "common.hpp"
#include "internal.hpp"

namespace mlff {
namespace {

constexpr int kTM = 16;

__device__ __forceinline__ f4 ld4(const float* p) { return *reinterpret_cast<const f4*>(p); }
__device__ __forceinline__ void st4(float* p, f4 v) { *reinterpret_cast<f4*>(p) = v; }
__device__ __forceinline__ float sigmoid(float a) { return 1.0f / (1.0f + expf(-a)); }
// silu'(a) and silu''(a) from s = sigmoid(a) and 1 - s = sigmoid(-a)
__device__ __forceinline__ float silu_d1(float a, float s, float q) { return s * fma_(a, q, 1.0f); }
__device__ __forceinline__ float silu_d2(float a, float s, float q) {
  return s * q * fma_(a, q - s, 2.0f);
}

// mma_tile_k4 with B given as [K][columns] (the transpose of a Linear's weight)
template <int RT, int NT, int K>
__device__ __forceinline__ void mma_tile_t(const float* __restrict__ A, int lda,
                                           const float* __restrict__ B, int ldb,
                                           const int (&cb)[NT], f4 (&acc)[RT][NT]) {
  constexpr int S = K / 16, PF = 2;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const float* arow = A + r * lda + 4 * g;
  Acc4<RT, NT> sum;
  f4 b[PF + 1][NT];
  auto load = [&](int sl) {
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        b[sl % (PF + 1)][ct][s] = B[(16 * sl + 4 * g + s) * ldb + cb[ct] + r];
  };
#pragma unroll
  for (int q = 0; q < PF && q < S; ++q) load(q);
#pragma unroll
  for (int sl = 0; sl < S; ++sl) {
    if (sl + PF < S) load(sl + PF);
    f4 a[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) a[rt] = ld4(arow + rt * 16 * lda + 16 * sl);
    sum.slab(a, b[sl % (PF + 1)]);
  }
  sum.add_to(acc);
}

struct FwdArgs {
  int n;
  const float *s, *v, *ds, *dv;              // block inputs (message outputs), tangents
  const float *w1, *b1, *w2, *b2, *mix;
  float *xin, *a, *h, *y, *mv, *s_out, *v_out;
  float *dxin, *da, *dh, *dy, *dmv, *ds_out, *dv_out;
};

// PRIM: the primal outputs are computed (else read); TAN: the tangent's are
template <int H, bool PRIM, bool TAN>
__global__ __launch_bounds__(4 * H) void train_update_fwd_kernel(FwdArgs p) {
  constexpr int RT = PRIM && TAN ? 2 : 1, TR = PRIM ? kTM : 0;   // first tangent row
  constexpr int LDX = 2 * H + 4, LDH = H + 4;
  __shared__ __align__(16) float x_lds[kTM * RT * LDX];
  __shared__ __align__(16) float h_lds[kTM * RT * LDH];
  const int base = blockIdx.x * kTM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  {
    const int m = threadIdx.x / (H / 4), c = 4 * (threadIdx.x % (H / 4));
    const bool in = base + m < p.n;
    const size_t i = min(base + m, p.n - 1);
    const float* vr = p.v + i * 3 * H + c;
    const f4 v0 = ld4(vr), v1 = ld4(vr + H), v2 = ld4(vr + 2 * H);
    f4 nrm;
    if (PRIM) {
      const f4 sv = ld4(p.s + i * H + c);
      const f4 sq = v0 * v0 + v1 * v1 + v2 * v2;
#pragma unroll
      for (int k = 0; k < 4; ++k) nrm[k] = sqrtf(sq[k]);
      st4(x_lds + m * LDX + c, sv);
      st4(x_lds + m * LDX + H + c, nrm);
      if (in) {
        st4(p.xin + i * 2 * H + c, sv);
        st4(p.xin + i * 2 * H + H + c, nrm);
      }
    } else {
      nrm = ld4(p.xin + i * 2 * H + H + c);
    }
    if (TAN) {
      const float* dr = p.dv + i * 3 * H + c;
      const f4 dsv = ld4(p.ds + i * H + c);
      const f4 dot = v0 * ld4(dr) + v1 * ld4(dr + H) + v2 * ld4(dr + 2 * H);
      f4 dn;
#pragma unroll
      for (int k = 0; k < 4; ++k) dn[k] = nrm[k] > 0.f ? dot[k] / nrm[k] : 0.f;
      st4(x_lds + (TR + m) * LDX + c, dsv);
      st4(x_lds + (TR + m) * LDX + H + c, dn);
      if (in) {
        st4(p.dxin + i * 2 * H + c, dsv);
        st4(p.dxin + i * 2 * H + H + c, dn);
      }
    }
  }
  __syncthreads();
  const int c = 16 * wave + r;      // the lane's channel
  {
    const int cb[1] = {16 * wave};
    f4 acc[RT][1];
    float av[4];
    if (!PRIM)
#pragma unroll
      for (int k = 0; k < 4; ++k) av[k] = p.a[(size_t)min(base + 4 * g + k, p.n - 1) * H + c];
    zero_acc(acc);
    mma_tile_k4<RT, 1, 2 * H>(x_lds, LDX, p.w1, 2 * H, cb, acc);
    const float b1 = PRIM ? p.b1[c] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int m = 4 * g + k;
      const bool in = base + m < p.n;
      const size_t o = (size_t)(base + m) * H + c;
      const float a = PRIM ? acc[0][0][k] + b1 : av[k];
      const float s = sigmoid(a);
      if (PRIM) {
        const float h = a * s;
        h_lds[m * LDH + c] = h;
        if (in) { p.a[o] = a; p.h[o] = h; }
      }
      if (TAN) {
        const float da = acc[RT - 1][0][k], dh = silu_d1(a, s, sigmoid(-a)) * da;
        h_lds[(TR + m) * LDH + c] = dh;
        if (in) { p.da[o] = da; p.dh[o] = dh; }
      }
    }
  }
  __syncthreads();
  float mx[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) mx[k] = p.mix[k];
  const int cb[3] = {16 * wave, H + 16 * wave, 2 * H + 16 * wave};
  float vv[4][3], dd[4][3], g1[4], g2[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const size_t i = min(base + 4 * g + k, p.n - 1);
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      vv[k][x] = p.v[(i * 3 + x) * H + c];
      if (TAN) dd[k][x] = p.dv[(i * 3 + x) * H + c];
    }
    if (!PRIM) {
      g1[k] = p.y[i * 3 * H + H + c];
      g2[k] = p.y[i * 3 * H + 2 * H + c];
    }
  }
  float bias[3] = {0.f, 0.f, 0.f};
  if (PRIM)
#pragma unroll
    for (int q = 0; q < 3; ++q) bias[q] = p.b2[q * H + c];
  f4 acc[RT][3];
  zero_acc(acc);
  mma_tile_k4<RT, 3, H>(h_lds, LDH, p.w2, H, cb, acc);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int m = 4 * g + k;
    if (base + m >= p.n) continue;
    const size_t i = base + m;
    float mv[3];
#pragma unroll
    for (int x = 0; x < 3; ++x)
      mv[x] = mx[3 * x] * vv[k][0] + mx[3 * x + 1] * vv[k][1] + mx[3 * x + 2] * vv[k][2];
    if (PRIM) {
      const float y0 = acc[0][0][k] + bias[0];
      g1[k] = acc[0][1][k] + bias[1];
      g2[k] = acc[0][2][k] + bias[2];
      float* yr = p.y + i * 3 * H + c;
      yr[0] = y0;
      yr[H] = g1[k];
      yr[2 * H] = g2[k];
      p.s_out[i * H + c] = x_lds[m * LDX + c] + y0;
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        p.mv[(i * 3 + x) * H + c] = mv[x];
        p.v_out[(i * 3 + x) * H + c] = vv[k][x] * g1[k] + mv[x] * g2[k];
      }
    }
    if (TAN) {
      const float y0 = acc[RT - 1][0][k], dg1 = acc[RT - 1][1][k], dg2 = acc[RT - 1][2][k];
      float* yr = p.dy + i * 3 * H + c;
      yr[0] = y0;
      yr[H] = dg1;
      yr[2 * H] = dg2;
      p.ds_out[i * H + c] = x_lds[(TR + m) * LDX + c] + y0;
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        const float dmv =
            mx[3 * x] * dd[k][0] + mx[3 * x + 1] * dd[k][1] + mx[3 * x + 2] * dd[k][2];
        p.dmv[(i * 3 + x) * H + c] = dmv;
        p.dv_out[(i * 3 + x) * H + c] =
            dd[k][x] * g1[k] + vv[k][x] * dg1 + dmv * g2[k] + mv[x] * dg2;
      }
    }
  }
}

struct BwdArgs {
  int n;
  const float *gs, *gv, *dgs, *dgv;                    // output gradients, tangents
  const float *v, *mv, *y, *a, *xin;                   // the forward's
  const float *dv, *dmv, *dy, *da, *dxin;
  const float *w1, *w2, *mix;
  float *gy, *ga, *gs_out, *gv_out, *gvg2;
  float *dgy, *dga, *dgs_out, *dgv_out, *dgvg2;
};

template <int H, bool TAN>
__global__ __launch_bounds__(4 * H) void train_update_bwd_kernel(BwdArgs p) {
  constexpr int RT = TAN ? 2 : 1;
  constexpr int LDY = 3 * H + 4, LDA = H + 4;
  __shared__ __align__(16) float y_lds[kTM * RT * LDY];
  __shared__ __align__(16) float a_lds[kTM * RT * LDA];
  const int base = blockIdx.x * kTM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  {
    const int m = threadIdx.x / (H / 4), c = 4 * (threadIdx.x % (H / 4));
    const bool in = base + m < p.n;
    const size_t i = min(base + m, p.n - 1);
    f4 q[3], vv[3], mm[3], dq[3], dd[3], dm[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const size_t o = (i * 3 + x) * H + c;
      q[x] = ld4(p.gv + o);
      vv[x] = ld4(p.v + o);
      mm[x] = ld4(p.mv + o);
      if (TAN) {
        dq[x] = ld4(p.dgv + o);
        dd[x] = ld4(p.dv + o);
        dm[x] = ld4(p.dmv + o);
      }
    }
    auto put = [&](int row, float* out, f4 y0, f4 y1, f4 y2) {
      float* o = y_lds + row * LDY + c;
      st4(o, y0);
      st4(o + H, y1);
      st4(o + 2 * H, y2);
      if (in) {
        float* w = out + i * 3 * H + c;
        st4(w, y0);
        st4(w + H, y1);
        st4(w + 2 * H, y2);
      }
    };
    put(m, p.gy, ld4(p.gs + i * H + c), q[0] * vv[0] + q[1] * vv[1] + q[2] * vv[2],
        q[0] * mm[0] + q[1] * mm[1] + q[2] * mm[2]);
    if (TAN)
      put(kTM + m, p.dgy, ld4(p.dgs + i * H + c),
          (dq[0] * vv[0] + q[0] * dd[0]) + (dq[1] * vv[1] + q[1] * dd[1]) +
              (dq[2] * vv[2] + q[2] * dd[2]),
          (dq[0] * mm[0] + q[0] * dm[0]) + (dq[1] * mm[1] + q[1] * dm[1]) +
              (dq[2] * mm[2] + q[2] * dm[2]));
  }
  __syncthreads();
  const int c = 16 * wave + r;      // the lane's channel
  {
    const int cb[1] = {16 * wave};
    float av[4], dav[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const size_t o = (size_t)min(base + 4 * g + k, p.n - 1) * H + c;
      av[k] = p.a[o];
      if (TAN) dav[k] = p.da[o];
    }
    f4 acc[RT][1];
    zero_acc(acc);
    mma_tile_t<RT, 1, 3 * H>(y_lds, LDY, p.w2, H, cb, acc);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int m = 4 * g + k;
      const bool in = base + m < p.n;
      const size_t o = (size_t)(base + m) * H + c;
      const float s = sigmoid(av[k]), q = sigmoid(-av[k]);
      const float d1 = silu_d1(av[k], s, q);
      const float gh = acc[0][0][k], ga = gh * d1;
      a_lds[m * LDA + c] = ga;
      if (in) p.ga[o] = ga;
      if (TAN) {
        const float dga = fma_(acc[RT - 1][0][k], d1, gh * silu_d2(av[k], s, q) * dav[k]);
        a_lds[(kTM + m) * LDA + c] = dga;
        if (in) p.dga[o] = dga;
      }
    }
  }
  __syncthreads();
  float mx[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) mx[k] = p.mix[k];
  const int cb[2] = {16 * wave, H + 16 * wave};
  // the epilogue's operands are requested before the product
  float y1[4], y2[4], nm[4], qv[4][3], vr[4][3], e1[4], e2[4], en[4], dqv[4][3], dvr[4][3];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const size_t i = min(base + 4 * g + k, p.n - 1);
    y1[k] = p.y[i * 3 * H + H + c];
    y2[k] = p.y[i * 3 * H + 2 * H + c];
    nm[k] = p.xin[i * 2 * H + H + c];
    if (TAN) {
      e1[k] = p.dy[i * 3 * H + H + c];
      e2[k] = p.dy[i * 3 * H + 2 * H + c];
      en[k] = p.dxin[i * 2 * H + H + c];
    }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const size_t o = (i * 3 + x) * H + c;
      qv[k][x] = p.gv[o];
      vr[k][x] = p.v[o];
      if (TAN) {
        dqv[k][x] = p.dgv[o];
        dvr[k][x] = p.dv[o];
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  f4 acc[RT][2];
  zero_acc(acc);
  mma_tile_t<RT, 2, H>(a_lds, LDA, p.w1, 2 * H, cb, acc);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int m = 4 * g + k;
    if (base + m >= p.n) continue;
    const size_t i = base + m;
    const float g1 = y1[k], g2 = y2[k];
    const float nrm = nm[k], inv = nrm > 0.f ? 1.0f / nrm : 0.f;
    const float gn = acc[0][1][k];
    const float(&q)[3] = qv[k];
    const float(&vv)[3] = vr[k];
    float qg[3], unit[3];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      qg[x] = q[x] * g2;
      unit[x] = vv[x] * inv;
      p.gvg2[(i * 3 + x) * H + c] = qg[x];
    }
    p.gs_out[i * H + c] = y_lds[m * LDY + c] + acc[0][0][k];
#pragma unroll
    for (int x = 0; x < 3; ++x)
      p.gv_out[(i * 3 + x) * H + c] =
          q[x] * g1 + (mx[x] * qg[0] + mx[3 + x] * qg[1] + mx[6 + x] * qg[2]) + gn * unit[x];
    if (TAN) {
      const float dg1 = e1[k], dg2 = e2[k], dninv2 = en[k] * inv * inv;
      const float dgn = acc[RT - 1][1][k];
      const float(&dq)[3] = dqv[k];
      float dqg[3], dunit[3];
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        dqg[x] = dq[x] * g2 + q[x] * dg2;
        dunit[x] = dvr[k][x] * inv - vv[x] * dninv2;
        p.dgvg2[(i * 3 + x) * H + c] = dqg[x];
      }
      p.dgs_out[i * H + c] = y_lds[(kTM + m) * LDY + c] + acc[RT - 1][0][k];
#pragma unroll
      for (int x = 0; x < 3; ++x)
        p.dgv_out[(i * 3 + x) * H + c] =
            dq[x] * g1 + q[x] * dg1 + (mx[x] * dqg[0] + mx[3 + x] * dqg[1] + mx[6 + x] * dqg[2]) +
            dgn * unit[x] + gn * dunit[x];
    }
  }
}

// ---------------------------------------------------------------------------
// The readout (student_model.py:606-618: H -> H/2 -> H/4 -> 1, SiLU between) of
// the training pass, 16 atoms per workgroup:
//   forward: r1 = s W1^T + b1, h3 = silu(r1), r2 = h3 W2^T + b2, h4 = silu(r2),
//            eps = h4 W3^T + b3, and/or the tangent;
//   adjoint: gr2 = g W3 silu'(r2), gr1 = (gr2 W2) silu'(r1), gs = gr1 W1 with the
//            atom's seed g, and with it the tangent.
// The products are a few thousand multiplications per atom, on the vector units:
// a thread takes one output column for four (two) of the tile's atoms and reads
// its weights once for them, its inputs from LDS.  Bound by its launches; as
// library products and elementwise kernels it was ten launches forward with the
// tangent, and eight adjoint.
// ---------------------------------------------------------------------------
constexpr int kReadBlock = 256;

struct ReadArgs {
  int n;
  const float *s, *ds, *w1, *b1, *w2, *b2, *w3, *b3;
  float *r1, *h3, *r2, *h4, *eps;
  float *dr1, *dh3, *dr2, *dh4;
};

// out[j][q] = sum_k x_j[q][k] w(k) for four atoms q of NX tiles x_j, four partial
// sums each; w(k) gives the weights k ... k + 3
template <int K, int LD, int NX, class W>
__device__ __forceinline__ void dot_rows(const float* const (&x)[NX], W w, float (&out)[NX][4]) {
  f4 acc[NX][4];
#pragma unroll
  for (int j = 0; j < NX; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[j][q] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = 0; k < K; k += 4) {
    const f4 wk = w(k);
#pragma unroll
    for (int j = 0; j < NX; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[j][q] = fma_(ld4(x[j] + q * LD + k), wk, acc[j][q]);
  }
#pragma unroll
  for (int j = 0; j < NX; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      out[j][q] = (acc[j][q][0] + acc[j][q][1]) + (acc[j][q][2] + acc[j][q][3]);
}
__device__ __forceinline__ auto row_of(const float* w) {
  return [=](int k) { return ld4(w + k); };
}
// the same with a column of a matrix of ldw columns; a pass per tile: with two
// tiles on one pass fewer loads are in flight (19 against 14 us)
template <int K, int LD>
__device__ __forceinline__ void dot_column(const float* x, const float* w, int ldw,
                                           float (&out)[4]) {
  const float* const rows[1] = {x};
  float v[1][4];
  dot_rows<K, LD, 1>(rows, [=](int k) {
    return f4{w[(size_t)k * ldw], w[(size_t)(k + 1) * ldw], w[(size_t)(k + 2) * ldw],
              w[(size_t)(k + 3) * ldw]};
  }, v);
#pragma unroll
  for (int q = 0; q < 4; ++q) out[q] = v[0][q];
}

template <int H, bool PRIM, bool TAN>
__global__ __launch_bounds__(kReadBlock) void train_readout_fwd_kernel(ReadArgs p) {
  constexpr int H2 = H / 2, H4 = H / 4, LX = H + 4, L2 = H2 + 4, L4 = H4 + 4;
  __shared__ __align__(16) float x[2][kTM * LX];
  __shared__ __align__(16) float h3[2][kTM * L2];
  __shared__ __align__(16) float h4[kTM * L4];
  __shared__ __align__(16) float w1[H2 * LX];    // rows a lane apart are far apart in memory
  constexpr int NX = PRIM && TAN ? 2 : 1, X0 = PRIM ? 0 : 1;
  const int base = blockIdx.x * kTM;
  for (int it = threadIdx.x; it < H2 * H / 4; it += kReadBlock) {
    const int c = it / (H / 4), k = 4 * (it % (H / 4));
    st4(w1 + c * LX + k, ld4(p.w1 + (size_t)c * H + k));
  }
  for (int it = threadIdx.x; it < kTM * H / 4; it += kReadBlock) {
    const int m = it / (H / 4), c = 4 * (it % (H / 4));
    const size_t o = (size_t)min(base + m, p.n - 1) * H + c;
    if (PRIM) st4(x[0] + m * LX + c, ld4(p.s + o));
    if (TAN) st4(x[1] + m * LX + c, ld4(p.ds + o));
  }
  __syncthreads();
  // items of four consecutive atoms and one column
  for (int it = threadIdx.x; it < H2 * kTM / 4; it += kReadBlock) {
    const int c = it % H2, m0 = 4 * (it / H2);
    const float* in_rows[NX];
    float v[NX][4];
#pragma unroll
    for (int j = 0; j < NX; ++j) in_rows[j] = x[X0 + j] + m0 * LX;
    dot_rows<H, LX, NX>(in_rows, row_of(w1 + c * LX), v);
    const float(&r)[4] = v[0];
    const float(&d)[4] = v[NX - 1];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = m0 + q;
      const bool in = base + m < p.n;
      const size_t o = (size_t)min(base + m, p.n - 1) * H2 + c;
      const float a = PRIM ? r[q] + p.b1[c] : p.r1[o], s = sigmoid(a);
      if (PRIM) {
        h3[0][m * L2 + c] = a * s;
        if (in) { p.r1[o] = a; p.h3[o] = a * s; }
      }
      if (TAN) {
        const float dh = silu_d1(a, s, sigmoid(-a)) * d[q];
        h3[1][m * L2 + c] = dh;
        if (in) { p.dr1[o] = d[q]; p.dh3[o] = dh; }
      }
    }
  }
  __syncthreads();
  for (int it = threadIdx.x; it < H4 * kTM / 4; it += kReadBlock) {
    const int c = it % H4, m0 = 4 * (it / H4);
    const float* in_rows[NX];
    float v[NX][4];
#pragma unroll
    for (int j = 0; j < NX; ++j) in_rows[j] = h3[X0 + j] + m0 * L2;
    dot_rows<H2, L2, NX>(in_rows, row_of(p.w2 + (size_t)c * H2), v);
    const float(&r)[4] = v[0];
    const float(&d)[4] = v[NX - 1];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int m = m0 + q;
      const bool in = base + m < p.n;
      const size_t o = (size_t)min(base + m, p.n - 1) * H4 + c;
      const float a = PRIM ? r[q] + p.b2[c] : p.r2[o], s = sigmoid(a);
      if (PRIM) {
        h4[m * L4 + c] = a * s;
        if (in) { p.r2[o] = a; p.h4[o] = a * s; }
      }
      if (TAN && in) {
        p.dr2[o] = d[q];
        p.dh4[o] = silu_d1(a, s, sigmoid(-a)) * d[q];
      }
    }
  }
  if constexpr (PRIM) {
    __syncthreads();
    if (threadIdx.x < kTM / 4) {
      const int m0 = 4 * threadIdx.x;
      const float* in_rows[1] = {h4 + m0 * L4};
      float e[1][4];
      dot_rows<H4, L4, 1>(in_rows, row_of(p.w3), e);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (base + m0 + q < p.n) p.eps[base + m0 + q] = e[0][q] + p.b3[0];
    }
  }
}

struct ReadAdjArgs {
  int n;
  const float *seed;                 // g of each structure
  const int64_t* batch;              // structure of each atom
  const float *r1, *r2, *dr1, *dr2, *w1, *w2, *w3;
  float *g4, *gr2, *gr1, *gs;        // g4 [n][4]: (g, 0, 0, 0)
  float *dgr2, *dgr1, *dgs;
};

template <int H, bool TAN>
__global__ __launch_bounds__(kReadBlock) void train_readout_bwd_kernel(ReadAdjArgs p) {
  constexpr int H2 = H / 2, H4 = H / 4, L2 = H2 + 4, L4 = H4 + 4;
  __shared__ __align__(16) float g2[2][kTM * L4];
  __shared__ __align__(16) float g1[2][kTM * L2];
  const int base = blockIdx.x * kTM;
  for (int it = threadIdx.x; it < kTM * H4; it += kReadBlock) {
    const int m = it / H4, c = it % H4;
    const bool in = base + m < p.n;
    const size_t i = min(base + m, p.n - 1), o = i * H4 + c;
    const float g = p.seed[p.batch[i]], gh = g * p.w3[c];
    const float a = p.r2[o], s = sigmoid(a), q = sigmoid(-a);
    const float v = gh * silu_d1(a, s, q);
    g2[0][m * L4 + c] = v;
    if (in) p.gr2[o] = v;
    if (TAN) {
      const float d = gh * silu_d2(a, s, q) * p.dr2[o];
      g2[1][m * L4 + c] = d;
      if (in) p.dgr2[o] = d;
    }
    if (in && c < 4) p.g4[4 * i + c] = c == 0 ? g : 0.f;
  }
  __syncthreads();
  for (int it = threadIdx.x; it < H2 * kTM / 4; it += kReadBlock) {
    const int c = it % H2, m0 = 4 * (it / H2);
    float v[4], d[4];
    dot_column<H4, L4>(g2[0] + m0 * L4, p.w2 + c, H2, v);
    if (TAN) dot_column<H4, L4>(g2[1] + m0 * L4, p.w2 + c, H2, d);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int m = m0 + k;
      const bool in = base + m < p.n;
      const size_t o = (size_t)min(base + m, p.n - 1) * H2 + c;
      const float a = p.r1[o], s = sigmoid(a), q = sigmoid(-a), d1 = silu_d1(a, s, q);
      const float t = v[k] * d1;
      g1[0][m * L2 + c] = t;
      if (in) p.gr1[o] = t;
      if (TAN) {
        const float u = fma_(d[k], d1, v[k] * silu_d2(a, s, q) * p.dr1[o]);
        g1[1][m * L2 + c] = u;
        if (in) p.dgr1[o] = u;
      }
    }
  }
  __syncthreads();
  for (int it = threadIdx.x; it < H * kTM / 4; it += kReadBlock) {
    const int c = it % H, m0 = 4 * (it / H);
    float v[4], d[4];
    dot_column<H2, L2>(g1[0] + m0 * L2, p.w1 + c, H, v);
    if (TAN) dot_column<H2, L2>(g1[1] + m0 * L2, p.w1 + c, H, d);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (base + m0 + k < p.n) {
        const size_t o = (size_t)(base + m0 + k) * H + c;
        p.gs[o] = v[k];
        if (TAN) p.dgs[o] = d[k];
      }
  }
}

bool aligned(std::initializer_list<const void*> ps) {
  for (const void* q : ps)
    if (reinterpret_cast<uintptr_t>(q) & 15) return false;
  return true;
}
bool present(std::initializer_list<const void*> ps) {
  for (const void* q : ps)
    if (!q) return false;
  return true;
}

int finish(const char* name) {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return MLFF_OK;
  set_error("%s: %s", name, hipGetErrorString(e));
  return MLFF_ERR_HIP;
}

}  // namespace
}  // namespace mlff

using namespace mlff;

extern "C" {

int mlff_train_update(void* stream, int parts, int n_atoms, int hidden_dim, const float* s_dev,
                      const float* v_dev, const float* ds_dev, const float* dv_dev,
                      const float* w1_dev, const float* b1_dev, const float* w2_dev,
                      const float* b2_dev, const float* mix_dev, float* xin_dev, float* a_dev,
                      float* h_dev, float* y_dev, float* mv_dev, float* s_out_dev,
                      float* v_out_dev, float* dxin_dev, float* da_dev, float* dh_dev,
                      float* dy_dev, float* dmv_dev, float* ds_out_dev, float* dv_out_dev) {
  const char* nm = "mlff_train_update";
  const bool prim = parts & 1, tan = parts & 2;
  if (n_atoms < 0 || parts < 1 || parts > 3) {
    set_error("%s: invalid size or parts", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_atoms == 0) return MLFF_OK;
  if (!present({v_dev, w1_dev, w2_dev, mix_dev, xin_dev, a_dev, y_dev}) ||
      (prim && !present({s_dev, b1_dev, b2_dev, h_dev, mv_dev, s_out_dev, v_out_dev})) ||
      (tan && !present({ds_dev, dv_dev, dxin_dev, da_dev, dh_dev, dy_dev, dmv_dev, ds_out_dev,
                        dv_out_dev}))) {
    set_error("%s: null buffer", nm);
    return MLFF_ERR_INVALID;
  }
  if (!aligned({s_dev, v_dev, ds_dev, dv_dev, w1_dev, w2_dev, xin_dev, dxin_dev})) {
    set_error("%s: buffers must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  const FwdArgs p = {n_atoms, s_dev, v_dev, ds_dev, dv_dev, w1_dev, b1_dev, w2_dev, b2_dev,
                     mix_dev, xin_dev, a_dev, h_dev, y_dev, mv_dev, s_out_dev, v_out_dev,
                     dxin_dev, da_dev, dh_dev, dy_dev, dmv_dev, ds_out_dev, dv_out_dev};
  auto run = [&](auto kernel) {
    kernel<<<(n_atoms + kTM - 1) / kTM, 4 * hidden_dim, 0, static_cast<hipStream_t>(stream)>>>(p);
    return finish(nm);
  };
#define MLFF_UPD(H)                                                   \
  case H:                                                             \
    return prim && tan ? run(train_update_fwd_kernel<H, true, true>)  \
           : prim      ? run(train_update_fwd_kernel<H, true, false>) \
                       : run(train_update_fwd_kernel<H, false, true>);
  switch (hidden_dim) {
    MLFF_UPD(32)
    MLFF_UPD(64)
    MLFF_UPD(128)
  }
#undef MLFF_UPD
  set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden_dim);
  return MLFF_ERR_UNSUPPORTED;
}

int mlff_train_update_adjoint(void* stream, int n_atoms, int hidden_dim, const float* gs_dev,
                              const float* gv_dev, const float* dgs_dev, const float* dgv_dev,
                              const float* v_dev, const float* mv_dev, const float* y_dev,
                              const float* a_dev, const float* xin_dev, const float* dv_dev,
                              const float* dmv_dev, const float* dy_dev, const float* da_dev,
                              const float* dxin_dev, const float* w1_dev, const float* w2_dev,
                              const float* mix_dev, float* gy_dev, float* ga_dev,
                              float* gs_out_dev, float* gv_out_dev, float* gvg2_dev,
                              float* dgy_dev, float* dga_dev, float* dgs_out_dev,
                              float* dgv_out_dev, float* dgvg2_dev) {
  const char* nm = "mlff_train_update_adjoint";
  const bool tan = dgs_dev != nullptr;
  if (n_atoms < 0) {
    set_error("%s: invalid size", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_atoms == 0) return MLFF_OK;
  if (!present({gs_dev, gv_dev, v_dev, mv_dev, y_dev, a_dev, xin_dev, w1_dev, w2_dev, mix_dev,
                gy_dev, ga_dev, gs_out_dev, gv_out_dev, gvg2_dev}) ||
      (tan && !present({dgv_dev, dv_dev, dmv_dev, dy_dev, da_dev, dxin_dev, dgy_dev, dga_dev,
                        dgs_out_dev, dgv_out_dev, dgvg2_dev}))) {
    set_error("%s: null buffer", nm);
    return MLFF_ERR_INVALID;
  }
  if (!aligned({gs_dev, gv_dev, dgs_dev, dgv_dev, v_dev, mv_dev, dv_dev, dmv_dev, gy_dev,
                dgy_dev})) {
    set_error("%s: buffers must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  const BwdArgs p = {n_atoms, gs_dev, gv_dev, dgs_dev, dgv_dev, v_dev, mv_dev, y_dev, a_dev,
                     xin_dev, dv_dev, dmv_dev, dy_dev, da_dev, dxin_dev, w1_dev, w2_dev, mix_dev,
                     gy_dev, ga_dev, gs_out_dev, gv_out_dev, gvg2_dev, dgy_dev, dga_dev,
                     dgs_out_dev, dgv_out_dev, dgvg2_dev};
  auto run = [&](auto kernel) {
    kernel<<<(n_atoms + kTM - 1) / kTM, 4 * hidden_dim, 0, static_cast<hipStream_t>(stream)>>>(p);
    return finish(nm);
  };
  switch (hidden_dim) {
    case 32: return tan ? run(train_update_bwd_kernel<32, true>) : run(train_update_bwd_kernel<32, false>);
    case 64: return tan ? run(train_update_bwd_kernel<64, true>) : run(train_update_bwd_kernel<64, false>);
    case 128: return tan ? run(train_update_bwd_kernel<128, true>) : run(train_update_bwd_kernel<128, false>);
  }
  set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden_dim);
  return MLFF_ERR_UNSUPPORTED;
}

int mlff_train_readout(void* stream, int parts, int n_atoms, int hidden_dim, const float* s_dev,
                       const float* ds_dev, const float* w1_dev, const float* b1_dev,
                       const float* w2_dev, const float* b2_dev, const float* w3_dev,
                       const float* b3_dev, float* r1_dev, float* h3_dev, float* r2_dev,
                       float* h4_dev, float* eps_dev, float* dr1_dev, float* dh3_dev,
                       float* dr2_dev, float* dh4_dev) {
  const char* nm = "mlff_train_readout";
  const bool prim = parts & 1, tan = parts & 2;
  if (n_atoms < 0 || parts < 1 || parts > 3) {
    set_error("%s: invalid size or parts", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_atoms == 0) return MLFF_OK;
  if (!present({w1_dev, w2_dev, r1_dev, r2_dev}) ||
      (prim && !present({s_dev, b1_dev, b2_dev, w3_dev, b3_dev, h3_dev, h4_dev, eps_dev})) ||
      (tan && !present({ds_dev, dr1_dev, dh3_dev, dr2_dev, dh4_dev}))) {
    set_error("%s: null buffer", nm);
    return MLFF_ERR_INVALID;
  }
  if (!aligned({s_dev, ds_dev, w1_dev, w2_dev, w3_dev})) {
    set_error("%s: buffers must be 16-byte aligned", nm);
    return MLFF_ERR_INVALID;
  }
  const ReadArgs p = {n_atoms, s_dev, ds_dev, w1_dev, b1_dev, w2_dev, b2_dev, w3_dev, b3_dev,
                      r1_dev, h3_dev, r2_dev, h4_dev, eps_dev, dr1_dev, dh3_dev, dr2_dev, dh4_dev};
  auto run = [&](auto kernel) {
    kernel<<<(n_atoms + kTM - 1) / kTM, kReadBlock, 0, static_cast<hipStream_t>(stream)>>>(p);
    return finish(nm);
  };
#define MLFF_READ(H)                                                   \
  case H:                                                              \
    return prim && tan ? run(train_readout_fwd_kernel<H, true, true>)  \
           : prim      ? run(train_readout_fwd_kernel<H, true, false>) \
                       : run(train_readout_fwd_kernel<H, false, true>);
  switch (hidden_dim) {
    MLFF_READ(32)
    MLFF_READ(64)
    MLFF_READ(128)
  }
#undef MLFF_READ
  set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden_dim);
  return MLFF_ERR_UNSUPPORTED;
}

int mlff_train_readout_adjoint(void* stream, int n_atoms, int hidden_dim, const float* seed_dev,
                               const int64_t* batch_dev, const float* r1_dev, const float* r2_dev,
                               const float* dr1_dev, const float* dr2_dev, const float* w1_dev,
                               const float* w2_dev, const float* w3_dev, float* g4_dev,
                               float* gr2_dev, float* gr1_dev, float* gs_dev, float* dgr2_dev,
                               float* dgr1_dev, float* dgs_dev) {
  const char* nm = "mlff_train_readout_adjoint";
  const bool tan = dr1_dev != nullptr;
  if (n_atoms < 0) {
    set_error("%s: invalid size", nm);
    return MLFF_ERR_INVALID;
  }
  if (n_atoms == 0) return MLFF_OK;
  if (!present({seed_dev, batch_dev, r1_dev, r2_dev, w1_dev, w2_dev, w3_dev, g4_dev, gr2_dev,
                gr1_dev, gs_dev}) ||
      (tan && !present({dr2_dev, dgr2_dev, dgr1_dev, dgs_dev}))) {
    set_error("%s: null buffer", nm);
    return MLFF_ERR_INVALID;
  }
  const ReadAdjArgs p = {n_atoms, seed_dev, batch_dev, r1_dev, r2_dev, dr1_dev, dr2_dev, w1_dev,
                         w2_dev, w3_dev, g4_dev, gr2_dev, gr1_dev, gs_dev, dgr2_dev, dgr1_dev,
                         dgs_dev};
  auto run = [&](auto kernel) {
    kernel<<<(n_atoms + kTM - 1) / kTM, kReadBlock, 0, static_cast<hipStream_t>(stream)>>>(p);
    return finish(nm);
  };
  switch (hidden_dim) {
    case 32: return tan ? run(train_readout_bwd_kernel<32, true>) : run(train_readout_bwd_kernel<32, false>);
    case 64: return tan ? run(train_readout_bwd_kernel<64, true>) : run(train_readout_bwd_kernel<64, false>);
    case 128: return tan ? run(train_readout_bwd_kernel<128, true>) : run(train_readout_bwd_kernel<128, false>);
  }
  set_error("%s: hidden_dim %d not supported (32, 64, 128)", nm, hidden_dim);
  return MLFF_ERR_UNSUPPORTED;
}

}  // extern "C"
