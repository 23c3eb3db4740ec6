// PaiNN student energy and hand-written adjoint (forces, virial) on gfx950.
//
// Forward follows StudentForceField.forward (student_model.py:634-757):
//   embedding -> L x [message (PaiNNMessage :346-387), update (PaiNNUpdate
//   :434-470)] -> energy_head (:599-605) -> per-structure sum (FP64 here).
// Forces are -dE/dx from the adjoint below instead of torch.autograd
// (student_model.py:788-793).
//
// Data layout (all float32, row-major): node scalars s [N][H], node vectors
// v [N][3][H] (xyz in the middle, as the reference); per unordered pair p
// (lo < hi): geometry {vec = p_hi - p_lo (+ image shift), d} and the filter
// output W_p [3H] = (W_s | W_v1 | W_v2) of each block.
//
// Kernels and what bounds them:
//   filter_table_fwd, filter_table_bwd (filter_table.hip)  pairs, the filters and their
//                adjoint from distance tables: HBM writes, table rows from beyond the L2
//   filter_fwd, filter_bwd  the same by the MLP per pair, where no table can stand and
//                behind the guard's flag until the host has read it:
//     forward    MFMA (R->H, SiLU, H->3H; the H->3H product on the bf16 matrix cores
//                with three-way split operands); 2(RH + 3H^2) flop/pair
//     adjoint    gathers both endpoints' features and gradients, MFMA (3H->H, H->R)
//                back to dE/dd and dE/du
//   message      receiver rows, gather of s_j, v_j, W_p (HBM/L2)
//   update_fwd   atoms, MFMA (2H->H, SiLU, H->3H) + gated vector epilogue
//   readout      atoms, MFMA head and its input gradient in one pass
//   update_bwd   atoms, MFMA (3H->H, H->2H) transposed products
//   force_gather receiver rows, forces and per-atom virial from dE/dvec
//   reduce       per structure FP64 sums (energy, virial)

#include <type_traits>

#include "common.hpp"
#include "internal.hpp"

namespace mlff {

namespace {

constexpr int kBlock = 256;
constexpr int kPairBlock = 512;       // 8 waves: each owns few output tiles, many in flight
constexpr int kPairWaves = kPairBlock / 64;
constexpr int kMaxRbf = 32;          // radial basis size limit (padded to 16: 16 or 32)
// pairs per tile, filter forward: 128 for the compact hidden size, 64 above
template <int H>
constexpr int kFwdPairs = H <= 32 ? 128 : 64;
// pairs per tile, filter adjoint: 64 for the compact hidden size (its tiles are
// short, so fewer, longer ones), 32 above (two blocks per CU fit the LDS)
template <int H>
constexpr int kBwdPairs = H <= 32 ? 64 : 32;
constexpr int kUpdWaves = 8;          // update kernels: waves per 32-atom tile
constexpr int kUpdBlock = 64 * kUpdWaves;
// Atoms up to which the update blocks run split over columns, and the update
// blocks and the readout on 16-atom tiles.  H = 128, forward + adjoint of a
// block: 60 atoms 24 us split, 34 us whole (33 with 16-atom tiles); 3000 atoms
// 42 us split, 41 us in 32-atom and 34 us in 16-atom tiles (one round of the
// CUs in either, half the products per CU); 14,000 atoms 89 us in 32-atom and
// 109 us in 16-atom tiles, which read the weights twice as often.
// Readout: 14 -> 7 us at 60 atoms, 15 -> 9 us at 3000.
// Where the lines lie, whole evaluations of 40-atom molecules, three blocks at H = 128
// (two at H = 32): split against 16-atom tiles 191 / 204 us at 720 atoms, 221 / 235 at
// 1000, 274 / 248 at 1240 (H = 32: 4 us behind from 240 atoms on); 16-atom against
// 32-atom tiles 533 / 556 us at 4000 atoms, 653 / 633 at 5000 (H = 32: ahead by 5 % up to
// 10,000).
constexpr int kSplitAtoms = 1024;
constexpr int kSmallTileAtoms = 4096;
// Message rows: sums per row, and the atoms up to which each has threads of its own.
// The same evaluations, split against whole rows: 143 / 151 us at 240 atoms, 166 / 166 at
// 480, 221 / 209 at 1000 (H = 32: 62 / 73, 69 / 79, 79 / 85, 98 / 96 at 2000).
constexpr int kMsgSums = 4;
constexpr int kMsgSplitAtoms = 1024;
// edges in flight per row in the message kernels (forward, adjoint)
constexpr int kMsgUnrollFwd = 8;
constexpr int kMsgUnrollBwd = 8;
// The other launch shape of each kernel, pre-instantiated so the launch-shape
// tuner can choose per workload (mlff_plan_set_tiles).  Results are
// bit-identical across shapes: every output element sums in the same order.
template <int H>
constexpr int kFwdPairsAlt = H <= 32 ? 64 : 32;
template <int H>
constexpr int kBwdPairsAlt = H <= 32 ? 32 : 64;
constexpr int kMsgUnrollFwdAlt = 4;
constexpr int kMsgUnrollBwdAlt = 4;

// Grid of a pair kernel: the plan's persistent grid, capped at the number of
// tiles the pair capacity allows (a multiple of 8 for the XCD-interleaved tile
// order), so small batches do not dispatch thousands of idle workgroups.
inline int pair_grid(const Buffers& b, int pairs_per_tile) {
  const int tiles = (b.pcap + pairs_per_tile - 1) / pairs_per_tile;
  return std::max(8, std::min(b.blocks, (tiles + 7) / 8 * 8));
}

template <int H>
__global__ void embed_kernel(int N, const int64_t* __restrict__ Z,
                             const float* __restrict__ emb, float* __restrict__ S0,
                             float* __restrict__ V0) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < N * (H / 4)) embed_item<H>(idx, Z, emb, S0, V0);
}

// ---------------------------------------------------------------------------
// filter forward: W_p = W2 silu(W1 e(d_p) + b1) + b2 for kFwdPairs<H> pairs per tile
// ---------------------------------------------------------------------------
template <int H, int TM>
__global__ __launch_bounds__(kPairBlock, 4) void filter_fwd_kernel(
    const float4* __restrict__ geom, const int32_t* __restrict__ counts, int32_t pcap,
    const float* __restrict__ w, LayerW lw, const float* __restrict__ centers,
    const float* __restrict__ widths, int R, int RP, float rc, float* __restrict__ Wout,
    const uint16_t* __restrict__ w2bf, const int32_t* __restrict__ gate) {
  if (gate != nullptr && *gate == 0) return;
  constexpr int RT = TM / 16;
  constexpr int LDE = kMaxRbf + 4;
  constexpr int LDHB = H + 8;          // bf16 row stride of the split hidden activations
  constexpr int PHB = TM * LDHB;       // plane stride
  constexpr int CT1 = H / 16, NT1 = (CT1 + kPairWaves - 1) / kPairWaves;
  constexpr int CT2 = 3 * H / 16, NT2 = (CT2 + kPairWaves - 1) / kPairWaves;
  static_assert(CT1 % NT1 == 0 && CT2 % NT2 == 0, "tile split");
  __shared__ __align__(16) float e_lds[TM * LDE];
  __shared__ __align__(16) uint16_t h_bf[3 * PHB];   // silu(W1 e + b1) as three bf16 planes
  __shared__ float mu_lds[kMaxRbf], gam_lds[kMaxRbf];
  __shared__ float d_lds[TM], fc_lds[TM];
  if (threadIdx.x < kMaxRbf) {
    const int k = threadIdx.x;
    mu_lds[k] = k < R ? centers[k] : 0.f;
    gam_lds[k] = k < R ? rbf_gamma(widths[k]) : 0.f;
  }
  const int P = min(counts[MLFF_COUNT_PAIRS], pcap);
  const int ntiles = (P + TM - 1) / TM;
  int t0, t1;
  int tstep;
  persistent_range(ntiles, t0, t1, tstep);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const float* f1w = w + lw.f1w;
  const float* f1b = w + lw.f1b;
  const float* f2b = w + lw.f2b;
  for (int tile = t0; tile < t1; tile += tstep) {
    const int pbase = tile * TM;
    if (threadIdx.x < TM) {   // the cutoff once per pair
      const int p = pbase + threadIdx.x;
      float d = 0.f, fc = 0.f, dfc;
      if (p < P) {
        d = geom[p].w;
        cosine_cutoff(d, rc, fc, dfc);
      }
      d_lds[threadIdx.x] = d;
      fc_lds[threadIdx.x] = fc;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < TM * RP; idx += kPairBlock) {
      const int m = idx / RP, k = idx - m * RP;
      const int p = pbase + m;
      float val = 0.f;
      if (p < P && k < R) val = edge_feature(d_lds[m], mu_lds[k], gam_lds[k], fc_lds[m]);
      e_lds[m * LDE + k] = val;
    }
    __syncthreads();
    if (wave < CT1 / NT1) {
      int cb[NT1];
      f4 acc[RT][NT1];
#pragma unroll
      for (int ct = 0; ct < NT1; ++ct) cb[ct] = (wave * NT1 + ct) * 16;
      zero_acc(acc);
      mma_tile<RT, NT1>(e_lds, LDE, f1w, RP, RP, cb, acc);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NT1; ++ct) {
          const int c = cb[ct] + r;
          const float bias = f1b[c];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int m = rt * 16 + 4 * g + i;
            uint16_t hh, hm, hl;
            split3_bf16(silu(acc[rt][ct][i] + bias), hh, hm, hl);
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
      // W_p = h W2^T + b2 on the bf16 matrix cores at float32 accuracy
      mma_tile_x6<RT, NT2, H>(h_bf, LDHB, PHB, w2bf, H, (int)wbf_plane(H), cb, acc);
      float bias[NT2];
#pragma unroll
      for (int ct = 0; ct < NT2; ++ct) bias[ct] = f2b[cb[ct] + r];
      // lane (r, g) holds rows rt*16 + 4g + i, columns cb[ct] + r.  W_p is
      // written once and read by a later kernel: non-temporal stores keep it
      // from displacing L2 lines.
      float* out = Wout + (size_t)(pbase + 4 * g) * 3 * H + r;
      if (pbase + TM <= P) {   // full tile: no per-element bounds checks
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int ct = 0; ct < NT2; ++ct)
              __builtin_nontemporal_store(acc[rt][ct][i] + bias[ct],
                                          &out[(size_t)(rt * 16 + i) * 3 * H + cb[ct]]);
      } else {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (pbase + rt * 16 + 4 * g + i >= P) continue;
#pragma unroll
            for (int ct = 0; ct < NT2; ++ct)
              __builtin_nontemporal_store(acc[rt][ct][i] + bias[ct],
                                          &out[(size_t)(rt * 16 + i) * 3 * H + cb[ct]]);
          }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// message (forward) and its node-gradient transpose (backward).
// FWD:  s'_i = s_i + sum_j s_j * Ws_p ;  v'_i = v_i + sum_j v_j * Wv1_p + u_ji (x) Wv2_p
// BWD:  gs_i = gs'_i + sum_j gs'_j * Ws_p ; gv_i = gv'_i + sum_j gv'_j * Wv1_p
// One channel per lane, H lanes per row, neighbours in ascending j; the operands
// of UNROLL edges are requested before any is added.  Edges
// e, e + 4, ... of a row have a sum of their own: shorter rounding chains, and with
// few rows (SPLIT) four times the threads, one sum each, same bits.
// A wave works on one row (H >= 64), so a row's neighbour and pair indices and
// unit vectors are scalar loads and the loop spends its vector registers on
// operands in flight only.  Bound by reading every W_p once per direction
// (HBM) on large batches, by the chain of load rounds per row on small ones.
// Four channels per lane, five edges in flight, took 209 / 155 us (forward /
// adjoint) for 256 molecules of 10-100 atoms at H = 128, 55 / 36 us for 1000
// waters and 32 / 21 us for one molecule of 60 atoms; this form 180 / 144,
// 47 / 32 and 10 / 7 us.  Twelve edges in flight: 180 / 143, 48 / 33, 12 / 7.
// SPLIT: 6.3 / 4.8 us for the molecule of 60 atoms.
// ZEROV: the first block, whose vectors are zero: their products with Wv1 add
// exact zeros (zero_vectors()), so neither is read.
// ---------------------------------------------------------------------------
template <int H, bool FWD, int UNROLL, bool SPLIT, bool ZEROV>
__global__ __launch_bounds__(SPLIT ? kMsgSums * H : kBlock) void message_kernel(
    int N, const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ col,
    const int32_t* __restrict__ edge_pair, int32_t ecap, const float4* __restrict__ unit,
    const float* __restrict__ Wf, const float* __restrict__ s_in, const float* __restrict__ v_in,
    float* __restrict__ s_out, float* __restrict__ v_out) {
  constexpr int RPB = SPLIT ? 1 : kBlock / H;
  constexpr int NA = SPLIT ? 1 : kMsgSums;       // sums of a thread
  constexpr int STEP = SPLIT ? kMsgSums : 1;     // edges from one of its edges to the next
  const int c = threadIdx.x % H;
  int i = xcd_block() * RPB + (SPLIT ? 0 : threadIdx.x / H);
  int part = SPLIT ? threadIdx.x / H : 0;
  if (H >= 64) part = __builtin_amdgcn_readfirstlane(part);
  if (H >= 64) i = __builtin_amdgcn_readfirstlane(i);   // uniform: indices in scalar registers
  if (i >= N) return;
  float as[NA], a0[NA], a1[NA], a2[NA];
#pragma unroll
  for (int o = 0; o < NA; ++o) as[o] = a0[o] = a1[o] = a2[o] = 0.f;
  const int e0 = min(row_ptr[i], ecap), e1 = min(row_ptr[i + 1], ecap);
  // neighbour and pair indices of the next step, requested a step ahead (past
  // the row's end: the last edge's)
  int jn[UNROLL], pn[UNROLL];
  auto indices = [&](int e) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int ec = min(e + STEP * u, e1 - 1);
      jn[u] = col[ec];
      pn[u] = edge_pair[ec];
    }
  };
  // UNROLL edges from e on: all their operands are requested before any is
  // used (the barrier keeps the compiler from moving loads behind the sums).
  // TAIL: edges past the row's end count with zero weights.
  auto step = [&](int e, auto tail) {
    constexpr bool TAIL = decltype(tail)::value;
    float ws[UNROLL], wv1[UNROLL], wv2[UNROLL], sj[UNROLL], v0[UNROLL], v1[UNROLL], v2[UNROLL];
    float4 uu[UNROLL];
    int jc[UNROLL];
    bool on[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int p = max(pn[u], 0);
      jc[u] = jn[u];
      on[u] = (!TAIL || e + STEP * u < e1) && pn[u] >= 0;
      const float* wp = Wf + (size_t)p * 3 * H;
      const float* vj = v_in + (size_t)jc[u] * 3 * H;
      ws[u] = wp[c];
      sj[u] = (s_in + (size_t)jc[u] * H)[c];
      if (!ZEROV) {
        wv1[u] = wp[H + c];
        v0[u] = vj[c];
        v1[u] = vj[H + c];
        v2[u] = vj[2 * H + c];
      }
      if (FWD) {
        wv2[u] = wp[2 * H + c];
        uu[u] = unit[p];
      }
    }
    if (!TAIL) indices(e + STEP * UNROLL);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const float w0 = on[u] ? ws[u] : 0.f;
      const int o = u % NA;   // UNROLL is a multiple of NA
      as[o] = fma_(sj[u], w0, as[o]);
      if (!ZEROV) {
        const float w1 = on[u] ? wv1[u] : 0.f;
        a0[o] = fma_(v0[u], w1, a0[o]);
        a1[o] = fma_(v1[u], w1, a1[o]);
        a2[o] = fma_(v2[u], w1, a2[o]);
      }
      if (FWD) {
        // u_ji = (p_j - p_i)/(d + eps): +pair vector when j is the pair's hi atom
        const float w2 = on[u] ? (jc[u] < i ? -wv2[u] : wv2[u]) : 0.f;
        a0[o] = fma_(uu[u].x, w2, a0[o]);
        a1[o] = fma_(uu[u].y, w2, a1[o]);
        a2[o] = fma_(uu[u].z, w2, a2[o]);
      }
    }
  };
  int e = e0 + part;
  if (e < e1) indices(e);
  for (; e + STEP * (UNROLL - 1) < e1; e += STEP * UNROLL) step(e, std::false_type{});
  if (e < e1) step(e, std::true_type{});
  float t[kMsgSums][4];
  if constexpr (SPLIT) {
    __shared__ float sh[kMsgSums][4][H];
    sh[part][0][c] = as[0];
    sh[part][1][c] = a0[0];
    sh[part][2][c] = a1[0];
    sh[part][3][c] = a2[0];
    __syncthreads();
    if (part != 0) return;
#pragma unroll
    for (int o = 0; o < kMsgSums; ++o)
#pragma unroll
      for (int k = 0; k < 4; ++k) t[o][k] = sh[o][k][c];
  } else {
#pragma unroll
    for (int o = 0; o < kMsgSums; ++o) {
      t[o][0] = as[o];
      t[o][1] = a0[o];
      t[o][2] = a1[o];
      t[o][3] = a2[o];
    }
  }
  auto sum = [&](int k) { return (t[0][k] + t[1][k]) + (t[2][k] + t[3][k]); };
  const float* vi = v_in + (size_t)i * 3 * H + c;
  float* vo = v_out + (size_t)i * 3 * H + c;
  s_out[(size_t)i * H + c] = s_in[(size_t)i * H + c] + sum(0);
  vo[0] = vi[0] + sum(1);
  vo[H] = vi[H] + sum(2);
  vo[2 * H] = vi[2 * H] + sum(3);
}

// a . b in x order, with the fused operations spelled out: every tile shape of a
// kernel gets the same bits
__device__ __forceinline__ float dot3(float a0, float a1, float a2, float b0, float b1, float b2) {
  return fma_(a2, b2, fma_(a1, b1, a0 * b0));
}

// ---------------------------------------------------------------------------
// update forward, TM atoms per tile.  The products run on four accumulator sets
// (mma_tile_k4): on one set they are the largest part of an energy's error
// (molecules with large biases: 4.7e-5 eV/atom rms with one set, 3.1e-5 with
// two, 2.3e-5 with four, in the same time).
// GATES: the vectors too; without, the scalars alone.  Nothing reads the last block's
// vectors (the energy is a function of its scalars), nor its gates in the adjoint
// (256 molecules 2032 -> 2011 us, 60 atoms 139.1 -> 137.6 us an MD step).
// ---------------------------------------------------------------------------
template <int H, int TM, bool GATES>
__global__ __launch_bounds__(kUpdBlock) void update_fwd_kernel(
    int N, const float* __restrict__ w, LayerW lw, const float* __restrict__ s_mid,
    const float* __restrict__ v_mid, float* __restrict__ s_out, float* __restrict__ v_out,
    float* __restrict__ a_upd, float* __restrict__ g12) {
  constexpr int RT = TM / 16;
  constexpr int LDX = 2 * H + 4, LDH = H + 4;
  constexpr int CT1 = H / 16, NT1 = (CT1 + kUpdWaves - 1) / kUpdWaves;
  constexpr int NTC = NT1, NS = GATES ? 3 : 1, NT2 = NS * NTC;
  __shared__ __align__(16) float x_lds[TM * LDX];
  __shared__ __align__(16) float h_lds[TM * LDH];
  constexpr int PER = TM * H / kUpdBlock;   // tile elements per thread
  static_assert(PER * kUpdBlock == TM * H, "tile split");
  const int base = blockIdx.x * TM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  {
    // every load of the tile in flight at once (rows past N read atom N-1
    // and are zeroed), then the norms
    float sv[PER], x0[PER], x1[PER], x2[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = threadIdx.x + k * kUpdBlock, m = idx / H, c = idx % H;
      const int i = min(base + m, N - 1);
      sv[k] = s_mid[(size_t)i * H + c];
      const float* vv = v_mid + (size_t)i * 3 * H;
      x0[k] = vv[c];
      x1[k] = vv[H + c];
      x2[k] = vv[2 * H + c];
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = threadIdx.x + k * kUpdBlock, m = idx / H, c = idx % H;
      const bool in = base + m < N;
      x_lds[m * LDX + c] = in ? sv[k] : 0.f;
      x_lds[m * LDX + H + c] = in ? norm3_exact(x0[k], x1[k], x2[k]) : 0.f;
    }
  }
  __syncthreads();
  if (wave < CT1 / NT1) {
    int cb[NT1];
    f4 acc[RT][NT1];
#pragma unroll
    for (int ct = 0; ct < NT1; ++ct) cb[ct] = (wave * NT1 + ct) * 16;
    zero_acc(acc);
    mma_tile_k4<RT, NT1, 2 * H>(x_lds, LDX, w + lw.u1w, 2 * H, cb, acc);
    const float* b1 = w + lw.u1b;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ct = 0; ct < NT1; ++ct) {
        const int c = cb[ct] + r;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int m = rt * 16 + 4 * g + k, i = base + m;
          const float a = acc[rt][ct][k] + b1[c];
          if (i < N) a_upd[(size_t)i * H + c] = a;
          h_lds[m * LDH + c] = silu(a);
        }
      }
  }
  __syncthreads();
  if (wave < CT1 / NTC) {
    int cb[NT2];
    f4 acc[RT][NT2];
#pragma unroll
    for (int q = 0; q < NTC; ++q)
#pragma unroll
      for (int sp = 0; sp < NS; ++sp) cb[sp * NTC + q] = sp * H + (wave * NTC + q) * 16;
    // the epilogue's operands (biases, mixing matrix, the tile's vectors)
    // are loaded before the product, so their latency hides behind it
    const float* b2 = w + lw.u2b;
    const float* U = w + lw.mix;
    float u[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) u[k] = GATES ? U[k] : 0.f;
    float bias[NTC][NS];
    float xv[RT][NTC][4][3];
#pragma unroll
    for (int q = 0; q < NTC; ++q) {
      const int c = (wave * NTC + q) * 16 + r;
#pragma unroll
      for (int sp = 0; sp < NS; ++sp) bias[q][sp] = b2[sp * H + c];
#pragma unroll
      for (int rt = 0; GATES && rt < RT; ++rt)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int i = min(base + rt * 16 + 4 * g + k, N - 1);
          const float* vv = v_mid + (size_t)i * 3 * H;
#pragma unroll
          for (int sp = 0; sp < 3; ++sp) xv[rt][q][k][sp] = vv[sp * H + c];
        }
    }
    zero_acc(acc);
    mma_tile_k4<RT, NT2, H>(h_lds, LDH, w + lw.u2w, H, cb, acc);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 0; q < NTC; ++q) {
        const int c = (wave * NTC + q) * 16 + r;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int m = rt * 16 + 4 * g + k, i = base + m;
          if (i >= N) continue;
          const float ds = acc[rt][q][k] + bias[q][0];
          s_out[(size_t)i * H + c] = x_lds[m * LDX + c] + ds;
          if constexpr (GATES) {
            const float gt1 = acc[rt][NTC + q][k] + bias[q][1];
            const float gt2 = acc[rt][2 * NTC + q][k] + bias[q][2];
            const float x0 = xv[rt][q][k][0], x1 = xv[rt][q][k][1], x2 = xv[rt][q][k][2];
            float* vo = v_out + (size_t)i * 3 * H;
            vo[c] = fma_(dot3(u[0], u[1], u[2], x0, x1, x2), gt2, x0 * gt1);
            vo[H + c] = fma_(dot3(u[3], u[4], u[5], x0, x1, x2), gt2, x1 * gt1);
            vo[2 * H + c] = fma_(dot3(u[6], u[7], u[8], x0, x1, x2), gt2, x2 * gt1);
            g12[(size_t)i * 2 * H + c] = gt1;
            g12[(size_t)i * 2 * H + H + c] = gt2;
          }
        }
      }
  }
}

// ---------------------------------------------------------------------------
// readout: eps_i = head(s_i) and gs_i = d eps_i / d s_i, TM atoms per tile
// ---------------------------------------------------------------------------
template <int H, int TM>
__global__ __launch_bounds__(kBlock) void readout_kernel(int N, const float* __restrict__ w,
                                                         ModelW mw, const float* __restrict__ sL,
                                                         float* __restrict__ eps,
                                                         float* __restrict__ gS) {
  constexpr int RT = TM / 16;
  constexpr bool kRegs = TM == 16;
  constexpr int HP2 = ((H / 2) + 15) & ~15, HP4 = ((H / 4) + 15) & ~15;
  constexpr int LDX = H + 4, LD2 = HP2 + 4, LD4 = HP4 + 4;
  __shared__ __align__(16) float x_lds[TM * LDX];
  __shared__ __align__(16) float a1_lds[TM * LD2];
  __shared__ __align__(16) float h1_lds[TM * LD2];
  __shared__ __align__(16) float a2_lds[TM * LD4];
  __shared__ __align__(16) float g2_lds[TM * LD4];
  const int base = blockIdx.x * TM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  // a wave's column tile of the two hidden layers, and its tiles of the input
  // gradient (waves past the last repeat the first's loads, unused)
  constexpr int CTG = H / 16, NTG = (CTG + 3) / 4;
  int c2[1] = {wave < HP2 / 16 ? wave * 16 : 0}, c4[1] = {wave < HP4 / 16 ? wave * 16 : 0},
      cg[NTG];
#pragma unroll
  for (int ct = 0; ct < NTG; ++ct) cg[ct] = (wave < CTG / NTG ? wave * NTG + ct : ct) * 16;
  Weights<1, H> wr1;
  Weights<1, HP2> wr2;
  Weights<1, HP4> wr2t;
  Weights<NTG, HP2> wr1t;
  if (kRegs) {
    load_weights(w + mw.r1w, H, c2, wr1);
    load_weights(w + mw.r2w, HP2, c4, wr2);
  }
  {
    constexpr int PER = TM * H / kBlock;
    static_assert(PER * kBlock == TM * H, "tile split");
    float xs[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = threadIdx.x + k * kBlock, m = idx / H, c = idx % H;
      xs[k] = sL[(size_t)min(base + m, N - 1) * H + c];
    }
    if (kRegs) {
      load_weights(w + mw.r2t, HP4, c2, wr2t);
      load_weights(w + mw.r1t, HP2, cg, wr1t);
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int idx = threadIdx.x + k * kBlock, m = idx / H, c = idx % H;
      x_lds[m * LDX + c] = (base + m < N) ? xs[k] : 0.f;
    }
  }
  __syncthreads();
  if (wave < HP2 / 16) {   // Linear(H, H/2) + SiLU, one column tile per wave
    f4 acc[RT][1];
    zero_acc(acc);
    if constexpr (kRegs) mma_regs(x_lds, LDX, wr1, acc);
    else mma_tile_k4<RT, 1, H>(x_lds, LDX, w + mw.r1w, H, c2, acc);
    const int c = c2[0] + r;
    const float bias = w[mw.r1b + c];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int m = rt * 16 + 4 * g + k;
        const float a = acc[rt][0][k] + bias;
        a1_lds[m * LD2 + c] = a;
        h1_lds[m * LD2 + c] = silu(a);
      }
  }
  __syncthreads();
  if (wave < HP4 / 16) {   // Linear(H/2, H/4)
    f4 acc[RT][1];
    zero_acc(acc);
    if constexpr (kRegs) mma_regs(h1_lds, LD2, wr2, acc);
    else mma_tile_k4<RT, 1, HP2>(h1_lds, LD2, w + mw.r2w, HP2, c4, acc);
    const int c = c4[0] + r;
    const float bias = w[mw.r2b + c];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int k = 0; k < 4; ++k) a2_lds[(rt * 16 + 4 * g + k) * LD4 + c] = acc[rt][0][k] + bias;
  }
  __syncthreads();
  const float* w3 = w + mw.r3w;
  // Linear(H/4, 1), its input gradient, and SiLU': eight lanes per atom, a run
  // of HP4 / 8 channels each
  if (threadIdx.x < TM * 8) {
    constexpr int RUN = HP4 / 8;
    const int m = threadIdx.x / 8, c0 = (threadIdx.x % 8) * RUN, i = base + m;
    float e = 0.f;
#pragma unroll
    for (int k = 0; k < RUN; ++k) {
      const float a = a2_lds[m * LD4 + c0 + k], q = w3[c0 + k];
      e = fma_(silu(a), q, e);
      g2_lds[m * LD4 + c0 + k] = q * silu_grad(a);
    }
    e = group_sum<8>(e);
    if (c0 == 0 && i < N) eps[i] = e + w[mw.r3b];
  }
  __syncthreads();
  if (wave < HP2 / 16) {   // d/dh1 = g2 W2, then SiLU'
    f4 acc[RT][1];
    zero_acc(acc);
    if constexpr (kRegs) mma_regs(g2_lds, LD4, wr2t, acc);
    else mma_tile_k4<RT, 1, HP4>(g2_lds, LD4, w + mw.r2t, HP4, c2, acc);
    const int c = c2[0] + r;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int m = rt * 16 + 4 * g + k;
        h1_lds[m * LD2 + c] = acc[rt][0][k] * silu_grad(a1_lds[m * LD2 + c]);
      }
  }
  __syncthreads();
  {   // d/ds = g1 W1 over H output columns
    if (wave < CTG / NTG) {
      f4 acc[RT][NTG];
      zero_acc(acc);
      if constexpr (kRegs) mma_regs(h1_lds, LD2, wr1t, acc);
      else mma_tile_k4<RT, NTG, HP2>(h1_lds, LD2, w + mw.r1t, HP2, cg, acc);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NTG; ++ct)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int i = base + rt * 16 + 4 * g + k;
            if (i < N) gS[(size_t)i * H + cg[ct] + r] = acc[rt][ct][k];
          }
    }
  }
}

// ---------------------------------------------------------------------------
// update backward, TM atoms per tile.  gv2 == nullptr means a zero gradient.
// ---------------------------------------------------------------------------
template <int H, int TM>
__global__ __launch_bounds__(kUpdBlock) void update_bwd_kernel(
    int N, const float* __restrict__ w, LayerW lw, const float* __restrict__ gs2,
    const float* __restrict__ gv2, const float* __restrict__ v_mid,
    const float* __restrict__ a_upd, const float* __restrict__ g12, float* __restrict__ gs1,
    float* __restrict__ gv1) {
  constexpr int RT = TM / 16;
  constexpr int LDY = 3 * H + 4, LDA = H + 4, LDX = 2 * H + 4;
  __shared__ __align__(16) float y_lds[TM * LDY];
  __shared__ __align__(16) float a_lds[TM * LDA];
  const int base = blockIdx.x * TM;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const float* U = w + lw.mix;
  float u[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) u[k] = U[k];
  // loads in batches of kB elements per thread, all of a batch in flight at
  // once (rows past N read atom N-1 and are zeroed)
  constexpr int PER = TM * H / kUpdBlock;
  constexpr int kB = PER < 4 ? PER : 4;
  static_assert(PER * kUpdBlock == TM * H && PER % kB == 0, "tile split");
#pragma unroll
  for (int kb = 0; kb < PER; kb += kB) {
    float y0[kB], x0[kB], x1[kB], x2[kB], q0[kB], q1[kB], q2[kB];
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int idx = threadIdx.x + (kb + k) * kUpdBlock, m = idx / H, c = idx % H;
      const int i = min(base + m, N - 1);
      y0[k] = gs2[(size_t)i * H + c];
      if (gv2 != nullptr) {
        const float* vv = v_mid + (size_t)i * 3 * H;
        const float* gg = gv2 + (size_t)i * 3 * H;
        x0[k] = vv[c]; x1[k] = vv[H + c]; x2[k] = vv[2 * H + c];
        q0[k] = gg[c]; q1[k] = gg[H + c]; q2[k] = gg[2 * H + c];
      }
    }
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int idx = threadIdx.x + (kb + k) * kUpdBlock, m = idx / H, c = idx % H;
      const bool in = base + m < N;
      float y1 = 0.f, y2 = 0.f;
      if (gv2 != nullptr) {
        y1 = dot3(q0[k], q1[k], q2[k], x0[k], x1[k], x2[k]);
        y2 = dot3(q0[k], q1[k], q2[k], dot3(u[0], u[1], u[2], x0[k], x1[k], x2[k]),
                  dot3(u[3], u[4], u[5], x0[k], x1[k], x2[k]),
                  dot3(u[6], u[7], u[8], x0[k], x1[k], x2[k]));
      }
      y_lds[m * LDY + c] = in ? y0[k] : 0.f;
      y_lds[m * LDY + H + c] = in ? y1 : 0.f;
      y_lds[m * LDY + 2 * H + c] = in ? y2 : 0.f;
    }
  }
  __syncthreads();
  {
    constexpr int CT = H / 16, NT = (CT + kUpdWaves - 1) / kUpdWaves;
    if (wave < CT / NT) {
      int cb[NT];
      f4 acc[RT][NT];
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) cb[ct] = (wave * NT + ct) * 16;
      float av[RT][NT][4];   // pre-activations, loaded before the product
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int i = min(base + rt * 16 + 4 * g + k, N - 1);
            av[rt][ct][k] = a_upd[(size_t)i * H + cb[ct] + r];
          }
      zero_acc(acc);
      mma_tile_k4<RT, NT, 3 * H, 2, true>(y_lds, LDY, w + lw.u2t, 3 * H, cb, acc);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int m = rt * 16 + 4 * g + k, i = base + m, c = cb[ct] + r;
            const float a = (i < N) ? av[rt][ct][k] : 0.f;
            a_lds[m * LDA + c] = acc[rt][ct][k] * silu_grad(a);
          }
    }
  }
  __syncthreads();
  float* x_lds = y_lds;   // y is dead after the barrier above
  {
    constexpr int CT = 2 * H / 16, NT = (CT + kUpdWaves - 1) / kUpdWaves;
    if (wave < CT / NT) {
      int cb[NT];
      f4 acc[RT][NT];
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) cb[ct] = (wave * NT + ct) * 16;
      zero_acc(acc);
      mma_tile_k4<RT, NT, H, 2, true>(a_lds, LDA, w + lw.u1t, H, cb, acc);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
#pragma unroll
          for (int k = 0; k < 4; ++k) x_lds[(rt * 16 + 4 * g + k) * LDX + cb[ct] + r] = acc[rt][ct][k];
    }
  }
  __syncthreads();
#pragma unroll
  for (int kb = 0; kb < PER; kb += kB) {
    float s2[kB], x0[kB], x1[kB], x2[kB], t1[kB], t2[kB], q0[kB], q1[kB], q2[kB];
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int idx = threadIdx.x + (kb + k) * kUpdBlock, m = idx / H, c = idx % H;
      const int i = min(base + m, N - 1);
      s2[k] = gs2[(size_t)i * H + c];
      const float* vv = v_mid + (size_t)i * 3 * H;
      x0[k] = vv[c]; x1[k] = vv[H + c]; x2[k] = vv[2 * H + c];
      if (gv2 != nullptr) {
        t1[k] = g12[(size_t)i * 2 * H + c];
        t2[k] = g12[(size_t)i * 2 * H + H + c];
        const float* gg = gv2 + (size_t)i * 3 * H;
        q0[k] = gg[c]; q1[k] = gg[H + c]; q2[k] = gg[2 * H + c];
      }
    }
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int idx = threadIdx.x + (kb + k) * kUpdBlock, m = idx / H, c = idx % H;
      const int i = base + m;
      if (i >= N) continue;
      gs1[(size_t)i * H + c] = s2[k] + x_lds[m * LDX + c];
      const float gn = x_lds[m * LDX + H + c];
      const float n = norm3_exact(x0[k], x1[k], x2[k]);
      const float sc = (n > 0.f) ? gn / n : 0.f;
      float o0 = sc * x0[k], o1 = sc * x1[k], o2 = sc * x2[k];
      if (gv2 != nullptr) {
        o0 = fma_(dot3(u[0], u[3], u[6], q0[k], q1[k], q2[k]), t2[k], fma_(q0[k], t1[k], o0));
        o1 = fma_(dot3(u[1], u[4], u[7], q0[k], q1[k], q2[k]), t2[k], fma_(q1[k], t1[k], o1));
        o2 = fma_(dot3(u[2], u[5], u[8], q0[k], q1[k], q2[k]), t2[k], fma_(q2[k], t1[k], o2));
      }
      float* go = gv1 + (size_t)i * 3 * H;
      go[c] = o0;
      go[H + c] = o1;
      go[2 * H + c] = o2;
    }
  }
}

// ---------------------------------------------------------------------------
// Update kernels for few atoms.  What one compute unit can have in flight from
// memory bounds a workgroup that takes a whole tile through the block at 17 us
// (it reads every weight, 0.3 MB at H = 128), however few atoms there are.  So a
// workgroup takes a 16-atom tile and 32 of the output channels.  Forward, its
// waves share the whole hidden layer between them (computed H / 32 times over,
// 0.9 us of products) and then the slice's columns of the second product: 10.1 us
// for 60 atoms, against 6.3 + 6.1 us as two launches.  The adjoint's first product
// has three times the weights, and there two launches are faster (7.3 + 4.4 us
// against 13.6).  All of a wave's weights are requested first.  Same sums as the
// whole-tile kernels, bit for bit.  Grid (16-atom tiles, H / 32).
// ---------------------------------------------------------------------------
template <int H, bool GATES>
__global__ __launch_bounds__(4 * H) void update_fwd_split_kernel(
    int N, const float* __restrict__ w, LayerW lw, const float* __restrict__ s_mid,
    const float* __restrict__ v_mid, float* __restrict__ s_out, float* __restrict__ v_out,
    float* __restrict__ a_upd, float* __restrict__ g12) {
  constexpr int BLK = 4 * H, WAVES = H / 16;
  constexpr int LDX = 2 * H + 4, LDH = H + 4, CT = GATES ? 6 : 2, LDY = 16 * CT + 4;
  constexpr int NT = (CT + WAVES - 1) / WAVES;   // second product: column tiles of ds, g1, g2
  constexpr int PE = 16 * 32 / BLK;              // outputs per thread
  __shared__ __align__(16) float x_lds[16 * LDX];
  __shared__ __align__(16) float h_lds[16 * LDH];
  __shared__ float y_lds[16 * LDY];
  const int base = blockIdx.x * 16, slice = blockIdx.y * 32;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int cb[1] = {16 * wave};
  Weights<1, 2 * H> w1;
  load_weights(w + lw.u1w, 2 * H, cb, w1);
  Weights<1, H> w2[NT];
  int col[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int t = min(wave + q * WAVES, CT - 1);
    col[q] = t / 2 * H + slice + 16 * (t % 2);
    const int c2[1] = {col[q]};
    load_weights(w + lw.u2w, H, c2, w2[q]);
  }
  {
    const int m = threadIdx.x / (H / 4), c = 4 * (threadIdx.x % (H / 4));
    const size_t i = min(base + m, N - 1);
    const float* vr = v_mid + i * 3 * H + c;
    auto ld = [](const float* q) { return *reinterpret_cast<const f4*>(q); };
    f4 sv = ld(s_mid + i * H + c);
    const f4 x0 = ld(vr), x1 = ld(vr + H), x2 = ld(vr + 2 * H);
    f4 n;
#pragma unroll
    for (int k = 0; k < 4; ++k) n[k] = norm3_exact(x0[k], x1[k], x2[k]);
    if (base + m >= N) sv = n = f4{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<f4*>(x_lds + m * LDX + c) = sv;
    *reinterpret_cast<f4*>(x_lds + m * LDX + H + c) = n;
  }
  float sm[PE], xv[PE][3], u[9];
#pragma unroll
  for (int k = 0; k < PE; ++k) {
    const int e = threadIdx.x + k * BLK, c = slice + e % 32;
    const size_t i = min(base + e / 32, N - 1);
    sm[k] = s_mid[i * H + c];
#pragma unroll
    for (int x = 0; x < 3; ++x) xv[k][x] = GATES ? v_mid[(i * 3 + x) * H + c] : 0.f;
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) u[k] = GATES ? (w + lw.mix)[k] : 0.f;
  const float b1 = (w + lw.u1b)[cb[0] + r];
  float b2[NT];
#pragma unroll
  for (int q = 0; q < NT; ++q) b2[q] = (w + lw.u2b)[col[q] + r];
  __syncthreads();
  {
    f4 acc[1][1];
    zero_acc(acc);
    mma_regs(x_lds, LDX, w1, acc);
    const int c = cb[0] + r;
    const bool own = cb[0] >= slice && cb[0] < slice + 32;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = base + 4 * g + k;
      const float a = acc[0][0][k] + b1;
      if (own && i < N) a_upd[(size_t)i * H + c] = a;
      h_lds[(4 * g + k) * LDH + c] = silu(a);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NT; ++q) {
    const int t = wave + q * WAVES;
    if (t >= CT) break;
    f4 acc[1][1];
    zero_acc(acc);
    mma_regs(h_lds, LDH, w2[q], acc);
#pragma unroll
    for (int k = 0; k < 4; ++k) y_lds[(4 * g + k) * LDY + 16 * t + r] = acc[0][0][k] + b2[q];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PE; ++k) {
    const int e = threadIdx.x + k * BLK, m = e / 32, c = slice + e % 32, i = base + m;
    if (i >= N) continue;
    const float* y = y_lds + m * LDY + e % 32;
    s_out[(size_t)i * H + c] = sm[k] + y[0];
    if (!GATES) continue;
    const float gt1 = y[32], gt2 = y[64];
    const float x0 = xv[k][0], x1 = xv[k][1], x2 = xv[k][2];
    float* vo = v_out + (size_t)i * 3 * H;
    vo[c] = fma_(dot3(u[0], u[1], u[2], x0, x1, x2), gt2, x0 * gt1);
    vo[H + c] = fma_(dot3(u[3], u[4], u[5], x0, x1, x2), gt2, x1 * gt1);
    vo[2 * H + c] = fma_(dot3(u[6], u[7], u[8], x0, x1, x2), gt2, x2 * gt1);
    g12[(size_t)i * 2 * H + c] = gt1;
    g12[(size_t)i * 2 * H + H + c] = gt2;
  }
}

constexpr int kSplitBlock = 128;

// ga = silu'(a) (gy W2), gy the gradient of (ds, g1, g2)
template <int H>
__global__ __launch_bounds__(kSplitBlock, 2) void update_hidden_bwd_kernel(
    int N, const float* __restrict__ w, LayerW lw, const float* __restrict__ gs2,
    const float* __restrict__ gv2, const float* __restrict__ v_mid,
    const float* __restrict__ a_upd, float* __restrict__ ga) {
  constexpr int LDY = 3 * H + 4, PER = 16 * H / kSplitBlock, kB = PER < 8 ? PER : 8;
  __shared__ __align__(16) float y_lds[16 * LDY];
  const int base = blockIdx.x * 16, wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int cb[1] = {(int)blockIdx.y * 32 + wave * 16};
  const int c1 = cb[0] + r;
  Weights<1, 3 * H> w1;
  load_weights(w + lw.u2t, 3 * H, cb, w1);
  float u[9], av[4];
#pragma unroll
  for (int k = 0; k < 9; ++k) u[k] = (w + lw.mix)[k];
#pragma unroll
  for (int k = 0; k < 4; ++k) av[k] = a_upd[(size_t)min(base + 4 * g + k, N - 1) * H + c1];
#pragma unroll
  for (int kb = 0; kb < PER; kb += kB) {
    float y0[kB], x0[kB], x1[kB], x2[kB], q0[kB], q1[kB], q2[kB];
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int idx = threadIdx.x + (kb + k) * kSplitBlock, m = idx / H, c = idx % H;
      const int i = min(base + m, N - 1);
      y0[k] = gs2[(size_t)i * H + c];
      if (gv2 != nullptr) {
        const float* vv = v_mid + (size_t)i * 3 * H;
        const float* gg = gv2 + (size_t)i * 3 * H;
        x0[k] = vv[c]; x1[k] = vv[H + c]; x2[k] = vv[2 * H + c];
        q0[k] = gg[c]; q1[k] = gg[H + c]; q2[k] = gg[2 * H + c];
      }
    }
#pragma unroll
    for (int k = 0; k < kB; ++k) {
      const int idx = threadIdx.x + (kb + k) * kSplitBlock, m = idx / H, c = idx % H;
      const bool in = base + m < N;
      float y1 = 0.f, y2 = 0.f;
      if (gv2 != nullptr) {
        y1 = dot3(q0[k], q1[k], q2[k], x0[k], x1[k], x2[k]);
        y2 = dot3(q0[k], q1[k], q2[k], dot3(u[0], u[1], u[2], x0[k], x1[k], x2[k]),
                  dot3(u[3], u[4], u[5], x0[k], x1[k], x2[k]),
                  dot3(u[6], u[7], u[8], x0[k], x1[k], x2[k]));
      }
      y_lds[m * LDY + c] = in ? y0[k] : 0.f;
      y_lds[m * LDY + H + c] = in ? y1 : 0.f;
      y_lds[m * LDY + 2 * H + c] = in ? y2 : 0.f;
    }
  }
  __syncthreads();
  f4 acc[1][1];
  zero_acc(acc);
  mma_regs(y_lds, LDY, w1, acc);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int i = base + 4 * g + k;
    if (i < N) ga[(size_t)i * H + c1] = acc[0][0][k] * silu_grad(av[k]);
  }
}

// gradient of the block's inputs from ga W1 and the gates
template <int H>
__global__ __launch_bounds__(kSplitBlock, 2) void update_input_bwd_kernel(
    int N, const float* __restrict__ w, LayerW lw, const float* __restrict__ gs2,
    const float* __restrict__ gv2, const float* __restrict__ v_mid, const float* __restrict__ ga,
    const float* __restrict__ g12, float* __restrict__ gs1, float* __restrict__ gv1) {
  constexpr int LDA = H + 4, PER = 16 * H / kSplitBlock;
  __shared__ __align__(16) float a_lds[16 * LDA];
  const int base = blockIdx.x * 16, wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int c = blockIdx.y * 32 + wave * 16 + r;
  const int cb[2] = {c - r, H + c - r};
  Weights<2, H> w1;
  load_weights(w + lw.u1t, H, cb, w1);
  float av[PER], u[9], s2[4], xv[4][3], t1[4], t2[4], q[4][3];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int idx = threadIdx.x + k * kSplitBlock, m = idx / H, cc = idx % H;
    av[k] = ga[(size_t)min(base + m, N - 1) * H + cc];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int i = min(base + 4 * g + k, N - 1);
    s2[k] = gs2[(size_t)i * H + c];
#pragma unroll
    for (int x = 0; x < 3; ++x) xv[k][x] = v_mid[((size_t)i * 3 + x) * H + c];
    if (gv2 != nullptr) {
      t1[k] = g12[(size_t)i * 2 * H + c];
      t2[k] = g12[(size_t)i * 2 * H + H + c];
#pragma unroll
      for (int x = 0; x < 3; ++x) q[k][x] = gv2[((size_t)i * 3 + x) * H + c];
    }
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) u[k] = (w + lw.mix)[k];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int idx = threadIdx.x + k * kSplitBlock, m = idx / H, cc = idx % H;
    a_lds[m * LDA + cc] = base + m < N ? av[k] : 0.f;
  }
  __syncthreads();
  f4 acc[1][2];
  zero_acc(acc);
  mma_regs(a_lds, LDA, w1, acc);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int i = base + 4 * g + k;
    if (i >= N) continue;
    gs1[(size_t)i * H + c] = s2[k] + acc[0][0][k];
    const float gn = acc[0][1][k], x0 = xv[k][0], x1 = xv[k][1], x2 = xv[k][2];
    const float n = norm3_exact(x0, x1, x2);
    const float sc = (n > 0.f) ? gn / n : 0.f;
    float o0 = sc * x0, o1 = sc * x1, o2 = sc * x2;
    if (gv2 != nullptr) {
      const float q0 = q[k][0], q1 = q[k][1], q2 = q[k][2];
      o0 = fma_(dot3(u[0], u[3], u[6], q0, q1, q2), t2[k], fma_(q0, t1[k], o0));
      o1 = fma_(dot3(u[1], u[4], u[7], q0, q1, q2), t2[k], fma_(q1, t1[k], o1));
      o2 = fma_(dot3(u[2], u[5], u[8], q0, q1, q2), t2[k], fma_(q2, t1[k], o2));
    }
    float* go = gv1 + (size_t)i * 3 * H;
    go[c] = o0;
    go[H + c] = o1;
    go[2 * H + c] = o2;
  }
}

// Partial dL/dd of a tile: (ga[:, k0:k0+KC] W1t[c0:c0+16, k0:k0+KC]^T) times
// de/dd for the 16 basis columns c0 + r, summed over those columns.
template <int RT, int KC, int TM>
__device__ __forceinline__ void gd_partial(const float* ga, int lda, const float* w1t, int ldb,
                                           int c0, int k0, const float* ed, float* out) {
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  int cb[1] = {c0};
  f4 acc[RT][1];
  zero_acc(acc);
  mma_tile_k<RT, 1, KC>(ga + k0, lda, w1t + k0, ldb, cb, acc);
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = rt * 16 + 4 * g + i;
      float t = acc[rt][0][i] * ed[m * kMaxRbf + c0 + r];
      t = group_sum<16>(t);
      if (r == 0) out[m] = t;
    }
}

// ---------------------------------------------------------------------------
// filter backward, kBwdPairs<H> pairs per tile.
// For pair p = (a < b): edge b->a carries s_b*Ws, v_b*Wv1 + u (x) Wv2 to a
// and edge a->b carries s_a*Ws, v_a*Wv1 - u (x) Wv2 to b, with
// u = (p_b - p_a)/(d + 1e-8).  The tile forms dL/dW_p from both directions,
// pushes it through W2^T, SiLU', W1^T to dL/de, then to dL/dd, and adds
// dL/du.  The running (dL/du, dL/dd) of all blocks is kept per pair; the
// last block processed turns it into dE/dvec.
// ---------------------------------------------------------------------------
// Pair indices of this thread's gather items of tile t (0 past the last tile
// or the last pair: those items are switched off by p >= P in the gather).
template <int TM, int C4, int NIT>
__device__ __forceinline__ void load_pair_indices(int t, int t1, int P,
                                                  const int32_t* __restrict__ pair_lo,
                                                  const int32_t* __restrict__ pair_hi,
                                                  int (&pa)[NIT], int (&pb)[NIT]) {
#pragma unroll
  for (int k = 0; k < NIT; ++k) {
    const int idx = threadIdx.x + k * kPairBlock;
    const int p = t * TM + idx / C4;
    const bool on = t < t1 && idx < TM * C4 && p < P;
    pa[k] = on ? pair_lo[p] : 0;
    pb[k] = on ? pair_hi[p] : 0;
  }
}

// PF: the pair indices of a thread's gather items of its next tile are loaded
// before the current tile's matrix products, so the next gather starts with
// its operand loads instead of a dependent index load (same arithmetic,
// bit-identical results).
template <int H, int TM, bool PF>
__global__ __launch_bounds__(kPairBlock, 4) void filter_bwd_kernel(
    const int32_t* __restrict__ counts, int32_t pcap, const int32_t* __restrict__ pair_lo,
    const int32_t* __restrict__ pair_hi, const float4* __restrict__ geom,
    const float* __restrict__ w, LayerW lw, const float* __restrict__ centers,
    const float* __restrict__ widths, int R, int RP, float rc, const float* __restrict__ Wf,
    const float* __restrict__ s_in, const float* __restrict__ v_in,
    const float* __restrict__ gs1, const float* __restrict__ gv1, float4* __restrict__ pacc,
    const int32_t* __restrict__ gate) {
  if (gate != nullptr && *gate == 0) return;
  constexpr int RT = TM / 16;
  constexpr int LDE = kMaxRbf + 4, LDG = 3 * H + 4, LDA = H + 4;
  constexpr int C4 = H / 4;                    // lanes per pair in the gather (4 channels each)
  constexpr int NPART = 1;                     // one dE/du partial per pair
  __shared__ __align__(16) float e_lds[TM * LDE];
  __shared__ __align__(16) float gw_lds[TM * LDG];
  __shared__ __align__(16) float ga_lds[TM * LDA];
  __shared__ float gu_lds[TM * NPART * 3];
  __shared__ float ed_lds[TM * kMaxRbf];       // d e_k / d d of each pair
  __shared__ float gd_lds[kPairWaves * TM];    // dL/dd partials, one set per wave
  __shared__ float mu_lds[kMaxRbf], gam_lds[kMaxRbf];
  __shared__ float d_lds[TM], fc_lds[TM], dfc_lds[TM];
  if (threadIdx.x < kMaxRbf) {
    const int k = threadIdx.x;
    mu_lds[k] = k < R ? centers[k] : 0.f;
    gam_lds[k] = k < R ? rbf_gamma(widths[k]) : 0.f;
  }
  const int P = min(counts[MLFF_COUNT_PAIRS], pcap);
  const int ntiles = (P + TM - 1) / TM;
  int t0, t1;
  int tstep;
  persistent_range(ntiles, t0, t1, tstep);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  constexpr int NIT = (TM * C4 + kPairBlock - 1) / kPairBlock;   // gather items per thread
  int pa[NIT], pb[NIT];
  if (PF) load_pair_indices<TM, C4, NIT>(t0, t1, P, pair_lo, pair_hi, pa, pb);
  for (int tile = t0; tile < t1; tile += tstep) {
    const int pbase = tile * TM;
    if (threadIdx.x < TM) {   // the cutoff once per pair
      const int p = pbase + threadIdx.x;
      float d = 0.f, fc = 0.f, dfc = 0.f;
      if (p < P) {
        d = geom[p].w;
        cosine_cutoff(d, rc, fc, dfc);
      }
      d_lds[threadIdx.x] = d;
      fc_lds[threadIdx.x] = fc;
      dfc_lds[threadIdx.x] = dfc;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < TM * RP; idx += kPairBlock) {
      const int m = idx / RP, k = idx - m * RP, p = pbase + m;
      float val = 0.f, der = 0.f;
      if (p < P && k < R)
        edge_feature_and_grad(d_lds[m], mu_lds[k], gam_lds[k], fc_lds[m], dfc_lds[m], val, der);
      e_lds[m * LDE + k] = val;
      ed_lds[m * kMaxRbf + k] = der;
    }
    // gather both endpoints, four channels per lane, every load of one item
    // issued up front (items one at a time: two blocks per CU fit the registers)
#pragma unroll 1
    for (int k = 0; k < NIT; ++k) {
      const int idx = threadIdx.x + k * kPairBlock;
      if (idx >= TM * C4) break;
      const int m = idx / C4, c = 4 * (idx - m * C4), p = pbase + m;
      f4 gws = {0.f, 0.f, 0.f, 0.f}, gwv1 = gws, gwv2 = gws;
      float gu0 = 0.f, gu1 = 0.f, gu2 = 0.f;
      if (p < P) {
        const int a = PF ? pa[k] : pair_lo[p], b = PF ? pb[k] : pair_hi[p];
        const float4 gm = geom[p];
        const float* va = v_in + (size_t)a * 3 * H + c;
        const float* vb = v_in + (size_t)b * 3 * H + c;
        const float* qa = gv1 + (size_t)a * 3 * H + c;
        const float* qb = gv1 + (size_t)b * 3 * H + c;
        const f4 sa = *reinterpret_cast<const f4*>(s_in + (size_t)a * H + c);
        const f4 sb = *reinterpret_cast<const f4*>(s_in + (size_t)b * H + c);
        const f4 ga = *reinterpret_cast<const f4*>(gs1 + (size_t)a * H + c);
        const f4 gb = *reinterpret_cast<const f4*>(gs1 + (size_t)b * H + c);
        const f4 va0 = *reinterpret_cast<const f4*>(va);
        const f4 va1 = *reinterpret_cast<const f4*>(va + H);
        const f4 va2 = *reinterpret_cast<const f4*>(va + 2 * H);
        const f4 vb0 = *reinterpret_cast<const f4*>(vb);
        const f4 vb1 = *reinterpret_cast<const f4*>(vb + H);
        const f4 vb2 = *reinterpret_cast<const f4*>(vb + 2 * H);
        const f4 qa0 = *reinterpret_cast<const f4*>(qa);
        const f4 qa1 = *reinterpret_cast<const f4*>(qa + H);
        const f4 qa2 = *reinterpret_cast<const f4*>(qa + 2 * H);
        const f4 qb0 = *reinterpret_cast<const f4*>(qb);
        const f4 qb1 = *reinterpret_cast<const f4*>(qb + H);
        const f4 qb2 = *reinterpret_cast<const f4*>(qb + 2 * H);
        const f4 wv2 = *reinterpret_cast<const f4*>(Wf + (size_t)p * 3 * H + 2 * H + c);
        const float den = gm.w + kEdgeEps;
        const float ux = gm.x / den, uy = gm.y / den, uz = gm.z / den;
        gws = ga * sb + gb * sa;
        gwv1 = qa0 * vb0 + qa1 * vb1 + qa2 * vb2 + qb0 * va0 + qb1 * va1 + qb2 * va2;
        const f4 d0 = qa0 - qb0, d1 = qa1 - qb1, d2 = qa2 - qb2;
        gwv2 = ux * d0 + uy * d1 + uz * d2;
        const f4 w0 = wv2 * d0, w1 = wv2 * d1, w2 = wv2 * d2;
        gu0 = (w0[0] + w0[1]) + (w0[2] + w0[3]);
        gu1 = (w1[0] + w1[1]) + (w1[2] + w1[3]);
        gu2 = (w2[0] + w2[1]) + (w2[2] + w2[3]);
      }
      *reinterpret_cast<f4*>(gw_lds + m * LDG + c) = gws;
      *reinterpret_cast<f4*>(gw_lds + m * LDG + H + c) = gwv1;
      *reinterpret_cast<f4*>(gw_lds + m * LDG + 2 * H + c) = gwv2;
      gu0 = group_sum<C4>(gu0);
      gu1 = group_sum<C4>(gu1);
      gu2 = group_sum<C4>(gu2);
      if (c == 0) {
        gu_lds[m * 3 + 0] = gu0;
        gu_lds[m * 3 + 1] = gu1;
        gu_lds[m * 3 + 2] = gu2;
      }
    }
    __syncthreads();
    if (PF) {   // the next tile's pair indices, in flight during the products below
      load_pair_indices<TM, C4, NIT>(tile + tstep, t1, P, pair_lo, pair_hi, pa, pb);
      __builtin_amdgcn_sched_barrier(0);
    }
    {
      // When the tile has at most one 16x16 output block per wave, each wave
      // takes one (row tile, column tile); otherwise every wave takes all row
      // tiles of its column tiles.  Each output element sums over K in the
      // same order either way.
      constexpr int CT = H / 16;
      constexpr bool kOneBlock = CT * RT <= kPairWaves;
      constexpr int RTW = kOneBlock ? 1 : RT;
      constexpr int NT = kOneBlock ? 1 : (CT + kPairWaves - 1) / kPairWaves;
      constexpr int NWB = kOneBlock ? CT * RT : CT / NT;
      if (wave < NWB) {
        const int r0 = kOneBlock ? wave / CT : 0;
        const int c0 = kOneBlock ? wave % CT : wave * NT;
        int cb[NT];
        f4 pre[RTW][NT], acc[RTW][NT];
#pragma unroll
        for (int ct = 0; ct < NT; ++ct) cb[ct] = (c0 + ct) * 16;
        zero_acc(pre);
        zero_acc(acc);
        mma_tile<RTW, NT>(e_lds + r0 * 16 * LDE, LDE, w + lw.f1w, RP, RP, cb, pre);
        mma_tile_k4<RTW, NT, 3 * H, 2, true>(gw_lds + r0 * 16 * LDG, LDG, w + lw.f2t, 3 * H, cb,
                                             acc);
        const float* b1 = w + lw.f1b;
#pragma unroll
        for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
          for (int ct = 0; ct < NT; ++ct) {
            const int c = cb[ct] + r;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const int m = (r0 + rt) * 16 + 4 * g + k;
              ga_lds[m * LDA + c] = acc[rt][ct][k] * silu_grad(pre[rt][ct][k] + b1[c]);
            }
          }
      }
    }
    __syncthreads();
    // dL/dd = sum_k (ga W1)_k de_k/dd.  All waves share the W1 product: wave
    // w takes basis columns 16 (w % ctiles) + r and the K (hidden) slice
    // w / ctiles; each multiplies its partial dL/de by de/dd, sums its 16
    // columns by shuffles, and the partials of all waves are added in wave
    // order below (the sum is linear in dL/de).
    const int ctiles = RP / 16;
    if (ctiles == 2) {
      constexpr int NP = (H / 16 < 4) ? H / 16 : 4, KC = H / NP;
      if (wave < 2 * NP) gd_partial<RT, KC, TM>(ga_lds, LDA, w + lw.f1t, H, (wave % 2) * 16,
                                                (wave / 2) * KC, ed_lds, gd_lds + wave * TM);
    } else {
      constexpr int NP = (H / 16 < 8) ? H / 16 : 8, KC = H / NP;
      if (wave < NP) gd_partial<RT, KC, TM>(ga_lds, LDA, w + lw.f1t, H, 0, wave * KC, ed_lds,
                                            gd_lds + wave * TM);
    }
    __syncthreads();
    if (threadIdx.x < TM) {
      const int m = threadIdx.x, p = pbase + m;
      if (p < P) {
        const int nparts = (RP > 16) ? 2 * ((H / 16 < 4) ? H / 16 : 4) : ((H / 16 < 8) ? H / 16 : 8);
        float gd = 0.f;
        for (int q = 0; q < nparts; ++q) gd += gd_lds[q * TM + m];
        float gx = 0.f, gy = 0.f, gz = 0.f;
#pragma unroll
        for (int part = 0; part < NPART; ++part) {
          gx += gu_lds[(m * NPART + part) * 3 + 0];
          gy += gu_lds[(m * NPART + part) * 3 + 1];
          gz += gu_lds[(m * NPART + part) * 3 + 2];
        }
        pacc[p] = make_float4(gx, gy, gz, gd);
      }
    }
    __syncthreads();
  }
}

// Gradient of pair p: its blocks' terms, from the last block to the first.
// Four blocks' loads are in flight at a time.
__device__ __forceinline__ float4 pair_sum(const float4* __restrict__ pacc, int32_t pcap, int L,
                                           int p, const float4& gm) {
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int lb = L - 1; lb >= 0; lb -= 4) {
    float4 t[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] = pacc[(size_t)max(lb - k, 0) * pcap + p];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (lb - k >= 0) { o.x += t[k].x; o.y += t[k].y; o.z += t[k].z; o.w += t[k].w; }
  }
  return pair_gradient(gm, o);
}

// Sums over one structure's atoms in FP64, in a fixed order: thread t of the
// workgroup takes atoms t, t + 256, ..., then lanes, then waves.  K values per
// atom: its energy and the nine entries of its virial.
template <int K>
__device__ __forceinline__ void structure_sums(int i0, int i1, const float* __restrict__ eps,
                                               const float* __restrict__ vir_atom,
                                               double (&acc)[K]) {
  __shared__ double sh[kBlock / 64][K];
  for (int k = 0; k < K; ++k) acc[k] = 0.0;
#pragma unroll 4
  for (int i = i0 + threadIdx.x; i < i1; i += kBlock) {
    acc[0] += (double)eps[i];
#pragma unroll
    for (int k = 1; k < K; ++k) acc[k] += (double)vir_atom[9 * (size_t)i + k - 1];
  }
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc[k] += __shfl_xor(acc[k], off, 64);
  if ((threadIdx.x & 63) == 0)
    for (int k = 0; k < K; ++k) sh[threadIdx.x >> 6][k] = acc[k];
  __syncthreads();
  for (int k = 0; k < K; ++k) acc[k] = (sh[0][k] + sh[1][k]) + (sh[2][k] + sh[3][k]);
}

// Forces F_i = sum_{j>i} G_p - sum_{j<i} G_p; per-atom virial sum_{j>i} vec (x) G.
// kGatherLanes lanes per atom take its edges in turn and add up at the end: with
// one thread per atom a row of 60 edges is 15 rounds of loads long (12.4 us in a
// launch of 60 atoms, 5.3 us so; 25 and 18 us in one of 10,000).  The workgroups past the atoms' add up the
// structures' energies (energy not null), which saves their launch.
constexpr int kGatherLanes = 32, kGatherAtoms = kBlock / kGatherLanes;

template <bool VIR>
__global__ __launch_bounds__(kBlock) void force_gather_kernel(
    int N, const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ col,
    const int32_t* __restrict__ edge_pair, int32_t ecap, const float4* __restrict__ pacc,
    int32_t pcap, int L, const float4* __restrict__ geom, float* __restrict__ forces,
    float* __restrict__ vir_atom, int B, const int32_t* __restrict__ mol_ptr,
    const float* __restrict__ eps, double* __restrict__ energy) {
  const int atom_blocks = (N + kGatherAtoms - 1) / kGatherAtoms;
  if ((int)blockIdx.x >= atom_blocks) {
    const int b = blockIdx.x - atom_blocks;
    double e[1];
    structure_sums<1>(mol_ptr[b], mol_ptr[b + 1], eps, nullptr, e);
    if (threadIdx.x == 0) energy[b] = e[0];
    return;
  }
  const int i = blockIdx.x * kGatherAtoms + threadIdx.x / kGatherLanes;
  const int lane = threadIdx.x % kGatherLanes;
  if (i >= N) return;
  constexpr int K = VIR ? 12 : 3;   // force, virial
  float o[K];
#pragma unroll
  for (int k = 0; k < K; ++k) o[k] = 0.f;
  const int e0 = min(row_ptr[i], ecap), e1 = min(row_ptr[i + 1], ecap);
  for (int e = e0 + lane; e < e1; e += kGatherLanes) {
    const int p = edge_pair[e];
    if (p < 0) continue;
    const float4 v = geom[p];
    const float4 G = pair_sum(pacc, pcap, L, p, v);
    if (col[e] > i) {
      o[0] += G.x; o[1] += G.y; o[2] += G.z;
      if constexpr (VIR) {
        o[3] += v.x * G.x; o[4] += v.x * G.y; o[5] += v.x * G.z;
        o[6] += v.y * G.x; o[7] += v.y * G.y; o[8] += v.y * G.z;
        o[9] += v.z * G.x; o[10] += v.z * G.y; o[11] += v.z * G.z;
      }
    } else {
      o[0] -= G.x; o[1] -= G.y; o[2] -= G.z;
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) o[k] = group_sum<kGatherLanes>(o[k]);
  if (lane != 0) return;
  if (forces != nullptr)
    for (int k = 0; k < 3; ++k) forces[3 * (size_t)i + k] = o[k];
  if constexpr (VIR)
    for (int k = 0; k < 9; ++k) vir_atom[9 * (size_t)i + k] = o[3 + k];
}

// per-structure FP64 sums (one workgroup per structure)
__global__ __launch_bounds__(kBlock) void reduce_kernel(const int32_t* __restrict__ mol_ptr,
                                                        const float* __restrict__ eps,
                                                        const float* __restrict__ vir_atom,
                                                        double* __restrict__ energy,
                                                        double* __restrict__ virial) {
  const int b = blockIdx.x;
  const int i0 = mol_ptr[b], i1 = mol_ptr[b + 1];
  if (vir_atom == nullptr) {
    double e[1];
    structure_sums<1>(i0, i1, eps, nullptr, e);
    if (threadIdx.x == 0 && energy != nullptr) energy[b] = e[0];
  } else {
    double a[10];
    structure_sums<10>(i0, i1, eps, vir_atom, a);
    if (threadIdx.x == 0) {
      if (energy != nullptr) energy[b] = a[0];
      for (int k = 0; k < 9; ++k) virial[9 * (size_t)b + k] = a[1 + k];
    }
  }
}

__global__ void copy_f32_kernel(int n, const float* __restrict__ src, float* __restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// bf16 planes of W2 [3H][H] of every block (dense in the blob); also clears the
// flag that the table kernels behind it raise
__global__ void split_filter_weights_kernel(const float* __restrict__ w, ModelW mw,
                                            uint16_t* __restrict__ wbf,
                                            int32_t* __restrict__ tab_bad) {
  if (tab_bad != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *tab_bad = 0;
  const int H = mw.H;
  const int64_t S = wbf_plane(H);
  const int64_t total = (int64_t)mw.L * S;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int l = (int)(idx / S);
    const int64_t e = idx % S;
    uint16_t h, m, lo;
    split3_bf16(w[mw.layer[l].f2w + e], h, m, lo);
    uint16_t* dst = wbf + wbf_f2w(H, l) + e;
    dst[0] = h;
    dst[S] = m;
    dst[2 * S] = lo;
  }
}

inline size_t nh(const Buffers& b) { return (size_t)b.N * b.H; }

// Launches in the plan's chosen shapes (Buffers::tile_fwd, tile_bwd,
// unroll_fwd, unroll_bwd; each is the default or its alternative).
// the direct filter kernels run: without tables, or beside tables not yet
// checked on the host (the flag picks one form)
bool direct_filters(const Buffers& b) { return !b.use_table || b.gate != nullptr; }

template <int H>
void launch_filter_fwd(const Buffers& b, hipStream_t st, int l) {
  const ModelW& mw = *b.mw;
  const float* centers = b.w + mw.centers;
  const float* widths = b.w + mw.widths;
  float* Wl = b.Wf + (size_t)l * b.pcap * 3 * H;
  const uint16_t* w2 = b.wbf + wbf_f2w(H, l);
  if (b.tile_fwd == kFwdPairsAlt<H>) {
    constexpr int TM = kFwdPairsAlt<H>;
    filter_fwd_kernel<H, TM><<<pair_grid(b, TM), kPairBlock, 0, st>>>(
        b.geom, b.counts, b.pcap, b.w, mw.layer[l], centers, widths, b.R, mw.RP, b.rc, Wl, w2,
        b.gate);
  } else {
    constexpr int TM = kFwdPairs<H>;
    filter_fwd_kernel<H, TM><<<pair_grid(b, TM), kPairBlock, 0, st>>>(
        b.geom, b.counts, b.pcap, b.w, mw.layer[l], centers, widths, b.R, mw.RP, b.rc, Wl, w2,
        b.gate);
  }
}

template <int H>
void launch_filter_bwd(const Buffers& b, hipStream_t st, int l) {
  const ModelW& mw = *b.mw;
  const float* centers = b.w + mw.centers;
  const float* widths = b.w + mw.widths;
  const float* Wl = b.Wf + (size_t)l * b.pcap * 3 * H;
  const float* Sl = b.S + (size_t)l * nh(b);
  const float* Vl = b.V + (size_t)l * 3 * nh(b);
  const float* gS1 = b.gS1 + (size_t)l * nh(b);
  const float* gV1 = b.gV1 + (size_t)l * 3 * nh(b);
  float4* pacc = b.pacc + (size_t)l * b.pcap;
  if (b.tile_bwd == kBwdPairsAlt<H>) {
    constexpr int TM = kBwdPairsAlt<H>;
    filter_bwd_kernel<H, TM, false><<<pair_grid(b, TM), kPairBlock, 0, st>>>(
        b.counts, b.pcap, b.pair_lo, b.pair_hi, b.geom, b.w, mw.layer[l], centers, widths, b.R,
        mw.RP, b.rc, Wl, Sl, Vl, gS1, gV1, pacc, b.gate);
  } else if (b.bwd_variant == 1) {
    constexpr int TM = kBwdPairs<H>;
    filter_bwd_kernel<H, TM, true><<<pair_grid(b, TM), kPairBlock, 0, st>>>(
        b.counts, b.pcap, b.pair_lo, b.pair_hi, b.geom, b.w, mw.layer[l], centers, widths, b.R,
        mw.RP, b.rc, Wl, Sl, Vl, gS1, gV1, pacc, b.gate);
  } else {
    constexpr int TM = kBwdPairs<H>;
    filter_bwd_kernel<H, TM, false><<<pair_grid(b, TM), kPairBlock, 0, st>>>(
        b.counts, b.pcap, b.pair_lo, b.pair_hi, b.geom, b.w, mw.layer[l], centers, widths, b.R,
        mw.RP, b.rc, Wl, Sl, Vl, gS1, gV1, pacc, b.gate);
  }
}

template <int H, bool FWD>
void launch_message(const Buffers& b, hipStream_t st, int l, const float* s_in, const float* v_in,
                    float* s_out, float* v_out) {
  constexpr int U0 = FWD ? kMsgUnrollFwd : kMsgUnrollBwd;
  constexpr int U1 = FWD ? kMsgUnrollFwdAlt : kMsgUnrollBwdAlt;
  const float* Wl = b.Wf + (size_t)l * b.pcap * 3 * H;
  auto run = [&](auto kernel, int rows_per_block, int block) {
    const int grid = ((b.N + rows_per_block - 1) / rows_per_block + 7) / 8 * 8;
    kernel<<<grid, block, 0, st>>>(b.N, b.row_ptr, b.col, b.edge_pair, b.ecap, b.unit, Wl, s_in,
                                   v_in, s_out, v_out);
  };
  auto shapes = [&](auto zero) {
    constexpr bool Z = decltype(zero)::value;
    if (b.N <= kMsgSplitAtoms)
      run(message_kernel<H, FWD, U0, true, Z>, 1, kMsgSums * H);
    else if ((FWD ? b.unroll_fwd : b.unroll_bwd) == U1)
      run(message_kernel<H, FWD, U1, false, Z>, kBlock / H, kBlock);
    else
      run(message_kernel<H, FWD, U0, false, Z>, kBlock / H, kBlock);
  };
  if constexpr (FWD) {
    if (l == 0 && zero_vectors(b)) return shapes(std::true_type{});
  }
  shapes(std::false_type{});
}

// Atom-side launches: the split or small forms for few atoms (kSplitAtoms,
// kSmallTileAtoms), 32-atom tiles above.  Same bits.
template <int H>
void launch_update_fwd(const Buffers& b, hipStream_t s, const LayerW& lw, const float* s_mid,
                       const float* v_mid, float* s_out, float* v_out, float* a_upd, float* g12,
                       bool gates) {
  if (b.N <= kSplitAtoms) {
    const dim3 grid((b.N + 15) / 16, H / 32);
    auto kernel = gates ? update_fwd_split_kernel<H, true> : update_fwd_split_kernel<H, false>;
    kernel<<<grid, 4 * H, 0, s>>>(b.N, b.w, lw, s_mid, v_mid, s_out, v_out, a_upd, g12);
  } else {
    auto run = [&](auto kernel, int tm) {
      kernel<<<(b.N + tm - 1) / tm, kUpdBlock, 0, s>>>(b.N, b.w, lw, s_mid, v_mid, s_out, v_out,
                                                       a_upd, g12);
    };
    if (b.N <= kSmallTileAtoms)
      run(gates ? update_fwd_kernel<H, 16, true> : update_fwd_kernel<H, 16, false>, 16);
    else
      run(gates ? update_fwd_kernel<H, 32, true> : update_fwd_kernel<H, 32, false>, 32);
  }
}

template <int H>
void launch_readout(const Buffers& b, hipStream_t s) {
  const float* sL = b.S + (size_t)b.L * nh(b);
  if (b.N <= kSmallTileAtoms)
    readout_kernel<H, 16><<<(b.N + 15) / 16, kBlock, 0, s>>>(b.N, b.w, *b.mw, sL, b.eps, b.gS0);
  else
    readout_kernel<H, 32><<<(b.N + 31) / 32, kBlock, 0, s>>>(b.N, b.w, *b.mw, sL, b.eps, b.gS0);
}

template <int H>
void launch_update_bwd(const Buffers& b, hipStream_t s, int l, const float* gs2,
                       const float* gv2) {
  const LayerW& lw = b.mw->layer[l];
  const float* vm = b.Vmid + (size_t)l * 3 * nh(b);
  const float* au = b.Aupd + (size_t)l * nh(b);
  const float* g12 = b.G12 + (size_t)l * 2 * nh(b);
  float* gs1 = b.gS1 + (size_t)l * nh(b);
  float* gv1 = b.gV1 + (size_t)l * 3 * nh(b);
  if (b.N <= kSplitAtoms) {
    const dim3 grid((b.N + 15) / 16, H / 32);
    update_hidden_bwd_kernel<H><<<grid, kSplitBlock, 0, s>>>(b.N, b.w, lw, gs2, gv2, vm, au, b.gA);
    update_input_bwd_kernel<H><<<grid, kSplitBlock, 0, s>>>(b.N, b.w, lw, gs2, gv2, vm, b.gA, g12,
                                                            gs1, gv1);
  } else {
    auto run = [&](auto kernel, int tm) {
      kernel<<<(b.N + tm - 1) / tm, kUpdBlock, 0, s>>>(b.N, b.w, lw, gs2, gv2, vm, au, g12, gs1,
                                                       gv1);
    };
    if (b.N <= kSmallTileAtoms) run(update_bwd_kernel<H, 16>, 16);
    else run(update_bwd_kernel<H, 32>, 32);
  }
}

void launch_force_gather(const Buffers& b, hipStream_t s, float* forces, bool want_virial,
                         double* energy) {
  const int grid = (b.N + kGatherAtoms - 1) / kGatherAtoms + (energy != nullptr ? b.B : 0);
  if (grid == 0) return;
  auto run = [&](auto kernel, float* vir_atom) {
    kernel<<<grid, kBlock, 0, s>>>(b.N, b.row_ptr, b.col, b.edge_pair, b.ecap, b.pacc, b.pcap, b.L,
                                   b.geom, forces, vir_atom, b.B, b.mol_ptr, b.eps, energy);
  };
  if (want_virial) run(force_gather_kernel<true>, b.vir_atom);
  else run(force_gather_kernel<false>, nullptr);
}

// Fork/join between the caller's stream and the filter stream.  Events order
// the two streams both eagerly and under graph capture (a wait on an event
// recorded in a capturing stream pulls the other stream into the capture).
struct Streams {
  hipStream_t main, filt;
  hipEvent_t* ev;
  hipError_t err = hipSuccess;
  Streams(const Buffers& b, hipStream_t s) : main(s), filt(b.aux ? b.aux : s), ev(b.ev) {}
  bool two() const { return filt != main; }
  // `to` waits for everything issued so far on `from`
  void order(hipStream_t from, hipStream_t to, int k) {
    if (!two() || err != hipSuccess) return;
    err = hipEventRecord(ev[k], from);
    if (err == hipSuccess) err = hipStreamWaitEvent(to, ev[k], 0);
  }
};

template <int H>
hipError_t forward_impl(const Buffers& b, hipStream_t s) {
  const ModelW& mw = *b.mw;
  const int N = b.N;
  const float* centers = b.w + mw.centers;
  const float* widths = b.w + mw.widths;
  Streams st(b, s);
  // the filters depend on the pair geometry only: all L of them run on the
  // filter stream while the caller's stream walks the atom-side chain
  st.order(s, st.filt, 0);
  const bool one = b.use_table && !st.two();
  if (one) launch_filter_table_fwd<H>(b, s, 0, b.L, true);
  for (int l = 0; l < b.L; ++l) {
    if (b.use_table && st.two()) launch_filter_table_fwd<H>(b, st.filt, l, l + 1, false);
    if (direct_filters(b)) launch_filter_fwd<H>(b, st.filt, l);
    if (st.two() && st.err == hipSuccess) st.err = hipEventRecord(b.ev[1 + l], st.filt);
  }
  if (!one) {
    const int total = N * (H / 4);
    embed_kernel<H><<<(unsigned)((total + kBlock - 1) / kBlock), kBlock, 0, s>>>(
        N, b.numbers, b.w + mw.emb, b.S, b.V);
  }
  for (int l = 0; l < b.L; ++l) {
    const LayerW& lw = mw.layer[l];
    if (st.two() && st.err == hipSuccess) st.err = hipStreamWaitEvent(s, b.ev[1 + l], 0);
    float* Sl = b.S + (size_t)l * nh(b);
    float* Vl = b.V + (size_t)l * 3 * nh(b);
    float* Sm = b.Smid + (size_t)l * nh(b);
    float* Vm = b.Vmid + (size_t)l * 3 * nh(b);
    launch_message<H, true>(b, s, l, Sl, Vl, Sm, Vm);
    launch_update_fwd<H>(b, s, lw, Sm, Vm, b.S + (size_t)(l + 1) * nh(b),
                         b.V + (size_t)(l + 1) * 3 * nh(b), b.Aupd + (size_t)l * nh(b),
                         b.G12 + (size_t)l * 2 * nh(b), l + 1 < b.L);
  }
  launch_readout<H>(b, s);
  if (st.err != hipSuccess) return st.err;
  return hipGetLastError();
}

template <int H>
hipError_t backward_impl(const Buffers& b, hipStream_t s, float* forces, bool want_virial,
                         double* energy) {
  const ModelW& mw = *b.mw;
  const int N = b.N;
  const float* centers = b.w + mw.centers;
  const float* widths = b.w + mw.widths;
  Streams st(b, s);
  // gradient w.r.t. the update outputs of the last block: (gS0, 0)
  float* gs2 = b.gS0;
  float* gv2 = nullptr;
  for (int l = b.L - 1; l >= 0; --l) {
    const LayerW& lw = mw.layer[l];
    // block l's message gradient has a slice of its own, so the filter
    // adjoint of block l (filter stream) and the message adjoint of block l
    // and update adjoint of block l-1 (caller's stream) run side by side
    float* gS1 = b.gS1 + (size_t)l * nh(b);
    float* gV1 = b.gV1 + (size_t)l * 3 * nh(b);
    launch_update_bwd<H>(b, s, l, gs2, gv2);
    st.order(s, st.filt, b.L + 1 + l);
    if (b.use_table && st.two()) launch_filter_table_bwd<H>(b, st.filt, l, l + 1);
    if (direct_filters(b)) launch_filter_bwd<H>(b, st.filt, l);
    if (l > 0) {
      launch_message<H, false>(b, s, l, gS1, gV1, b.gS0, b.gV0);
      gs2 = b.gS0;
      gv2 = b.gV0;
    }
  }
  // on one stream all blocks' adjoints go in one launch
  if (b.use_table && !st.two()) launch_filter_table_bwd<H>(b, s, 0, b.L);
  st.order(st.filt, s, 2 * b.L + 1);
  launch_force_gather(b, s, forces, want_virial, energy);
  if (st.err != hipSuccess) return st.err;
  return hipGetLastError();
}

template <int H>
hipError_t stage_impl(const Buffers& b, hipStream_t s, int stage, int l) {
  const ModelW& mw = *b.mw;
  const int N = b.N;
  const float* centers = b.w + mw.centers;
  const float* widths = b.w + mw.widths;
  const LayerW& lw = mw.layer[l];
  switch (stage) {
    case MLFF_STAGE_FILTER_FWD:
      if (b.use_table) launch_filter_table_fwd<H>(b, s, l, l + 1, false);
      if (direct_filters(b)) launch_filter_fwd<H>(b, s, l);
      break;
    case MLFF_STAGE_MESSAGE_FWD:
      launch_message<H, true>(b, s, l, b.S + (size_t)l * nh(b),
                              b.V + (size_t)l * 3 * nh(b), b.Smid + (size_t)l * nh(b),
                              b.Vmid + (size_t)l * 3 * nh(b));
      break;
    case MLFF_STAGE_UPDATE_FWD:
      launch_update_fwd<H>(b, s, lw, b.Smid + (size_t)l * nh(b), b.Vmid + (size_t)l * 3 * nh(b),
                           b.S + (size_t)(l + 1) * nh(b), b.V + (size_t)(l + 1) * 3 * nh(b),
                           b.Aupd + (size_t)l * nh(b), b.G12 + (size_t)l * 2 * nh(b),
                           l + 1 < b.L);
      break;
    case MLFF_STAGE_READOUT:
      launch_readout<H>(b, s);
      break;
    case MLFF_STAGE_UPDATE_BWD:
      // reads gS0/gV0, writes block l's slice of gS1/gV1
      launch_update_bwd<H>(b, s, l, b.gS0, (l == b.L - 1) ? nullptr : b.gV0);
      break;
    case MLFF_STAGE_FILTER_BWD:
      if (b.use_table) launch_filter_table_bwd<H>(b, s, l, l + 1);
      if (direct_filters(b)) launch_filter_bwd<H>(b, s, l);
      break;
    case MLFF_STAGE_MESSAGE_BWD:
      // no evaluation runs block 0's, so its Wv1 columns may not be there
      if (l == 0 && zero_vectors(b)) launch_filter_table_fwd<H>(b, s, 0, 1, false, true);
      launch_message<H, false>(b, s, l, b.gS1 + (size_t)l * nh(b),
                               b.gV1 + (size_t)l * 3 * nh(b), b.gS0, b.gV0);
      break;
    case MLFF_STAGE_FORCES:
      launch_force_gather(b, s, nullptr, true, nullptr);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

int default_shape(int H, int which) {
  switch (which) {
    case 0: return H <= 32 ? kFwdPairs<32> : kFwdPairs<128>;
    case 1: return H <= 32 ? kBwdPairs<32> : kBwdPairs<128>;
    case 2: return kMsgUnrollFwd;
    case 3: return kMsgUnrollBwd;
    case 4: return 0;
    default: return 0;
  }
}

int alternative_shape(int H, int which) {
  switch (which) {
    case 0: return H <= 32 ? kFwdPairsAlt<32> : kFwdPairsAlt<128>;
    case 1: return H <= 32 ? kBwdPairsAlt<32> : kBwdPairsAlt<128>;
    case 2: return kMsgUnrollFwdAlt;
    case 3: return kMsgUnrollBwdAlt;
    case 4: return 1;
    default: return 0;
  }
}

int shapes_used(const Buffers& b) {
  return (direct_filters(b) ? 1 << 0 | 1 << 1 | 1 << 4 : 0) |
         (b.N > kMsgSplitAtoms ? 1 << 2 | 1 << 3 : 0);
}

hipError_t prepare_filters(const Buffers& b, hipStream_t s) {
  if (b.wbf == nullptr || b.L < 1) return hipSuccess;
  split_filter_weights_kernel<<<256, 256, 0, s>>>(b.w, *b.mw, b.wbf, b.tab_bad);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && b.tab != nullptr) e = build_tables(b, s);
  return e;
}

hipError_t launch_stage(const Buffers& b, hipStream_t s, int stage, int layer) {
  if (layer < 0 || layer >= b.L) return hipErrorInvalidValue;
  switch (b.H) {
    case 32: return stage_impl<32>(b, s, stage, layer);
    case 64: return stage_impl<64>(b, s, stage, layer);
    case 128: return stage_impl<128>(b, s, stage, layer);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_forward(const Buffers& b, hipStream_t s) {
  switch (b.H) {
    case 32: return forward_impl<32>(b, s);
    case 64: return forward_impl<64>(b, s);
    case 128: return forward_impl<128>(b, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_backward(const Buffers& b, hipStream_t s, float* forces, bool want_virial,
                           double* energy) {
  switch (b.H) {
    case 32: return backward_impl<32>(b, s, forces, want_virial, energy);
    case 64: return backward_impl<64>(b, s, forces, want_virial, energy);
    case 128: return backward_impl<128>(b, s, forces, want_virial, energy);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_reduce(const Buffers& b, hipStream_t s, double* energy, double* virial,
                         float* atom_energy) {
  if (b.B > 0 && (energy != nullptr || virial != nullptr))
    reduce_kernel<<<b.B, kBlock, 0, s>>>(b.mol_ptr, b.eps, virial ? b.vir_atom : nullptr,
                                         energy, virial);
  if (atom_energy != nullptr && b.N > 0)
    copy_f32_kernel<<<(b.N + 255) / 256, 256, 0, s>>>(b.N, b.eps, atom_energy);
  return hipGetLastError();
}

}  // namespace mlff
