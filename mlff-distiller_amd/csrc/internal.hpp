// Internal declarations shared by the kernel translation units and the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mlff_amd.h"
#include "common.hpp"

namespace mlff {

// Per-interaction-block weight offsets (floats into the packed blob).
struct LayerW {
  int64_t f1w, f1b, f1t;   // filter Linear(R,H): W [H][RP], b [H], W^T [RP][H]
  int64_t f2w, f2b, f2t;   // filter Linear(H,3H): W [3H][H], b [3H], W^T [H][3H]
  int64_t u1w, u1b, u1t;   // update Linear(2H,H): W [H][2H], b [H], W^T [2H][H]
  int64_t u2w, u2b, u2t;   // update Linear(H,3H): W [3H][H], b [3H], W^T [H][3H]
  int64_t mix;             // mixing matrix [3][3]
};

struct ModelW {
  int H, L, R, RP, HP2, HP4, max_z;
  int64_t emb, centers, widths;
  int64_t r1w, r1b, r1t;   // Linear(H, H/2): [HP2][H], b [HP2], W^T [H][HP2]
  int64_t r2w, r2b, r2t;   // Linear(H/2, H/4): [HP4][HP2], b [HP4], W^T [HP2][HP4]
  int64_t r3w, r3b;        // Linear(H/4, 1): w [HP4], b [1] (stored padded to 16)
  LayerW layer[8];
  int64_t total;
};

int build_layout(int H, int L, int R, int max_z, ModelW* mw, mlff_slot* slots, int max_slots,
                 int* n_slots);

// Neighbour-list launches (nl.hip).
constexpr int kSmallAtoms = 4096;   // largest list that is counted and filled in two launches
constexpr int kCellRowMax = 256;    // cell-list rows up to here are kept from the count pass
struct NLArgs {
  const float* pos; int N; int B;
  const int32_t* mol_ptr; const int32_t* atom_mol;
  const float* cells; const uint8_t* pbc; float rc;
  int32_t* deg; int32_t* udeg; int32_t* row_ptr; int32_t* pair_ptr;
  int32_t* col; int32_t* edge_shift; int32_t* edge_pair; int32_t ecap;
  int32_t* pair_lo; int32_t* pair_hi; int32_t* pair_shift; float4* geom; float4* unit; int32_t pcap;
  int32_t* counts;
  // cell list (periodic structures): grid[b] = {nc0, nc1, nc2, base}, nc0 == 0 -> brute force
  const int4* grid; int32_t n_cells;
  int32_t* cell_count; int32_t* cell_start; int32_t* cell_atoms; int32_t* atom_cell;
  uint64_t* mask;            // [N][ceil(N / 64)] hit masks; null: none
  int32_t* hits;             // [N][kCellRowMax] neighbours of the cell-list rows, unsorted
  int32_t* edge_tmp_shift;   // [ecap*3] image shifts of cell-list rows before sorting
};
hipError_t launch_neighbor_list(const NLArgs& a, hipStream_t s, bool build_pairs);

// Distance tables of the filter MLP (filter_table.hip): K intervals of width
// h for W', Kc of width 2h for W, over [0, rc] of every block.
constexpr int64_t kTableMaxBytes = 64ll << 20;   // per plan; larger: direct product only
struct TableShape {
  double h;
  int K, Kc;
  int64_t d_off, layer_floats;      // floats: start of the W' part, size of a block's table
  int64_t bytes;                    // all blocks; 0: no table for this configuration
};
TableShape table_shape(int H, int R, int L, float rc);

// One block's table as a kernel reads it.
struct TableView {
  const float* w;                   // [Kc+1][2][C]: W, 2h W'
  const float* d;                   // [K+1][2][C]: W', h W''
  float inv, inv_c;                 // 1/h, 1/(2h): powers of two
  int K, Kc;
};
__host__ __device__ inline TableView table_view(const TableShape& t, const float* tab, int l,
                                                int C) {
  const float* w = tab + l * t.layer_floats;
  return TableView{w, w + t.d_off, (float)(1.0 / t.h), (float)(0.5 / t.h), t.K, t.Kc};
}
// Interval k of distance d and the weights of its cubic Hermite interpolant
//   f0 + h01 (f1 - f0) + h10 g0 + h11 g1
// of the knot values f and scaled slopes g.  inv is a power of two, so x, k
// and t carry no rounding.
struct TableAt {
  int k;
  float h01, h10, h11;
};
__device__ __forceinline__ TableAt table_at(float d, float inv, int K) {
  const float x = d * inv;
  const int k = min((int)x, K - 1);
  const float t = x - (float)k, u = 1.f - t;
  return TableAt{k, t * t * (3.f - 2.f * t), t * u * u, -t * t * u};
}
// The fused operations are spelled out here and in the message terms, so that
// every kernel that evaluates them gets the same bits.
template <typename T>
__device__ __forceinline__ T hermite(const TableAt& a, const T& f0, const T& g0, const T& f1,
                                     const T& g1) {
  return f0 + fma_(a.h01, f1 - f0, fma_(a.h10, g0, a.h11 * g1));
}

// Model launches (painn.hip).
struct Buffers {
  int N, B, H, L, R;
  float rc;
  int32_t ecap, pcap;
  int blocks;                       // persistent grid for pair kernels
  // launch shapes: pairs per filter tile (forward, adjoint) and edges in
  // flight per message row (forward, adjoint); default_shape() or
  // alternative_shape() of each
  int tile_fwd, tile_bwd, unroll_fwd, unroll_bwd;
  int bwd_variant;    // filter adjoint: 0 plain, 1 next-tile pair-index prefetch
  const float* w;                   // weight blob
  const ModelW* mw;
  // bf16 three-plane copies of the filter's second layer, per block l:
  // W2 [3H][H] at wbf + wbf_f2w(l); plane stride 3H^2
  uint16_t* wbf;
  // filter tables of every block, and the flag their guard raises.  use_table:
  // the pair kernels read the tables; gate (not null): they were not checked
  // on the host yet, so both forms are launched and the flag picks one
  TableShape ts;
  float* tab;
  int32_t* tab_bad;
  bool use_table;
  const int32_t* gate;
  const int64_t* numbers;
  const int32_t* mol_ptr;
  const int32_t* atom_mol;
  const float* cells;
  int32_t* counts;
  const int32_t* row_ptr; const int32_t* col; const int32_t* edge_pair;
  const int32_t* pair_lo; const int32_t* pair_hi; const int32_t* pair_shift;
  const float4* geom;               // {p_hi - p_lo, d}
  const float4* unit;               // {(p_hi - p_lo) / (d + eps), d}
  float4* pacc;                     // [L][pcap]: per pair and block (dE/du, dE/dd)
  float* Wf;                        // [L][pcap][3H]
  float* S; float* V;               // [L+1][N][H], [L+1][N][3][H]
  float* Smid; float* Vmid;         // [L][N][H], [L][N][3][H]
  float* Aupd; float* G12;          // [L][N][H], [L][N][2H]
  float* gS0; float* gV0;           // gradient w.r.t. the update outputs of the block below
  float* gS1; float* gV1;           // [L][N][H], [L][N][3][H]: gradient w.r.t. message outputs
  float* gA;                        // [N][H]: hidden gradient of the split update adjoint
  float* eps;                       // [N]
  float* vir_atom;                  // [N][9]
  // second stream for the filter kernels (overlaps the memory-bound message
  // kernels); ev holds 3L+2 events.  aux == nullptr: one stream.
  hipStream_t aux;
  hipEvent_t* ev;
};
// The first block reads neither its vectors, which are zero, nor what multiplies
// them (Wv1 and its derivative).  Only with checked tables: the check fails for
// infinities and NaN in a filter, whose products with zero are no zeros.
inline bool zero_vectors(const Buffers& b) { return b.use_table && b.gate == nullptr; }
__host__ __device__ inline int64_t wbf_plane(int H) { return 3 * (int64_t)H * H; }
__host__ __device__ inline int64_t wbf_f2w(int H, int l) { return (int64_t)l * 3 * wbf_plane(H); }
__host__ __device__ inline int64_t wbf_elems(int H, int L) { return (int64_t)L * 3 * wbf_plane(H); }
// Launch shapes (which: 0 filter-forward pairs per tile, 1 filter-adjoint
// pairs per tile, 2 message-forward edges in flight, 3 message-adjoint edges
// in flight, 4 filter-adjoint variant, default tile only): the default for
// hidden size H and the pre-instantiated alternative (kind 4: the highest
// variant number; every value up to it exists).
int default_shape(int H, int which);
int alternative_shape(int H, int which);
// bit k: the launches of an evaluation read the shape of kind k
int shapes_used(const Buffers& b);
// What the pair kernels read beside the weight blob, remade on stream s for
// new weights: the filters' bf16 planes and their tables with the guard's flag.
hipError_t prepare_filters(const Buffers& b, hipStream_t s);
// Fill and check every block's table (tab_bad must be 0 before).
hipError_t build_tables(const Buffers& b, hipStream_t s);
// Blocks l0 ... l1 - 1 in one launch; embed: the atoms' first features too; all: the
// columns too that the first block has no use for (zero_vectors).
template <int H>
void launch_filter_table_fwd(const Buffers& b, hipStream_t s, int l0, int l1, bool embed,
                             bool all = false);
template <int H>
void launch_filter_table_bwd(const Buffers& b, hipStream_t s, int l0, int l1);
hipError_t launch_forward(const Buffers& b, hipStream_t s);
// energy (may be null): the structures' sums too, in the last launch
hipError_t launch_backward(const Buffers& b, hipStream_t s, float* forces, bool want_virial,
                           double* energy);
// One model stage (mlff_stage 1..8) of block `layer`, on the workspace as the
// last full evaluation left it.
hipError_t launch_stage(const Buffers& b, hipStream_t s, int stage, int layer);
hipError_t launch_reduce(const Buffers& b, hipStream_t s, double* energy, double* virial,
                         float* atom_energy);

// MD launches (md.hip).
// counts (may be null): the step counter is advanced here, by the steps of the run;
// launch_vv_second then writes the rows of the step `back` before it and, with turn,
// starts the next step
hipError_t launch_vv_first(int N, double* x, double* p, const double* inv_mass, const float* F,
                           float* pos32, double dt, int32_t* counts, int advance,
                           hipStream_t s);
hipError_t launch_vv_second(int N, int B, const int32_t* mol_ptr, double* p,
                            const double* inv_mass, const float* F, double dt,
                            const double* epot, double* ledger, int ledger_len,
                            const int32_t* counts, int back, bool turn, double* x,
                            float* pos32, double* fx, double* fp, float* fF, int n_frames,
                            hipStream_t s);

hipError_t launch_mts_kick(int N, double* p, const float* Fa, const float* Fb, double coef,
                           hipStream_t s);
hipError_t launch_mts_select(int N, const int32_t* atom_mol, const uint8_t* flag,
                             const float* F_full, const float* F_fast, float* F_in,
                             hipStream_t s);
hipError_t launch_mts_disagree(int N, const int32_t* atom_mol, const float* F_full,
                               const float* F_fast, float* dis_max, hipStream_t s);
hipError_t launch_mts_ledger(int B, const int32_t* mol_ptr, const double* p,
                             const double* inv_mass, const double* epot, double* ledger,
                             int ledger_len, int32_t* counts, hipStream_t s);

// S0 = emb[Z] and V0 = 0, four channels per item: item t of an atom's H/4
// writes S0 channels 4t..4t+3 and the same channels of the three V0 components
// (16-byte stores; rows are 16-byte aligned since H % 4 == 0)
template <int H>
__device__ __forceinline__ void embed_item(int idx, const int64_t* __restrict__ Z,
                                           const float* __restrict__ emb, float* __restrict__ S0,
                                           float* __restrict__ V0) {
  constexpr int Q = H / 4;
  const int i = idx / Q, c = idx % Q;
  const float4 e = reinterpret_cast<const float4*>(emb + Z[i] * H)[c];
  reinterpret_cast<float4*>(S0)[idx] = e;
  float4* v = reinterpret_cast<float4*>(V0) + (size_t)i * 3 * Q + c;
  const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
  v[0] = z;
  v[Q] = z;
  v[2 * Q] = z;
}

void set_error(const char* fmt, ...);

}  // namespace mlff
