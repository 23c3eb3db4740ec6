// Directed edges grouped by an endpoint, for the interaction blocks on a
// caller-given edge list (student_model.py:346-387: index_add_ over the
// receivers, and over the sources in its adjoint).
//
// A stable counting sort: count per atom, scan, place through an atomic cursor,
// then every row is put into ascending edge order, so the result does not
// depend on the order of the atomics.  Bound by its launches at 40,000 edges;
// a stable 64-bit key sort, histogram, scan and four range reductions of torch
// took 300 us for both groupings there, this takes 30.

#include "common.hpp"
#include "internal.hpp"

namespace mlff {
namespace {

constexpr int kCsrBlock = 256;
constexpr int kRegRow = 64;      // rows up to here are ranked in a wave's registers
constexpr int kRankRow = 2048;   // up to here by comparisons with the whole row, above by a scan
                                 // over all edges (there are at most E / kRankRow such rows)

// list l (blockIdx.y): 0 grouped by receiver, 1 by source
__global__ __launch_bounds__(kCsrBlock) void csr_zero_kernel(int N, int lists,
                                                             int32_t* __restrict__ row_ptr,
                                                             int32_t* __restrict__ cursor,
                                                             int32_t* __restrict__ bad) {
  const int i = blockIdx.x * kCsrBlock + threadIdx.x;
  if (i < lists * (N + 1)) row_ptr[i] = 0;
  if (i < lists * N) cursor[i] = 0;
  if (i == 0) *bad = 0;
}

// counts into row_ptr[key + 1]; an edge with an endpoint outside [0, N) raises
// the flag and is left out of the lists
__global__ __launch_bounds__(kCsrBlock) void csr_count_kernel(
    int E, int N, int lists, const int64_t* __restrict__ src, const int64_t* __restrict__ dst,
    int32_t* __restrict__ ends, int32_t* __restrict__ row_ptr, int32_t* __restrict__ bad) {
  const int e = blockIdx.x * kCsrBlock + threadIdx.x;
  if (e >= E) return;
  const int64_t s = src[e], d = dst[e];
  const bool ok = s >= 0 && s < N && d >= 0 && d < N;
  ends[e] = ok ? (int32_t)d : -1;
  ends[(size_t)E + e] = ok ? (int32_t)s : -1;
  if (!ok) {
    *bad = 1;
    return;
  }
  atomicAdd(&row_ptr[d + 1], 1);
  if (lists > 1) atomicAdd(&row_ptr[N + 1 + s + 1], 1);
}

// inclusive scan of a list's counts in place, one workgroup per list
__global__ __launch_bounds__(1024) void csr_scan_kernel(int N, int32_t* __restrict__ row_ptr) {
  __shared__ int wsum[16];
  int32_t* p = row_ptr + (size_t)blockIdx.x * (N + 1) + 1;
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  int base = 0;
  for (int b = 0; b < N; b += 1024) {
    const int i = b + t;
    int v = i < N ? p[i] : 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int u = __shfl_up(v, off, 64);
      if (lane >= off) v += u;
    }
    if (lane == 63) wsum[wv] = v;
    __syncthreads();
    int before = base, all = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      if (q < wv) before += wsum[q];
      all += wsum[q];
    }
    if (i < N) p[i] = v + before;
    base += all;
    __syncthreads();
  }
}

__global__ __launch_bounds__(kCsrBlock) void csr_place_kernel(
    int E, int N, const int32_t* __restrict__ ends, const int32_t* __restrict__ row_ptr,
    int32_t* __restrict__ cursor, int32_t* __restrict__ placed) {
  const int e = blockIdx.x * kCsrBlock + threadIdx.x, l = blockIdx.y;
  if (e >= E) return;
  const int k = ends[(size_t)l * E + e];
  if (k < 0) return;
  const int slot = row_ptr[(size_t)l * (N + 1) + k] + atomicAdd(&cursor[(size_t)l * N + k], 1);
  placed[(size_t)l * E + slot] = e;
}

// One wave per row: the row's edges in ascending order, and their other ends.
__global__ __launch_bounds__(kCsrBlock) void csr_rows_kernel(
    int E, int N, const int32_t* __restrict__ ends, const int32_t* __restrict__ row_ptr,
    const int32_t* __restrict__ placed, int32_t* __restrict__ col, int32_t* __restrict__ eid) {
  const int i = (int)(((int64_t)blockIdx.x * kCsrBlock + threadIdx.x) >> 6), l = blockIdx.y;
  const int lane = threadIdx.x & 63;
  if (i >= N) return;
  const int32_t* key = ends + (size_t)l * E;
  const int32_t* other = ends + (size_t)(1 - l) * E;
  const int lo = row_ptr[(size_t)l * (N + 1) + i];
  const int n = row_ptr[(size_t)l * (N + 1) + i + 1] - lo;
  placed += (size_t)l * E + lo;
  col += (size_t)l * E + lo;
  eid += (size_t)l * E + lo;
  if (n <= kRegRow) {
    const int v = lane < n ? placed[lane] : 0x7fffffff;
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += (__shfl(v, j, 64) < v) ? 1 : 0;
    if (lane < n) {
      eid[rank] = v;
      col[rank] = other[v];
    }
  } else if (n <= kRankRow) {
    for (int b = 0; b < n; b += 64) {
      const int v = b + lane < n ? placed[b + lane] : 0x7fffffff;
      int rank = 0;
      for (int q = 0; q < n; q += 64) {
        const int u = q + lane < n ? placed[q + lane] : 0x7fffffff;
#pragma unroll 8
        for (int j = 0; j < 64; ++j) rank += (__shfl(u, j, 64) < v) ? 1 : 0;
      }
      if (b + lane < n) {
        eid[rank] = v;
        col[rank] = other[v];
      }
    }
  } else {
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    int k = 0;
    for (int b = 0; b < E; b += 64) {
      const int e = b + lane;
      const bool h = e < E && key[e] == i;
      const uint64_t m = __ballot(h);
      if (h) {
        const int slot = k + __popcll(m & below);
        eid[slot] = e;
        col[slot] = other[e];
      }
      k += __popcll(m);
    }
  }
}

// (row, column) of every entry of a CSR list as int64, one wave per row
__global__ __launch_bounds__(kCsrBlock) void edge_index_kernel(int N, int E,
                                                               const int32_t* __restrict__ row_ptr,
                                                               const int32_t* __restrict__ col,
                                                               int64_t* __restrict__ out) {
  const int i = (int)(((int64_t)blockIdx.x * kCsrBlock + threadIdx.x) >> 6);
  if (i >= N) return;
  const int e1 = min(row_ptr[i + 1], E);
  for (int e = row_ptr[i] + (int)(threadIdx.x & 63); e < e1; e += 64) {
    out[e] = i;
    out[(size_t)E + e] = col[e];
  }
}

}  // namespace
}  // namespace mlff

using namespace mlff;

extern "C" int mlff_edge_index(void* stream, int n_atoms, int n_edges, const int32_t* row_ptr_dev,
                               const int32_t* col_dev, int64_t* edge_index_dev) {
  if (n_atoms < 0 || n_edges < 0) {
    set_error("mlff_edge_index: invalid sizes");
    return MLFF_ERR_INVALID;
  }
  if (n_atoms == 0 || n_edges == 0) return MLFF_OK;
  if (!row_ptr_dev || !col_dev || !edge_index_dev) {
    set_error("mlff_edge_index: null pointer");
    return MLFF_ERR_INVALID;
  }
  const int blocks = (int)(((int64_t)n_atoms * 64 + kCsrBlock - 1) / kCsrBlock);
  edge_index_kernel<<<blocks, kCsrBlock, 0, static_cast<hipStream_t>(stream)>>>(
      n_atoms, n_edges, row_ptr_dev, col_dev, edge_index_dev);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("mlff_edge_index: %s", hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}

extern "C" int mlff_edge_csr(void* stream, int n_edges, int n_atoms, int lists,
                             const int64_t* src_dev, const int64_t* dst_dev, int32_t* row_ptr_dev,
                             int32_t* col_dev, int32_t* edge_id_dev, int32_t* ends_dev,
                             int32_t* scratch_dev, int32_t* bad_dev) {
  if (n_edges < 0 || n_atoms < 0 || n_atoms > (1 << 29) || lists < 1 || lists > 2) {
    set_error("mlff_edge_csr: invalid sizes");
    return MLFF_ERR_INVALID;
  }
  if (!row_ptr_dev || !scratch_dev || !bad_dev ||
      (n_edges > 0 && (!src_dev || !dst_dev || !col_dev || !edge_id_dev || !ends_dev))) {
    set_error("mlff_edge_csr: null pointer");
    return MLFF_ERR_INVALID;
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int E = n_edges, N = n_atoms;
  int32_t* cursor = scratch_dev;
  int32_t* placed = scratch_dev + (size_t)lists * N;
  const int zero = lists * (N + 1);
  csr_zero_kernel<<<(zero + kCsrBlock - 1) / kCsrBlock, kCsrBlock, 0, st>>>(N, lists, row_ptr_dev,
                                                                            cursor, bad_dev);
  if (E > 0) {
    const int eb = (int)(((int64_t)E + kCsrBlock - 1) / kCsrBlock);
    csr_count_kernel<<<eb, kCsrBlock, 0, st>>>(E, N, lists, src_dev, dst_dev, ends_dev,
                                               row_ptr_dev, bad_dev);
    if (N > 0) {
      csr_scan_kernel<<<lists, 1024, 0, st>>>(N, row_ptr_dev);
      csr_place_kernel<<<dim3(eb, lists), kCsrBlock, 0, st>>>(E, N, ends_dev, row_ptr_dev, cursor,
                                                              placed);
      const int rb = (int)(((int64_t)N * 64 + kCsrBlock - 1) / kCsrBlock);
      csr_rows_kernel<<<dim3(rb, lists), kCsrBlock, 0, st>>>(E, N, ends_dev, row_ptr_dev, placed,
                                                             col_dev, edge_id_dev);
    }
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("mlff_edge_csr: %s", hipGetErrorString(e));
    return MLFF_ERR_HIP;
  }
  return MLFF_OK;
}
