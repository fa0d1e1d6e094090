// Declarations shared by the GEMM sources: the groups of a call, what a
// launch of the matrix-core kernels is given, and which tile a workgroup takes.
#pragma once

#include "tl_common.h"

namespace tlg {

// Products that share A (q/k/v, gate/up): C_g = A . B_g, B_g (k x n_g), for
// g < count, run as one tile space in one launch.  tile0[g] is group g's
// first tile in that space (tile0[count] = all tiles); col0[g] its first
// column in the concatenated width (the split-K partials).
constexpr int kMaxGroups = 4;
struct GemmGroups {
  int count;
  const void* b[kMaxGroups];
  void* c[kMaxGroups];
  int n[kMaxGroups];
  int64_t ldb[kMaxGroups], ldc[kMaxGroups];
  int tile0[kMaxGroups + 1];
  int col0[kMaxGroups + 1];
};

// The group whose tiles (or columns, with col0) include t.
__device__ __forceinline__ int find_group(const int (&first)[kMaxGroups + 1], int count, int t) {
  int g = 0;
#pragma unroll
  for (int i = 1; i < kMaxGroups; ++i)
    if (i < count && t >= first[i]) g = i;
  return g;
}

struct GemmParams {
  const void* a;
  int m, k;
  int64_t lda;
  GemmGroups G;   // tile0 counts the kernel's tiles of C
  int tiles_m, per_xcd;
  int vec_store;  // bit g: C_g's rows and base allow vector stores (16 bytes whole, 4 columns where K is split)
  // Split K (ksplit > 1): item (slice s, tile t) covers stages
  // [s kt_per, (s + 1) kt_per) and stores its fp32 partial tile at
  // ws + ws_off[g] + (s m + row) n_g + col; split_reduce_kernel sums them.
  int ksplit, kt_per;
  float* ws;
  int64_t ws_off[kMaxGroups];
};

// Bytes from a view's first element to the end of its last: what a buffer
// resource over it may reach.  rows * ld instead would pass the end of the
// allocation where the view is the last columns of wider rows, and a tile that is
// only partly inside the view reads there.
__host__ __device__ __forceinline__ uint32_t view_bytes(int64_t rows, int64_t ld, int64_t cols, int esize) {
  return rows > 0 ? (uint32_t)(((rows - 1) * ld + cols) * esize) : 0u;
}

// Work item of workgroup L: each XCD (workgroups are dealt to the 8 XCDs in
// turn) takes a contiguous run of items, so the workgroups an XCD runs at once
// share their B column tiles and A row tiles in its L2; items are slice-major (all
// tiles of K-slice 0, then slice 1).  A group's tiles are taken in panels of up to
// kPanelRows row tiles, rows fastest, so that the tiles an XCD runs at once (32)
// stay near 8 x 4 whatever the product's height.
constexpr int kPanelRows = 8;
__device__ __forceinline__ bool gemm_tile(const GemmParams& p, int& grp, int& tm, int& tn, int& ks) {
  const int L = blockIdx.x;
  const int it = (L % 8) * p.per_xcd + L / 8;
  const int tiles = p.G.tile0[p.G.count];
  if (it >= tiles * p.ksplit) return false;
  ks = p.ksplit > 1 ? it / tiles : 0;
  const int t = it - ks * tiles;
  grp = find_group(p.G.tile0, p.G.count, t);
  const int local = t - p.G.tile0[grp];
  // no more divisions than the height needs: each is a chain of some 30 instructions
  // ahead of the first load
  if (p.tiles_m == 1) {
    tm = 0;
    tn = local;
  } else if (p.tiles_m <= kPanelRows) {
    tn = local / p.tiles_m;
    tm = local - tn * p.tiles_m;
  } else {
    const int tiles_n = (p.G.tile0[grp + 1] - p.G.tile0[grp]) / p.tiles_m;
    const int panel = local / (kPanelRows * tiles_n);
    const int in = local - panel * kPanelRows * tiles_n;
    const int h = min(kPanelRows, p.tiles_m - panel * kPanelRows);
    tm = panel * kPanelRows + in % h;
    tn = in / h;
  }
  return true;
}

}  // namespace tlg
