// Dense projections of the model step: C = A . B on the library stream.
//
// Reference behaviour being replaced: triton_llm/kernels/gemm.py:14-108, a
// Triton fp32 tile GEMM (64 x 64 x 32 blocks, tl.dot) used for every
// projection of the model (q/k/v/o, gate/up/down, lm_head).
//
// Two regimes:
//   * a prompt (m > kSkinnyMaxM rows) is a compute-bound GEMM on the matrix
//     cores with fp32 accumulation: gemm_wide_kernel (tl_gemm_wide.hip) for the
//     16-bit types, gemm_f32_kernel (tl_gemm_f32.hip) for fp32, the simple
//     fp32-FMA gemm_simple_kernel where rows are not 16-byte aligned.
//     A batch of decoded tokens (a few dozen rows) has too few tiles to fill
//     the device: K is split into slices with fp32 partials and a reduce pass;
//   * a decoded token (m <= kSkinnyMaxM rows) reads every weight once for a
//     handful of multiply-adds per element: an HBM-bound skinny product,
//     where rocBLAS measured 0.4-0.7 TB/s.  skinny_partial_kernel cuts B
//     into (64-column x TK-row) tiles, about a thousand of them, so enough
//     weight bytes are in flight to stream at HBM speed; each tile's
//     partial sums go to the workspace and skinny_reduce_kernel adds the
//     K-slices and rounds to the output type.
#include "tl_gemm.h"
#include "tl_gemm_plan.h"

using namespace tlg;

namespace {

constexpr int kSkinnyMaxM = 8;     // rows of A handled by the skinny path
constexpr int kMaxSplit = 32;      // K-slices at most of a matrix-core product
constexpr int kSkThreads = 256;    // 4 waves
constexpr int kSkUnroll = 16;      // row loads in flight per lane
constexpr int kSkMaxTk = 1024;     // rows per K-slice at most (A's slice is staged in LDS)
constexpr int kSkRowsPerStep = 16; // rows one workgroup load instruction round covers
constexpr int kSkTargetTiles = 1024;
constexpr int kAuxNt = 2;          // buffer-load cache policy: nontemporal (weights are read once)

bool fits_int(int64_t x) { return x >= 0 && x <= INT32_MAX; }

// Skinny tiling: 64 fp32 (or 128 16-bit) columns per tile -- 16 lanes x 16
// bytes per row -- and TK rows, TK a multiple of the 16 rows one workgroup
// load round covers, chosen for about kSkTargetTiles tiles.  (A slice that
// ends inside an unrolled step loads zeros past its end, with no memory
// access.)
struct SkinnyPlan {
  int cols;     // columns per tile
  int n_tiles;  // column tiles
  int tk;       // rows per K-slice
  int ks;       // K-slices
};

SkinnyPlan skinny_plan(const GemmGroups& G, int k, int esize) {
  SkinnyPlan s;
  s.cols = 256 / esize;
  s.n_tiles = 0;
  for (int g = 0; g < G.count; ++g) s.n_tiles += (G.n[g] + s.cols - 1) / s.cols;
  const int step = kSkRowsPerStep;
  const int ks_target = kSkTargetTiles / s.n_tiles > 1 ? kSkTargetTiles / s.n_tiles : 1;
  int tk = (k + ks_target - 1) / ks_target;
  tk = (tk + step - 1) / step * step;
  tk = tk < kSkMaxTk ? tk : kSkMaxTk;
  s.tk = tk;
  s.ks = (k + tk - 1) / tk;
  return s;
}

size_t skinny_workspace_bytes(int m, const GemmGroups& G, int k, int esize) {
  const SkinnyPlan s = skinny_plan(G, k, esize);
  if (s.ks == 1) return 0;  // single K-slice: stored to C directly
  size_t ntot = 0;
  for (int g = 0; g < G.count; ++g) ntot += (size_t)G.n[g];
  return (size_t)s.ks * m * ntot * sizeof(float);
}

template <typename T>
__device__ __forceinline__ void unpack_words(const u32x4& w, float (&f)[16 / T::size]) {
  if constexpr (T::size == 4) {
    f[0] = __uint_as_float(w.x); f[1] = __uint_as_float(w.y); f[2] = __uint_as_float(w.z); f[3] = __uint_as_float(w.w);
  } else {
    unpack2<T>(w.x, f[0], f[1]); unpack2<T>(w.y, f[2], f[3]); unpack2<T>(w.z, f[4], f[5]); unpack2<T>(w.w, f[6], f[7]);
  }
}

// One workgroup: K-slice blockIdx.y (rows [k0, k0 + tk)) x column tile
// blockIdx.x of the groups' tile space.  Lane (wave w, row group r = lane / 16, chunk c = lane % 16)
// reads 16 bytes of row k0 + 16 i + 4 w + r, columns chunk c; its MT x CPC
// sums cover the rows it read.  The four row groups of a wave, then the four
// waves, are added up and the slice's partial product is stored.
// With a single K-slice (gridDim.y == 1) the sums are the result: they are
// rounded and stored to C directly, and no reduce pass follows.
template <typename T, int MT>
__global__ __launch_bounds__(kSkThreads) void skinny_partial_kernel(const void* __restrict__ a, GemmGroups G,
                                                                     float* __restrict__ ws, int m, int k, int64_t lda,
                                                                     int ntot, int tk) {
  constexpr int CPC = 16 / T::size;  // columns per 16-byte chunk
  constexpr int COLS = 16 * CPC;     // columns per tile
  using Bits = typename T::bits;
  __shared__ float s_a[MT][kSkMaxTk];
  __shared__ float s_sum[4][MT][COLS];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int r = lane >> 4, c = lane & 15;
  const int k0 = blockIdx.y * tk;
  const int k1 = min(k, k0 + tk);
  const int grp = find_group(G.tile0, G.count, blockIdx.x);
  const void* b = G.b[grp];
  const int n = G.n[grp];
  const int64_t ldb = G.ldb[grp];
  // The tile's rows of B as one buffer that ends at the last row's last
  // column inside the matrix: loads of rows past the slice read zeros with no
  // memory access.  (Chunks past column n of earlier rows read the next
  // row's data; those columns are never stored.)
  const int tile_col0 = (blockIdx.x - G.tile0[grp]) * COLS;
  const Bits* bbase = (const Bits*)b + (int64_t)k0 * ldb + tile_col0;
  const int rows = k1 - k0;
  const int last_cols = min(COLS, n - tile_col0);
  const uint32_t nbytes = (uint32_t)((int64_t)(rows - 1) * ldb * T::size + (int64_t)last_cols * T::size);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)bbase, (short)0, (int)nbytes, kBufRsrcWord3);
  const uint32_t row_bytes = (uint32_t)(ldb * T::size);
  float acc[MT][CPC];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CPC; ++j) acc[i][j] = 0.f;
  u32x4 w[kSkUnroll];
  auto load_round = [&](int kb) {
#pragma unroll
    for (int u = 0; u < kSkUnroll; ++u) {
      const int row = kb + kSkRowsPerStep * u + 4 * wave + r;  // row within the slice
      w[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)row * row_bytes + (uint32_t)(c * 16), 0, kAuxNt));
    }
  };
  // The first round's weight loads go out before A's slice is staged, so
  // the two latencies overlap.
  load_round(0);
  for (int idx = tid; idx < MT * rows; idx += kSkThreads) {
    const int mi = idx / rows, kk = idx - mi * rows;
    s_a[mi][kk] = mi < m ? to_f32<T>(((const Bits*)a)[(int64_t)mi * lda + k0 + kk]) : 0.f;
  }
  __syncthreads();
  for (int kb = 0; kb < rows; kb += kSkRowsPerStep * kSkUnroll) {
    if (kb > 0) load_round(kb);
#pragma unroll
    for (int u = 0; u < kSkUnroll; ++u) {
      float f[CPC];
      unpack_words<T>(w[u], f);
      const int kk = kb + kSkRowsPerStep * u + 4 * wave + r;
      if (kk < rows) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const float x = s_a[i][kk];
#pragma unroll
          for (int j = 0; j < CPC; ++j) acc[i][j] = fmaf(x, f[j], acc[i][j]);
        }
      }
    }
  }
  // Row groups of the wave (lanes 16 apart), then the waves through LDS.
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CPC; ++j) {
      float v = acc[i][j];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      acc[i][j] = v;
    }
  __syncthreads();
  if (r == 0) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < CPC; ++j) s_sum[wave][i][c * CPC + j] = acc[i][j];
  }
  __syncthreads();
  for (int idx = tid; idx < MT * COLS; idx += kSkThreads) {
    const int mi = idx / COLS, cc = idx % COLS;
    const int col = tile_col0 + cc;
    if (mi < m && col < n) {
      const float v = s_sum[0][mi][cc] + s_sum[1][mi][cc] + s_sum[2][mi][cc] + s_sum[3][mi][cc];
      if (gridDim.y == 1)
        ((Bits*)G.c[grp])[(int64_t)mi * G.ldc[grp] + col] = from_f32<T>(v);
      else
        ws[((int64_t)blockIdx.y * m + mi) * ntot + G.col0[grp] + col] = v;
    }
  }
}

// One or two decoded tokens against a short K: a whole column tile (8 lanes x 16
// bytes) per workgroup of 16 waves, the waves' row groups covering all of K with
// every load in flight at once, so the product is one launch and one round trip
// to memory.  Latency-bound.  With K-slices the same product took two launches
// and two round trips: SmolLM2-360M fp32 at one token, rotated weights, o 8.8 ->
// 5.0 us, q/k/v 7.8 -> 6.3, gate/up 9.8 -> 8.7; two tokens o 9.3 -> 6.1.  K of
// 2560 takes three rounds and lost (9.3 -> 11.5 us), and so do four or more rows
// of 16-bit weights (10.1 -> 11.5): their unpacking is not spread over enough
// workgroups.  Narrower tiles read lines in parts: q/k/v 8.6 us with 16 bytes a row.
constexpr int kWholeThreads = 1024;
constexpr int kWholeChunks = 8;                                     // lanes across a row
constexpr int kWholeUnroll = 8;                                     // loads in flight per lane
constexpr int kWholeMaxK = kWholeThreads / kWholeChunks * kWholeUnroll;  // 1024: one round
constexpr int kWholeMaxTiles = 256;                                 // one token; a quarter of it for two

template <typename T, int MT>
__global__ __launch_bounds__(kWholeThreads) void skinny_whole_kernel(const void* __restrict__ a, GemmGroups G, int m, int k,
                                                                     int64_t lda, int per_xcd) {
  constexpr int CW = kWholeChunks;
  constexpr int CPC = 16 / T::size;  // columns per 16-byte chunk
  constexpr int COLS = CW * CPC;     // columns per tile
  constexpr int RW = 64 / CW;        // rows a wave's load covers
  constexpr int WV = kWholeThreads / 64;
  using Bits = typename T::bits;
  __shared__ float s_a[MT][kWholeMaxK];
  __shared__ float s_sum[WV][MT * COLS];
  // adjacent tiles on one XCD: their lines meet in its L2
  const int t = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (t >= G.tile0[G.count]) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane % CW, r = lane / CW;
  const int grp = find_group(G.tile0, G.count, t);
  const int n = G.n[grp];
  const int64_t ldb = G.ldb[grp];
  const int col0 = (t - G.tile0[grp]) * COLS;
  const uint32_t nbytes = (uint32_t)((int64_t)(k - 1) * ldb * T::size + (int64_t)min(COLS, n - col0) * T::size);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)((const Bits*)G.b[grp] + col0), (short)0,
                                                                      (int)nbytes, kBufRsrcWord3);
  const uint32_t row_bytes = (uint32_t)(ldb * T::size);
  u32x4 w[kWholeUnroll];
#pragma unroll
  for (int u = 0; u < kWholeUnroll; ++u)  // rows past k: zeros, with no memory access
    w[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
        rs, (uint32_t)(RW * (WV * u + wave) + r) * row_bytes + (uint32_t)(c * 16), 0, 0));
  for (int idx = tid; idx < MT * k; idx += kWholeThreads) {
    const int mi = idx / k, kk = idx - mi * k;
    s_a[mi][kk] = mi < m ? to_f32<T>(((const Bits*)a)[(int64_t)mi * lda + kk]) : 0.f;
  }
  float acc[MT][CPC];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CPC; ++j) acc[i][j] = 0.f;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kWholeUnroll; ++u) {
    const int kk = RW * (WV * u + wave) + r;
    float f[CPC];
    unpack_words<T>(w[u], f);
    if (kk < k) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const float x = s_a[i][kk];
#pragma unroll
        for (int j = 0; j < CPC; ++j) acc[i][j] = fmaf(x, f[j], acc[i][j]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < CPC; ++j) {
      float v = acc[i][j];
#pragma unroll
      for (int d = CW; d < 64; d <<= 1) v += __shfl_xor(v, d);
      if (r == 0) s_sum[wave][i * COLS + c * CPC + j] = v;
    }
  __syncthreads();
  for (int idx = tid; idx < MT * COLS; idx += kWholeThreads) {
    const int mi = idx / COLS, col = col0 + idx % COLS;
    float v[WV];
#pragma unroll
    for (int q = 0; q < WV; ++q) v[q] = s_sum[q][idx];
#pragma unroll
    for (int d = WV / 2; d >= 1; d /= 2)  // by halves: four roundings where a chain has sixteen
#pragma unroll
      for (int q = 0; q < d; ++q) v[q] += v[q + d];
    if (mi < m && col < n) ((Bits*)G.c[grp])[(int64_t)mi * G.ldc[grp] + col] = from_f32<T>(v[0]);
  }
}

// C_g[mi][col] = sum over K-slices of the partials, rounded to T, for every
// column of the concatenated width.  The sum is latency-bound: up to
// kReduceBatch slices' loads are in flight at once (one round trip for the
// usual 4-24 slices), added in slice order.
constexpr int kReduceBatch = 32;  // measured: SmolLM2-360M one-token layer 41.0 -> 37.5 us against 8
template <typename T>
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float* __restrict__ ws, GemmGroups G, int m, int ntot,
                                                            int ks) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (int64_t)m * ntot) return;
  const int mi = (int)(idx / ntot), colg = (int)(idx % ntot);
  const int grp = find_group(G.col0, G.count, colg);
  const int64_t stride = (int64_t)m * ntot;
  float s = 0.f;
  for (int q0 = 0; q0 < ks; q0 += kReduceBatch) {
    float v[kReduceBatch];
#pragma unroll
    for (int j = 0; j < kReduceBatch; ++j) v[j] = q0 + j < ks ? ws[(int64_t)(q0 + j) * stride + idx] : 0.f;
#pragma unroll
    for (int j = 0; j < kReduceBatch; ++j) s += v[j];
  }
  ((typename T::bits*)G.c[grp])[(int64_t)mi * G.ldc[grp] + (colg - G.col0[grp])] = from_f32<T>(s);
}

template <typename T>
int launch_skinny(const void* a, GemmGroups G, int m, int k, int64_t lda, void* ws, bool in_place, hipStream_t st) {
  if (m <= 2 && k <= kWholeMaxK && !in_place) {
    constexpr int cols = kWholeChunks * (16 / T::size);
    int64_t tiles = 0;
    for (int g = 0; g < G.count; ++g) tiles += (G.n[g] + cols - 1) / cols;
    if (tiles <= (m == 1 ? kWholeMaxTiles : kWholeMaxTiles / 4)) {
      G.tile0[0] = 0;
      for (int g = 0; g < G.count; ++g) G.tile0[g + 1] = G.tile0[g] + (G.n[g] + cols - 1) / cols;
      const int per_xcd = (G.tile0[G.count] + 7) / 8;
      const dim3 grid((unsigned)(8 * per_xcd)), block(kWholeThreads);
      if (m == 1)
        hipLaunchKernelGGL((skinny_whole_kernel<T, 1>), grid, block, 0, st, a, G, m, k, lda, per_xcd);
      else
        hipLaunchKernelGGL((skinny_whole_kernel<T, 2>), grid, block, 0, st, a, G, m, k, lda, per_xcd);
      return tl_launch_status();
    }
  }
  const SkinnyPlan s = skinny_plan(G, k, T::size);
  int ntot = 0;
  G.tile0[0] = 0;
  G.col0[0] = 0;
  for (int g = 0; g < G.count; ++g) {
    G.tile0[g + 1] = G.tile0[g] + (G.n[g] + s.cols - 1) / s.cols;
    G.col0[g + 1] = G.col0[g] + G.n[g];
    ntot += G.n[g];
  }
  dim3 grid((unsigned)s.n_tiles, (unsigned)s.ks);
  float* w = (float*)ws;
  if (m <= 1)
    hipLaunchKernelGGL((skinny_partial_kernel<T, 1>), grid, dim3(kSkThreads), 0, st, a, G, w, m, k, lda, ntot, s.tk);
  else if (m <= 2)
    hipLaunchKernelGGL((skinny_partial_kernel<T, 2>), grid, dim3(kSkThreads), 0, st, a, G, w, m, k, lda, ntot, s.tk);
  else if (m <= 4)
    hipLaunchKernelGGL((skinny_partial_kernel<T, 4>), grid, dim3(kSkThreads), 0, st, a, G, w, m, k, lda, ntot, s.tk);
  else
    hipLaunchKernelGGL((skinny_partial_kernel<T, 8>), grid, dim3(kSkThreads), 0, st, a, G, w, m, k, lda, ntot, s.tk);
  int e = tl_launch_status();
  if (e || s.ks == 1) return e;
  const int64_t outs = (int64_t)m * ntot;
  hipLaunchKernelGGL((skinny_reduce_kernel<T>), dim3((unsigned)((outs + 255) / 256)), dim3(256), 0, st,
                     (const float*)ws, G, m, ntot, s.ks);
  return tl_launch_status();
}

// Split-K finish: C_g = sum over the K-slices of the fp32 partial tiles
// (slice 0 first, so the result does not depend on timing), rounded to T.
// One 4-column run per thread, grid-stride; blockIdx.y = group.
template <typename T>
__global__ __launch_bounds__(256) void split_reduce_kernel(GemmParams p) {
  using Bits = typename T::bits;
  const int g = blockIdx.y;
  const int n = p.G.n[g];
  const int q4 = n / 4;
  const int runs = p.m * q4;
  const float* w = p.ws + p.ws_off[g];
  const int64_t slice = (int64_t)p.m * n;
  Bits* c = (Bits*)p.G.c[g];
  const int64_t ldc = p.G.ldc[g];
  const bool vec = (p.vec_store >> g) & 1;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < runs; i += gridDim.x * 256) {
    const int r = i / q4;
    const int col = (i - r * q4) * 4;
    f32x4 sum = *(const f32x4*)(w + (int64_t)r * n + col);
    for (int ks = 1; ks < p.ksplit; ++ks) sum += *(const f32x4*)(w + ks * slice + (int64_t)r * n + col);
    Bits* dst = c + (int64_t)r * ldc + col;
    if constexpr (T::size == 4) {
      if (vec) {
        *(f32x4*)dst = sum;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = from_f32<T>(sum[e]);
      }
    } else {
      const float x0[2] = {sum[0], sum[1]}, x1[2] = {sum[2], sum[3]};
      if (vec) {
        *(u32x2*)dst = u32x2{pack2<T>(x0), pack2<T>(x1)};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e] = from_f32<T>(sum[e]);
      }
    }
  }
}

// Any shape and alignment (the MFMA kernels need 16-byte aligned rows):
// 64 x 64 tiles of C_g (g = blockIdx.z), 256 threads with 4 x 4 outputs
// each, fp32 FMA over 16-deep K slices staged in LDS with bounds checks.
// Used for small or odd shapes only.
template <typename T>
__global__ __launch_bounds__(256) void gemm_simple_kernel(GemmParams p) {
  using Bits = typename T::bits;
  __shared__ float sa[16][65];
  __shared__ float sb[16][65];
  const int grp = blockIdx.z;
  const int n_g = p.G.n[grp];
  const Bits* bg = (const Bits*)p.G.b[grp];
  const int64_t ldb = p.G.ldb[grp];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  if (n0 >= n_g) return;  // the grid spans the widest group
  float acc[4][4] = {};
  for (int k0 = 0; k0 < p.k; k0 += 16) {
    for (int i = threadIdx.x; i < 16 * 64; i += 256) {
      const int kk = i / 64, mm = i % 64;
      const int m = m0 + mm, k = k0 + kk;
      sa[kk][mm] = (m < p.m && k < p.k) ? to_f32<T>(((const Bits*)p.a)[(int64_t)m * p.lda + k]) : 0.f;
      const int n = n0 + mm;
      sb[kk][mm] = (n < n_g && k < p.k) ? to_f32<T>(bg[(int64_t)k * ldb + n]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(sa[kk][ty * 4 + i], sb[kk][tx * 4 + j], acc[i][j]);
    __syncthreads();
  }
  Bits* cg = (Bits*)p.G.c[grp];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < p.m && n < n_g) cg[(int64_t)m * p.G.ldc[grp] + n] = from_f32<T>(acc[i][j]);
    }
}

// K-slices whose fp32 partials are about half as large as B in 16 bits, as large as
// B in fp32: B is what a product of few rows streams.
int few_rows_split(int m, int k, int esize) {
  return esize == 2 ? (int)(((int64_t)k + 4 * (int64_t)m - 1) / (4 * (int64_t)m)) : k / m;
}

// The most K-slices a plan may choose: those, 32 at most; of an fp32 product, whose
// matrix-core time outweighs the partials' traffic at any height, four.
int max_split(int m, int k, int esize) {
  const int few = few_rows_split(m, k, esize), least = esize == 4 ? 4 : 1;
  return few > kMaxSplit ? kMaxSplit : few > least ? few : least;
}

PromptPlan prompt_plan(int m, int k, const GemmGroups& G, int esize, int min_split, int max_split) {
  PromptPlan P{};
  if (esize == 4) {
    const F32Plan f = gemm_f32_plan(m, k, G, min_split, max_split);
    P.tm = f.tm, P.tn = 128, P.ksplit = f.ksplit, P.kt_per = f.kt_per;
  } else {
    P.wide = gemm_wide_plan(m, k, G, min_split, max_split);
    P.tm = P.wide.tm, P.tn = P.wide.tn, P.ksplit = P.wide.ksplit, P.kt_per = P.wide.kt_per;
  }
  return P;
}

}  // namespace

namespace tlg {

PromptPlan gemm_prompt_plan(int m, int k, const GemmGroups& G, int esize, bool in_place, bool workspace) {
  const int most = workspace ? max_split(m, k, esize) : 1;
  const PromptPlan P = prompt_plan(m, k, G, esize, 1, most);
  // exactly two: the workspace query's room where it counts on one
  return in_place && P.ksplit == 1 && most > 1 ? prompt_plan(m, k, G, esize, 2, 2) : P;
}

size_t gemm_split_bytes(int m, const GemmGroups& G, int ksplit) {
  size_t ncols = 0;
  for (int g = 0; g < G.count; ++g) ncols += (size_t)G.n[g];
  return ksplit > 1 ? (size_t)ksplit * m * ncols * sizeof(float) : 0;
}

}  // namespace tlg

namespace {

// Whether an output shares bytes with A or with a B.  Such a product comes out
// right where K is cut: every operand is read before the reduce pass writes the
// first output.  So it is cut where the workspace allows.
bool writes_inputs(const void* a, const GemmGroups& G, int m, int k, int64_t lda, int esize) {
  for (int g = 0; g < G.count; ++g) {
    const size_t nc = ((m - 1) * G.ldc[g] + G.n[g]) * esize;
    if (tl_overlap(G.c[g], nc, a, ((m - 1) * lda + k) * esize)) return true;
    for (int h = 0; h < G.count; ++h)
      if (tl_overlap(G.c[g], nc, G.b[h], ((k - 1) * G.ldb[h] + G.n[h]) * esize)) return true;
  }
  return false;
}

template <typename T>
int launch_gemm(const void* a, const GemmGroups& G, int m, int k, int64_t lda, void* workspace,
                size_t workspace_bytes, bool in_place, hipStream_t st) {
  GemmParams p{};
  p.a = a;
  p.m = m;
  p.k = k;
  p.lda = lda;
  p.G = G;
  const int64_t esize = T::size;
  const int64_t vec = 16 / esize;  // elements per 16-byte chunk
  // Every operand's rows must be 16-byte aligned for the loads, and all of A and
  // each B addressable with 32-bit offsets (counted up to a tile past A's last row
  // and two stages past B's).
  bool aligned = lda % vec == 0 && ((uintptr_t)a % 16) == 0 &&
                 ((int64_t)m + 257) * lda * esize < ((int64_t)1 << 32);
  int widest = 0;
  for (int g = 0; g < G.count; ++g) {
    aligned = aligned && G.ldb[g] % vec == 0 && G.n[g] % vec == 0 && ((uintptr_t)G.b[g] % 16) == 0 &&
              ((int64_t)k + 64 + 1) * G.ldb[g] * esize < ((int64_t)1 << 32);
    widest = G.n[g] > widest ? G.n[g] : widest;
  }
  if (aligned) {
    PromptPlan P = gemm_prompt_plan(m, k, G, (int)esize, in_place);
    if (P.ksplit > 1 &&
        (!workspace || workspace_bytes < gemm_split_bytes(m, G, P.ksplit) || ((uintptr_t)workspace % 16) != 0))
      P = gemm_prompt_plan(m, k, G, (int)esize, in_place, false);
    // columns of one store: 16 bytes from the kernels, 4 from the reduce
    const int run = P.ksplit > 1 || esize == 4 ? 4 : 8;
    p.tiles_m = (m + P.tm - 1) / P.tm;
    int64_t off = 0;
    for (int g = 0; g < G.count; ++g) {
      p.G.tile0[g + 1] = p.G.tile0[g] + p.tiles_m * ((G.n[g] + P.tn - 1) / P.tn);
      if (G.ldc[g] % run == 0 && ((uintptr_t)G.c[g] % (run * esize)) == 0) p.vec_store |= 1 << g;
      p.ws_off[g] = off;
      off += (int64_t)P.ksplit * m * G.n[g];
    }
    p.ksplit = P.ksplit;
    p.kt_per = P.kt_per;
    p.ws = (float*)workspace;
    p.per_xcd = (p.G.tile0[G.count] * P.ksplit + 7) / 8;
    const int e = T::size == 4 ? launch_gemm_f32(p, P.tm, st) : launch_gemm_wide(p, P.wide, (int)T::code, st);
    if (e || p.ksplit == 1) return e;
    int64_t runs = 0;
    for (int g = 0; g < G.count; ++g) runs = (int64_t)m * (G.n[g] / 4) > runs ? (int64_t)m * (G.n[g] / 4) : runs;
    const unsigned rb = (unsigned)((runs + 255) / 256 < 4096 ? (runs + 255) / 256 : 4096);
    hipLaunchKernelGGL((split_reduce_kernel<T>), dim3(rb, G.count), dim3(256), 0, st, p);
    return tl_launch_status();
  }
  dim3 grid((unsigned)((widest + 63) / 64), (unsigned)((m + 63) / 64), (unsigned)G.count);
  hipLaunchKernelGGL((gemm_simple_kernel<T>), grid, dim3(256), 0, st, p);
  return tl_launch_status();
}

// Checks shared by both entry points; fills the group table.
int make_groups(GemmGroups& G, int count, const void* const* b, void* const* c, const int* n, const int64_t* ldb,
                const int64_t* ldc) {
  if (count < 1 || count > kMaxGroups || !b || !c || !n || !ldb || !ldc) return TL_ERR_INVALID;
  G = GemmGroups{};
  G.count = count;
  for (int g = 0; g < count; ++g) {
    G.b[g] = b[g];
    G.c[g] = c[g];
    G.n[g] = n[g];
    G.ldb[g] = ldb[g];
    G.ldc[g] = ldc[g];
  }
  return 0;
}

int gemm_groups(const void* a, const GemmGroups& G, int m, int k, int64_t lda, void* workspace,
                size_t workspace_bytes, int dtype, void* stream) {
  if (m < 0 || k < 0) return TL_ERR_INVALID;
  if (dtype != TL_DTYPE_F32 && dtype != TL_DTYPE_F16 && dtype != TL_DTYPE_BF16) return TL_ERR_INVALID;
  if (m == 0) return 0;
  for (int g = 0; g < G.count; ++g) {
    if (G.n[g] < 0) return TL_ERR_INVALID;
    if (G.n[g] == 0) continue;
    if (!G.c[g] || G.ldc[g] < G.n[g] || (k > 0 && (!G.b[g] || G.ldb[g] < G.n[g]))) return TL_ERR_INVALID;
    if (!fits_int(G.ldb[g]) || !fits_int(G.ldc[g])) return TL_ERR_UNSUPPORTED;
  }
  if (k > 0 && (!a || lda < k)) return TL_ERR_INVALID;
  if (!fits_int(lda)) return TL_ERR_UNSUPPORTED;
  const size_t esize = dtype == TL_DTYPE_F32 ? 4 : 2;
  hipStream_t st = tl_resolve_stream(stream);
  // Groups with no columns take no part.
  GemmGroups live{};
  for (int g = 0; g < G.count; ++g) {
    if (G.n[g] == 0) continue;
    const int i = live.count++;
    live.b[i] = G.b[g];
    live.c[i] = G.c[g];
    live.n[i] = G.n[g];
    live.ldb[i] = G.ldb[g];
    live.ldc[i] = G.ldc[g];
  }
  if (live.count == 0) return 0;
  if (k == 0) {  // empty sum: zeros, row by row when C is a strided view
    for (int g = 0; g < live.count; ++g) {
      if (live.ldc[g] == live.n[g]) {
        const int e = tl_fill_bytes(live.c[g], 0, (size_t)m * live.n[g] * esize, st);
        if (e) return e;
        continue;
      }
      for (int r = 0; r < m; ++r) {
        const int e = tl_fill_bytes((char*)live.c[g] + (size_t)r * live.ldc[g] * esize, 0,
                                    (size_t)live.n[g] * esize, st);
        if (e) return e;
      }
    }
    return 0;
  }
  const bool in_place = writes_inputs(a, live, m, k, lda, (int)esize);
  if (m <= kSkinnyMaxM) {
    bool ok = true;
    const int cpc = 16 / (int)esize;
    for (int g = 0; g < live.count; ++g)
      ok = ok && live.n[g] % cpc == 0 && live.ldb[g] % cpc == 0 && ((uintptr_t)live.b[g] % 16) == 0 &&
           (int64_t)(k - 1) * live.ldb[g] * (int64_t)esize < INT32_MAX;
    if (ok) {
      const size_t need = skinny_workspace_bytes(m, live, k, (int)esize);
      if (need && (!workspace || workspace_bytes < need)) return TL_ERR_INVALID;
      switch (dtype) {
        case TL_DTYPE_F32: return launch_skinny<F32>(a, live, m, k, lda, workspace, in_place, st);
        case TL_DTYPE_F16: return launch_skinny<F16>(a, live, m, k, lda, workspace, in_place, st);
        default: return launch_skinny<BF16>(a, live, m, k, lda, workspace, in_place, st);
      }
    }
  }
  switch (dtype) {
    case TL_DTYPE_F32: return launch_gemm<F32>(a, live, m, k, lda, workspace, workspace_bytes, in_place, st);
    case TL_DTYPE_F16: return launch_gemm<F16>(a, live, m, k, lda, workspace, workspace_bytes, in_place, st);
    default: return launch_gemm<BF16>(a, live, m, k, lda, workspace, workspace_bytes, in_place, st);
  }
}

size_t groups_workspace_bytes(int m, int k, const GemmGroups& G, int dtype) {
  if (m <= 0 || k <= 0) return 0;
  GemmGroups live{};
  for (int g = 0; g < G.count; ++g)
    if (G.n[g] > 0) live.n[live.count++] = G.n[g];
  if (live.count == 0) return 0;
  const int esize = dtype == TL_DTYPE_F32 ? 4 : 2;
  // few rows: the K-slice partials; more: those of the plan's slices, and of two
  // where they are cheap, for a C that overlaps A or B (a product that falls back to
  // the simple kernel uses none of it)
  if (m <= kSkinnyMaxM) return skinny_workspace_bytes(m, live, k, esize);
  const int chosen = gemm_prompt_plan(m, k, live, esize, false).ksplit;
  return gemm_split_bytes(m, live, chosen > 1 ? chosen : few_rows_split(m, k, esize) > 1 ? 2 : 1);
}

}  // namespace

extern "C" {

size_t tl_gemm_workspace_bytes(int m, int n, int k, int dtype) {
  GemmGroups G{};
  G.count = 1;
  G.n[0] = n;
  return groups_workspace_bytes(m, k, G, dtype);
}

int tl_gemm(const void* a, const void* b, void* c, int m, int n, int k, int64_t lda, int64_t ldb, int64_t ldc,
            void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  if (n < 0) return TL_ERR_INVALID;
  GemmGroups G{};
  const int st = make_groups(G, 1, &b, &c, &n, &ldb, &ldc);
  if (st) return st;
  return gemm_groups(a, G, m, k, lda, workspace, workspace_bytes, dtype, stream);
}

size_t tl_gemm_grouped_workspace_bytes(int m, int k, int count, const int* n, int dtype) {
  if (count < 1 || count > kMaxGroups || !n) return 0;
  GemmGroups G{};
  G.count = count;
  for (int g = 0; g < count; ++g) G.n[g] = n[g];
  return groups_workspace_bytes(m, k, G, dtype);
}

int tl_gemm_grouped(const void* a, int m, int k, int64_t lda, int count, const void* const* b, void* const* c,
                    const int* n, const int64_t* ldb, const int64_t* ldc, void* workspace, size_t workspace_bytes,
                    int dtype, void* stream) {
  GemmGroups G{};
  const int st = make_groups(G, count, b, c, n, ldb, ldc);
  if (st) return st;
  return gemm_groups(a, G, m, k, lda, workspace, workspace_bytes, dtype, stream);
}

}  // extern "C"
