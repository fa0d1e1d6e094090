// fp32 prompt products on the 16-bit matrix cores: gemm_f32_kernel and the
// choice of its tile.  tl_gemm.hip launches it.
#include "tl_gemm_f32.h"

namespace tlg {
namespace {

typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) float lds_f32;

constexpr int kBk = 32;  // k per LDS stage

struct F32Tile {
  int tm, at_once;     // rows; workgroups a CU holds
  double tile_us;      // launch, first loads, stores
  double stage_us[3];  // a 32-k stage of one, two, three of them on a CU
};
// Both heights; a split's partials are written, read and summed at about 6.7 TB/s, with
// one more launch and a part per slice.  Fitted to 139 products of 9 to 2048 rows
// (SmolLM2 and Llama-3.2-3B widths, weights rotated through 0.8 GB) run on both heights
// and every split: the choice is the fastest, or within 2% of it, but for three, within 4%.
// Of 104 such products 78 run at 0.98 to 2.9 times the speed of the best fp32 MFMA plan;
// 26, of 9 to 1000 rows at K 576 to 2560, at 0.89 to 0.98 (32 x 576 x 576 10.8 -> 12.1
// us, the widest): a few stages a slice, whose loads, splits and range check follow one
// another.
const F32Tile kF32Tiles[] = {{128, 2, 5.7, {1.65, 2.75, 0}}, {64, 3, 5.1, {1.3, 1.8, 2.47}}};

// x0, x1 as three pairs of bf16 whose sums are x0 and x1 exactly (8 significant
// bits each, rounded to nearest, so every remainder is exact).
__device__ __forceinline__ void split3(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
  const float a[2] = {x0, x1};
  h = pack2<BF16>(a);
  const float r[2] = {x0 - __uint_as_float(h << 16), x1 - __uint_as_float(h & 0xFFFF0000u)};
  m = pack2<BF16>(r);
  const float s[2] = {r[0] - __uint_as_float(m << 16), r[1] - __uint_as_float(m & 0xFFFF0000u)};
  l = pack2<BF16>(s);
}

// The wave's largest value, with no LDS: by rows of 16 lanes, then the four rows'.
__device__ __forceinline__ float wave_max(float x) {
  x = fmaxf(x, dpp_mov<0xB1>(x));   // quad_perm [1,0,3,2]
  x = fmaxf(x, dpp_mov<0x4E>(x));   // quad_perm [2,3,0,1]
  x = fmaxf(x, dpp_mov<0x141>(x));  // row_half_mirror
  x = fmaxf(x, dpp_mov<0x140>(x));  // row_mirror
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __uint_as_float(__builtin_amdgcn_readlane((int)__float_as_uint(x), 16 * i));
  return fmaxf(fmaxf(r[0], r[1]), fmaxf(r[2], r[3]));
}

// Workgroup tile 32 MB x 128 of C, four waves of 16 MB x 64.  Each fp32 operand is
// the exact sum of three bf16 parts (Henry, Tang, Heinecke: Leveraging the bfloat16
// Artificial Intelligence Datatype For Higher-Precision Computations, ARITH 2019),
// and a product is six 16x16x32 bf16 MFMAs (2.5 PFLOP/s / 6) where the fp32 MFMA's
// peak is 157 TFLOP/s.  A stage's fp32 values are loaded to registers two stages ahead, split there once per workgroup
// while the current stage's MFMAs run, and stored as three bf16 planes in one LDS
// buffer (48 or 36 KiB: two or three workgroups a CU cover each other's
// barriers); the next stage's splits start when every wave holds its operands.
//
// Error against 64 bits, 2048 x 3072 x 16384 (relative 2-norm): 3.8e-7, with the
// fp32 MFMA 9.9e-7; 1023 x 960 x 5120: 2.0e-7, 3.2e-7.  The products are exact in
// fp32 accumulators; the five small ones of a stage are summed apart, so a sum
// takes two roundings per 32 k where the fp32 MFMA's chain took sixteen (one
// accumulator for all six: 8.6e-7).
//
// Measured against the fp32 MFMA tiles it replaced, Llama-3.2-3B at 2048 rows:
// gate/up 1555 -> 1071 us (193 TFLOP/s), q/k/v 522 -> 367, o 318 -> 223, down 809
// -> 565; SmolLM2-360M at 1023 rows gate/up 108 -> 77, q/k/v 44 -> 39, o 31 -> 28,
// down 53 -> 45.  What bounds it with two
// workgroups a CU is the issue port (about 240 VALU instructions, 96 MFMAs and 49
// LDS ones per wave and stage); a lone one waits on its own LDS reads.
template <int MB>
__global__ __launch_bounds__(256, MB == 2 ? 3 : 2) void gemm_f32_kernel(GemmParams p) {
  constexpr int TM = 32 * MB, TN = 128, NB = 4;
  constexpr int SA = TM * 64, SB = kBk * 256;  // bytes of one plane of a stage
  __shared__ __attribute__((aligned(1024))) char smem[3 * (SA + SB)];
  __shared__ float s_row[TM], s_col[8][TN], s_max[4], s_amax[4], s_bmax[4], s_least[4];

  int grp, tm, tn, ks;
  if (!gemm_tile(p, grp, tm, tn, ks)) return;
  const int pn = p.G.n[grp];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int wm = wave & 1, wn = wave >> 1;
  const int m_tile = tm * TM, n_tile = tn * TN;
  __attribute__((address_space(3))) char* const lds = (__attribute__((address_space(3))) char*)smem;

  const int km = p.k & ~3;  // whole 16-byte chunks; the last k % 4 are added at the end
  const int n_kt = (km + kBk - 1) / kBk;
  const int kt_lo = ks * p.kt_per;
  const int kt_hi = min(n_kt, kt_lo + p.kt_per);
  const int k_hi = min(km, kt_hi * kBk);
  const float* const a = (const float*)p.a;
  const float* const b = (const float*)p.G.b[grp];
  const int64_t lda = p.lda, ldb = p.G.ldb[grp];

  // Loads of a stage.  A: thread -> rows tid / 8 + 32 i, k 4 (tid % 8) .. + 3.
  // B: thread -> rows (tid / 32) + 8 i, columns 4 (tid % 32) .. + 3.  Buffer
  // resources end at the tile's last row's and the slice's last k and n: zeros past them.
  constexpr int AI = TM / 32, BI = 4;
  const int rows = min(TM, p.m - m_tile);
  const uint32_t lda4 = (uint32_t)lda * 4, ldb4 = (uint32_t)ldb * 4;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a + (int64_t)m_tile * lda), (short)0, (int)view_bytes(rows, lda, k_hi, 4), kBufRsrcWord3);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void*)b, (short)0, (int)view_bytes(k_hi, ldb, pn, 4), kBufRsrcWord3);
  const int a_row = tid >> 3, a_k = 4 * (tid & 7);
  const int b_row = tid >> 5, b_n = 4 * (tid & 31);
  u32x4 av[AI], bv[BI];  // the next stage's
  auto load = [&](int kt, u32x4 (&av)[AI], u32x4 (&bv)[BI]) __attribute__((always_inline)) {
    const int k0 = min(kt, kt_hi) * kBk;  // past the slice: zeros, and no offset that wraps
    const bool a_in = k0 + a_k < k_hi;
#pragma unroll
    for (int i = 0; i < AI; ++i)
      av[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
          ra, a_in ? (uint32_t)(a_row + 32 * i) * lda4 + (uint32_t)(k0 + a_k) * 4 : 0xFFFFFFF0u, 0, 0));
#pragma unroll
    for (int i = 0; i < BI; ++i)
      bv[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
          rb, (uint32_t)(b_row + 8 * i) * ldb4 + (uint32_t)(n_tile + b_n) * 4, (uint32_t)k0 * ldb4, 0));
  };
  // Largest magnitude each thread saw of its rows of A and its columns of B.
  float a_max[AI], b_max[4];
#pragma unroll
  for (int i = 0; i < AI; ++i) a_max[i] = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) b_max[i] = 0.f;
  auto store = [&](const u32x4 (&av)[AI], const u32x4 (&bv)[BI]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      const int row = a_row + 32 * i;
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[e] = __uint_as_float(av[i][e]);
        a_max[i] = __builtin_elementwise_maximum(a_max[i], fabsf(f[e]));
      }
      uint32_t w[3][2];
      split3(f[0], f[1], w[0][0], w[1][0], w[2][0]);
      split3(f[2], f[3], w[0][1], w[1][1], w[2][1]);
      const int at = row * 64 + (((a_k >> 3) ^ ((row >> 2) & 3)) << 4) + 8 * ((a_k >> 2) & 1);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(lds_u32x2*)(lds + q * SA + at) = u32x2{w[q][0], w[q][1]};
    }
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      const int row = b_row + 8 * i;
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[e] = __uint_as_float(bv[i][e]);
        b_max[e] = __builtin_elementwise_maximum(b_max[e], fabsf(f[e]));
      }
      uint32_t w[3][2];
      split3(f[0], f[1], w[0][0], w[1][0], w[2][0]);
      split3(f[2], f[3], w[0][1], w[1][1], w[2][1]);
      const int swz = (4 * (row & 3)) ^ (2 * ((row >> 3) & 1));
      const int at = 3 * SA + row * 256 + (((b_n >> 3) ^ swz) << 4) + 8 * ((b_n >> 2) & 1);
#pragma unroll
      for (int q = 0; q < 3; ++q) *(lds_u32x2*)(lds + q * SB + at) = u32x2{w[q][0], w[q][1]};
    }
  };

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int lc = lane & 15, g = lane >> 4;
  const int ar = 16 * MB * wm + lc;
  const int a_rd = ar * 64 + ((g ^ ((ar >> 2) & 3)) << 4);
  int b_rd[NB];
  {
    const int e = lc >> 2, pp = lc & 3, row = 8 * g + e;
    const int swz = (4 * (row & 3)) ^ (2 * ((row >> 3) & 1));
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      b_rd[nb] = 3 * SA + row * 256 + (((8 * wn + 2 * nb + (pp >> 1)) ^ swz) << 4) + 8 * (pp & 1);
  }

  {  // both stages on their way at once: a slice of a few stages is a chain of latencies
    u32x4 a0[AI], b0[BI];
    load(kt_lo, a0, b0);
    load(kt_lo + 1, av, bv);
    store(a0, b0);
  }
  for (int kt = kt_lo; kt < kt_hi; ++kt) {
    lds_barrier();
    bf16x8 af[3][MB], bf[3][NB];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(lds + (q * SB + b_rd[nb])));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(lds + (q * SB + b_rd[nb] + 4 * 256)));
        const u32x2 x = __builtin_bit_cast(u32x2, lo), y = __builtin_bit_cast(u32x2, hi);
        bf[q][nb] = __builtin_bit_cast(bf16x8, u32x4{x.x, x.y, y.x, y.y});
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        af[q][mb] = __builtin_bit_cast(bf16x8, *(lds_u32x4*)(lds + (q * SA + a_rd + 16 * 64 * mb)));
    }
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    // The small products first, into sums of their own; the middle part times the
    // smallest, either way, and the smallest times itself are left out: up to 2^-24.2
    // of the product, 2^-27 in the root mean square.
    constexpr int PA[5] = {0, 2, 1, 0, 1}, PB[5] = {2, 0, 1, 1, 0};
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x4 lo[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) lo[mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 5; ++q)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          lo[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[PB[q]][nb], af[PA[q]][mb], lo[mb], 0, 0, 0);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[0][nb], af[0][mb], acc[mb][nb], 0, 0, 0);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb][nb] += lo[mb];
    }
    store(av, bv);         // the next stage's parts, beside the MFMAs
    load(kt + 2, av, bv);  // past the slice: zeros, with no memory access
    // one MFMA, then up to three of the splits' VALU instructions, and so on
#pragma unroll
    for (int i = 0; i < 24 * MB; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      if (i % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
    }
  }

  // From here on lane values are made again: none of them is kept through the loop.
  int tid_e = (int)threadIdx.x;
  asm volatile("" : "+v"(tid_e));
  const int wave_e = __builtin_amdgcn_readfirstlane(tid_e >> 6);
  const int lc_e = tid_e & 15, g_e = (tid_e >> 4) & 3;
  const int m_e = 16 * MB * (wave_e & 1), n_e = 64 * (wave_e >> 1);  // the wave's corner in the tile
  const int a_row_e = tid_e >> 3, b_row_e = tid_e >> 5, b_n_e = 4 * (tid_e & 31);

  // The parts stand for every fp32 value between 2^-102 and 2^127.  Two things send
  // the tile through the fp32 MFMA: a row of A or a column of B whose largest
  // magnitude is not between 2^-40 and 2^60 (NaN and infinity included; all zeros are
  // fine), and a sum below 2^-44 of its row's largest times its column's, which may
  // be made of entries below 2^-102 alone (above it they weigh k 2^-42 at most).
  // First by what needs no exchange but the tile's largest magnitudes: every
  // thread's own largest in range, the tile's smallest sum against them.  The rows and
  // columns one by one only where that falls short, which took 0.5 us a product.
  float a_most = 0.f, b_most = 0.f, least = INFINITY;
  bool fine = true;
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    a_most = fmaxf(a_most, a_max[i]);
    fine &= a_max[i] == 0.f || (a_max[i] >= 0x1p-40f && a_max[i] <= 0x1p60f);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    b_most = fmaxf(b_most, b_max[e]);
    fine &= b_max[e] == 0.f || (b_max[e] >= 0x1p-40f && b_max[e] <= 0x1p60f);
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const f32x4 c = acc[mb][nb];
      const bool inside = m_tile + m_e + 16 * mb + lc_e < p.m && n_tile + n_e + 16 * nb + 4 * g_e < pn;
      least = fminf(least, inside ? fminf(fminf(fabsf(c[0]), fabsf(c[1])), fminf(fabsf(c[2]), fabsf(c[3]))) : INFINITY);
    }
  fine = __all(fine);
  a_most = wave_max(a_most);
  b_most = wave_max(b_most);
  least = -wave_max(-least);
  if ((tid_e & 63) == 0) {
    s_amax[wave_e] = fine ? a_most : INFINITY;
    s_bmax[wave_e] = b_most;
    s_least[wave_e] = least;
  }
  __syncthreads();
  const float a_all = fmaxf(fmaxf(s_amax[0], s_amax[1]), fmaxf(s_amax[2], s_amax[3]));
  const float b_all = fmaxf(fmaxf(s_bmax[0], s_bmax[1]), fmaxf(s_bmax[2], s_bmax[3]));
  const float least_all = fminf(fminf(s_least[0], s_least[1]), fminf(s_least[2], s_least[3]));
  bool plain = a_all == INFINITY || least_all < a_all * 0x1p-44f * b_all;
  if (plain) {
#pragma unroll
    for (int i = 0; i < AI; ++i) {
      float v = a_max[i];
#pragma unroll
      for (int o = 4; o >= 1; o >>= 1) v = __builtin_elementwise_maximum(v, __shfl_xor(v, o));
      if ((tid_e & 7) == 0) s_row[a_row_e + 32 * i] = v;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s_col[b_row_e][b_n_e + e] = b_max[e];
    __syncthreads();
    float v = 0.f;  // waves 0 and 1: a row's largest magnitude, 2 and 3: a column's
    if (tid_e < TM) {
      v = s_row[tid_e];
    } else if (tid_e >= 128) {
      v = s_col[0][tid_e - 128];
#pragma unroll
      for (int i = 1; i < 8; ++i) v = __builtin_elementwise_maximum(v, s_col[i][tid_e - 128]);
      if (n_tile + tid_e - 128 >= pn) v = 0.f;  // columns past n hold the next row's values
      s_col[0][tid_e - 128] = v;
    }
    const bool in_range = __all(v == 0.f || (v >= 0x1p-40f && v <= 0x1p60f));
    v = wave_max(v);
    if ((tid_e & 63) == 0) s_max[wave_e] = in_range ? v : INFINITY;
    __syncthreads();
    const float most = fmaxf(s_max[0], s_max[1]) * 0x1p-44f * fmaxf(s_max[2], s_max[3]);
    plain = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3])) == INFINITY;
    if (!plain && least_all < most) {
      float short_of = 0.f;  // by how much a sum falls short of its bound, at most
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const float row = s_row[m_e + 16 * mb + lc_e] * 0x1p-44f;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int e = 0; e < 4; ++e)  // 0 past n, and past m
            short_of = fmaxf(short_of, fmaf(row, s_col[0][n_e + 16 * nb + 4 * g_e + e], -fabsf(acc[mb][nb][e])));
      }
      plain = __syncthreads_or(short_of > 0.f);
    }
  }

  const int mw = m_tile + m_e, nw = n_tile + n_e;
  if (plain) {
    // Once more, on 16x16x4 fp32 MFMAs: rows of A of 128 bytes, chunk c of row r at
    // slot c ^ ((r >> 1) & 7); rows of B of 512 bytes, chunk c of row r at slot c ^
    // 4 ((r >> 2) & 3).  Step t of a 16-k half takes k = 4 g + t, so that one 16-byte
    // read of A serves four steps.  2048 x 3072 x 3072, with one NaN, a row times
    // 1e-30, all of A times 1e-30: 222 us, 450, 454, 503 (an fp32 MFMA kernel alone: 318).
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int B0 = TM * 128;
    static_assert(B0 + kBk * 512 <= 3 * (SA + SB), "a stage of fp32 operands fits the planes' room");
    load(kt_lo, av, bv);
    for (int kt = kt_lo; kt < kt_hi; ++kt) {
      lds_barrier();
#pragma unroll
      for (int i = 0; i < AI; ++i) {
        const int row = a_row_e + 32 * i;
        *(lds_u32x4*)(lds + row * 128 + (((tid_e & 7) ^ ((row >> 1) & 7)) << 4)) = av[i];
      }
#pragma unroll
      for (int i = 0; i < BI; ++i) {
        const int row = b_row_e + 8 * i;
        *(lds_u32x4*)(lds + B0 + row * 512 + (((b_n_e >> 2) ^ (4 * ((row >> 2) & 3))) << 4)) = bv[i];
      }
      load(kt + 1, av, bv);
      lds_barrier();
#pragma unroll 1
      for (int half = 0; half < 2; ++half) {
        u32x4 x[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const int row = m_e + 16 * mb + lc_e;
          x[mb] = *(lds_u32x4*)(lds + row * 128 + (((4 * half + g_e) ^ ((row >> 1) & 7)) << 4));
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            const int col = n_e + 16 * nb + lc_e;
            const float y = *(lds_f32*)(lds + B0 + (16 * half + 4 * g_e + t) * 512 + (((col >> 2) ^ (4 * g_e)) << 4) + 4 * (col & 3));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
              acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, __uint_as_float(x[mb][t]), acc[mb][nb], 0, 0, 0);
          }
      }
    }
  }

  if (ks == 0)
    for (int k = km; k < p.k; ++k)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const f32x4 y = *(const f32x4*)(b + (int64_t)k * ldb + min(nw + 16 * nb + 4 * g_e, pn - 4));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          const float x = a[(int64_t)min(mw + 16 * mb + lc_e, p.m - 1) * lda + k];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[mb][nb][e] = fmaf(x, y[e], acc[mb][nb][e]);
        }
      }

  // Lane (lc, g) holds row 16 mb + lc of the wave's block, columns 16 nb + 4 g + 0..3.
  float* out = (float*)p.G.c[grp];
  int64_t ldo = p.G.ldc[grp];
  bool vec = (p.vec_store >> grp) & 1;
  if (p.ksplit > 1) {
    out = p.ws + p.ws_off[grp] + (int64_t)ks * p.m * pn;
    ldo = pn;
    vec = true;  // n_g is a multiple of 4 here
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = mw + 16 * mb + lc_e;
    if (m >= p.m) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int n = nw + 16 * nb + 4 * g_e;
      if (n >= pn) continue;
      if (vec) {
        *(f32x4*)(out + (int64_t)m * ldo + n) = acc[mb][nb];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) out[(int64_t)m * ldo + n + e] = acc[mb][nb][e];
      }
    }
  }
}

}  // namespace

F32Plan gemm_f32_plan(int m, int k, const GemmGroups& G, int min_split, int max_split) {
  F32Plan best{};
  const int cus = tl_device_cus();
  const int stages = (k / 4 * 4 + kBk - 1) / kBk;
  int64_t ncols = 0;
  for (int g = 0; g < G.count; ++g) ncols += G.n[g];
  for (const F32Tile& c : kF32Tiles) {
    int64_t tiles = 0;
    for (int g = 0; g < G.count; ++g) tiles += (int64_t)((m + c.tm - 1) / c.tm) * ((G.n[g] + 127) / 128);
    for (int S = min_split; S <= max_split && (S == min_split || stages >= S); ++S) {
      const int64_t per_cu = (tiles * S + cus - 1) / cus;
      const int rest = (int)(per_cu % c.at_once);
      const double stage = (double)(per_cu / c.at_once) * c.stage_us[c.at_once - 1] + (rest ? c.stage_us[rest - 1] : 0.0);
      const double reduce = S > 1 ? (8.0 * S + 4) * m * (double)ncols / 6.7e6 + 3.7 + 0.26 * S : 0.0;
      const double t = stage * ((stages + S - 1) / S) + c.tile_us + reduce;
      if (best.tm == 0 || t < best.us) best = F32Plan{c.tm, S, (stages + S - 1) / S, t};
    }
  }
  return best;
}

int launch_gemm_f32(const GemmParams& p, int tm, hipStream_t st) {
  const dim3 grid((unsigned)(8 * p.per_xcd)), block(256);
  if (tm == 128)
    hipLaunchKernelGGL((gemm_f32_kernel<4>), grid, block, 0, st, p);
  else
    hipLaunchKernelGGL((gemm_f32_kernel<2>), grid, block, 0, st, p);
  return tl_launch_status();
}

}  // namespace tlg
