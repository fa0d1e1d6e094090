// 16-bit prompt products (and batches of decoded tokens) on the matrix cores:
// gemm_wide_kernel and the choice of its tile.  tl_gemm.hip launches it.
#include "tl_gemm_wide.h"

namespace tlg {
namespace {

// Every tile built, with what one costs (measured, every CU busy, bf16: whole
// products of 1 to 8 rounds at k 960 to 8192): a larger one does more per byte
// moved, a smaller one leaves fewer CUs idle in the last round.  A split costs its
// reduce's launch, a part per slice and the partials' traffic.  Of 180 products of 9 to
// 2048 rows run on every tile and split (SmolLM2 and Llama-3.2-3B widths, weights
// rotated through 0.8 GB) the choice is the fastest, or within 4% of it, but for nine,
// within 13% (320 rows of q/k/v 30.4 against 27.0 us, the widest); the mean is 0.6%, and
// constants fitted to these very products leave 0.4%.
const WidePlan kWidePlans[] = {{256, 256, 9.0, 0.755}, {192, 256, 8.0, 0.53}, {128, 256, 7.0, 0.42},
                               {128, 192, 6.0, 0.365}, {128, 128, 5.0, 0.27}, {64, 128, 4.0, 0.21}};

typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;

// acc += a . b with the accumulator held in AGPRs.  Inline assembly: every
// definition of an accumulator is then an AGPR output, and the register
// allocator has no copy to make; with the builtin it moved most of the 256
// accumulators between VGPRs and AGPRs, and to scratch, in every pass of the loop.
// The compiler does not see these as MFMAs: whoever reads an accumulator waits
// first (mma_drain), and operands come from LDS reads, never from a VALU
// instruction just before.  The build checks the assembly for both
// (triton_llm/_build.py check_mfma_asm).
template <typename T>
__device__ __forceinline__ void mma16(f32x4& acc, const u32x4& a, const u32x4& b) {
  if constexpr (T::code == TL_DTYPE_BF16)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mma_zero(f32x4& acc) {
  acc = f32x4{0.f, 0.f, 0.f, 0.f};
  asm volatile("" : "+a"(acc));
}
// The accumulator's value from here on: keeps its copy to VGPRs next to its use.
__device__ __forceinline__ const f32x4& mma_take(f32x4& acc) {
  asm volatile("" : "+a"(acc));
  return acc;
}
__device__ __forceinline__ void mma_drain() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// Workgroup tile 32 MB x 32 NB of C, four waves in 2 x 2, each 16 MB x 16 NB in
// 16 x 16 blocks, one wave per SIMD.  K is walked in 32-k stages held in a ring
// of NST LDS buffers (up to the whole 160 KiB), every tile moved global -> LDS by
// LDS-DMA NST - 1 stages ahead.  While a wave issues stage kt's MFMAs it reads
// stage kt + 1's operands into its other register set and loads stage kt + NST -
// 1, one such job between MFMAs; one barrier a stage.
//
// Why this shape (2048-row Llama-3.2-3B prompt, bf16, measured):
//   * 16x16x32 MFMAs: with random operands the chip's power limit holds a stream
//     of them at 2.1 PFLOP/s (2.09 GHz) and one of 32x32x16 at 1.8 (1.78 GHz).
//   * 128 x 128 a wave: an LDS byte read feeds twice the MFMAs of 64 x 64 waves, and
//     one wave per SIMD has the registers for it (256 accumulators in AGPRs, two
//     operand sets in VGPRs).
//   * Operands a stage ahead: nothing waits on an LDS read, and the stage's
//     1024 MFMA cycles take 1050-1250 with operands from L2, 1500 where weights
//     come from HBM (their latency; deeper rings than LDS has would help).
//   * Five ring stages against four: 8192^3 912 -> 1447 TFLOP/s together with the
//     panel order of gemm_tile (hipBLASLt: 1290).
//   * C through LDS, whole row pieces: epilogue 16600 -> 9000 cycles of a tile's
//     150000, against 8-byte stores from the accumulators.
// Against 64- to 256-row tiles of 32x32x16 MFMAs, weights rotated through 1 GB:
// gate/up 205 -> 162 us (1270 TFLOP/s), down 141 -> 118, q/k/v 102 -> 65; 64 rows
// gate/up 28.2 -> 26.5, down 24.2 -> 20.3; of 74 products of 9 to 4096 rows at these
// models' widths 66 ran at 0.98 to 1.76 times their speed.  The others: gate/up at 384
// rows 51.9 -> 56.2 us, 55.7 -> 56.3 when repeated (448 rows 60.0 -> 49.4: 192 tiles of
// 128 x 256 take longer than 256 do), q/k/v at 256 24.5 -> 26.3, and six of 9 to 64 rows
// of K 960 and 1536, up to 1 us each (64 x 960 x (2560, 2560) 12.1 -> 13.1).  What
// bounds it now: at 4 and more rounds the power limit (1.67 GHz), at one or two
// the HBM latency of the weights and each tile's first loads and stores.
//
// LDS layouts (16-byte chunks, XOR-swizzled; the counters show conflicts in 25% to 35% of
// the LDS cycles, behind reads made a stage ahead):
//   A: rows (m) of 64 bytes (k), chunk c of row r at slot c ^ ((r >> 2) & 3); lane
//      (l % 16, g = l / 16) reads 8 consecutive k of row l % 16: chunk g.
//   B: rows (k) of 64 NB bytes (n), chunk c of row r at slot c ^ b_swz(r): the
//      four rows of a transposing read fall in distinct 64-byte banks groups, its
//      two 16-lane groups in distinct halves of them.  ds_read_b64_tr_b16: lane
//      4 e + p of group g reads row 8 g + 4 t + e, columns 4 p .. 4 p + 3, and lane
//      16 g + j receives column j, rows 8 g + 4 t + 0..3 (t = 0, 1: two reads).
template <typename T, int MB, int NB, int NST>
__global__ __launch_bounds__(256, 1) void gemm_wide_kernel(GemmParams p) {
  using Bits = typename T::bits;
  constexpr int TM = 32 * MB, TN = 32 * NB;
  constexpr int BK = 32;
  constexpr int AROW = BK * 2;       // bytes of an A row in LDS
  constexpr int BROW = TN * 2;       // bytes of a B row in LDS
  constexpr int SA = TM * AROW, SB = BK * BROW, STAGE = SA + SB;
  constexpr int A_REG = SA / 4096, B_REG = SB / 4096, PER = A_REG + B_REG;  // 1 KiB regions per wave
  constexpr int BCH = BROW / 16;
  static_assert(SA % 4096 == 0 && SB % 4096 == 0, "every wave fills whole 1 KiB regions");
  static_assert((NST - 2) * PER < 64, "vmcnt is 6 bits");
  __shared__ __attribute__((aligned(1024))) char smem[NST * STAGE];

  int grp, tm, tn, ks;
  if (!gemm_tile(p, grp, tm, tn, ks)) return;
  const int pn = p.G.n[grp];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int wm = wave & 1, wn = wave >> 1;
  const int m_tile = tm * TM, n_tile = tn * TN;
  __attribute__((address_space(3))) char* const lds = (__attribute__((address_space(3))) char*)smem;
  const uint32_t lds0 = (uint32_t)(size_t)lds;

  const int n_kt = (p.k + BK - 1) / BK;
  const int kt_lo = ks * p.kt_per;
  const int kt_hi = min(n_kt, kt_lo + p.kt_per);
  // Where k ends inside a 16-byte chunk the last 32-k block comes first, as stage 0:
  // what its chunk holds past k is then cleared in LDS once (below), before the ring
  // turns.  The blocks of the other stages are whole.
  const bool ragged = (p.k & 7) != 0, ends_first = ragged && ks == 0;
  const int block = ragged ? (ends_first ? n_kt - 1 : kt_lo - 1) : kt_lo;  // of the first stage
  const uint32_t lda2 = (uint32_t)(p.lda * 2), ldb2 = (uint32_t)(p.G.ldb[grp] * 2);
  const int rows = min(TM, p.m - m_tile);
  // A from this tile's first row, to the end of its last row's last chunk; B to its
  // last row's n.  The range check covers voff + soff, and what is past it reads as
  // zeros: rows past m, k rows past the last.  A's chunks past the slice are sent to
  // the resource's end (a_cur below), B's stages past it too (b_soff): no sum of
  // offsets passes 32 bits that an address of the operands does not.  A stage of zeros
  // adds nothing, so the ring needs no tail.
  const uint32_t a_end = view_bytes(rows, p.lda, (p.k + 7) & ~7, 2), b_end = (uint32_t)p.k * ldb2;
  const i32x4 ra = uniform_rsrc((const char*)p.a + (int64_t)m_tile * lda2, a_end);
  const i32x4 rb = uniform_rsrc(p.G.b[grp], view_bytes(p.k, p.G.ldb[grp], pn, 2));

  auto b_swz = [](int row) __attribute__((always_inline)) {
    return (BCH % 16 == 0 ? 4 * (row & 3) : 4 * ((row >> 1) & 1)) ^ (2 * ((row >> 3) & 1));
  };
  uint32_t a_voff, b_off[B_REG], a_soff[A_REG];
  int a_left;                   // k left of this lane's chunk in the next stage to load
  int b_left = kt_hi - kt_lo;   // stages left
  {
    const int row = 16 * wave + lane / 4;
    const int ch = (lane & 3) ^ ((row >> 2) & 3);
    a_voff = (uint32_t)row * lda2 + (uint32_t)(ch * 16) + (uint32_t)(block * AROW);
    a_left = (ragged && !ends_first ? (kt_hi - kt_lo) * BK : min(p.k, (ends_first ? n_kt : kt_hi) * BK) - block * BK) - 8 * ch;
#pragma unroll
    for (int j = 0; j < A_REG; ++j) a_soff[j] = (uint32_t)(64 * j) * lda2;
#pragma unroll
    for (int j = 0; j < B_REG; ++j) {
      const int pos = (wave + 4 * j) * 1024 + lane * 16;
      const int r = pos / BROW, slot = (pos % BROW) / 16;
      b_off[j] = (uint32_t)r * ldb2 + (uint32_t)(n_tile * 2) + (uint32_t)((slot ^ b_swz(r)) * 16);
    }
  }
  uint32_t b_soff = (uint32_t)min(block * BK, p.k) * ldb2;
  uint32_t a_cur = 0;
  // load j of the next stage in turn; j = 0 fixes the stage's A offset, the last moves on
  auto load_one = [&](uint32_t buf_base, int j) __attribute__((always_inline)) {
    if (j == 0) a_cur = a_left > 0 ? a_voff : a_end;
    if (j < A_REG)
      lds_dma16(ra, a_cur, buf_base + (wave + 4 * j) * 1024, a_soff[j]);
    else
      lds_dma16(rb, b_off[j - A_REG], buf_base + SA + (wave + 4 * (j - A_REG)) * 1024, b_soff);
    if (j == PER - 1) {
      a_voff += AROW;
      a_left -= BK;
      b_soff = --b_left > 0 ? b_soff + (uint32_t)BK * ldb2 : b_end;
    }
  };

  f32x4 acc[MB][NB];
  const int lc = lane & 15, g = lane >> 4;
  uint32_t a_rd, b_rd[NB];
  {
    const int row = 16 * MB * wm + lc;
    a_rd = (uint32_t)(row * AROW + ((g ^ ((row >> 2) & 3)) << 4));
    const int e = lc >> 2, pp = lc & 3;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int c = 2 * NB * wn + 2 * nb + (pp >> 1);
      b_rd[nb] = (uint32_t)(SA + (8 * g + e) * BROW + ((c ^ b_swz(8 * g + e)) << 4) + 8 * (pp & 1));
    }
  }
  u32x4 af[2][MB];
  u32x2 bf[2][NB][2];
  constexpr int NRD = MB + 2 * NB;
  // read i of a stage into set s: B 0, the A blocks, the other B blocks
  auto read_one = [&](uint32_t base, int s, int i) __attribute__((always_inline)) {
    if (i >= 2 && i < 2 + MB) {
      af[s][i - 2] = *(lds_u32x4*)(lds + (base + a_rd + (uint32_t)(16 * (i - 2) * AROW)));
    } else {
      const int k = i < 2 ? i : i - MB;
      const int nb = k >> 1, t = k & 1;
      bf[s][nb][t] = __builtin_bit_cast(
          u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(lds + (base + b_rd[nb] + (uint32_t)(4 * t * BROW)))));
    }
  };
  auto mfma_one = [&](int s, int i) __attribute__((always_inline)) {
    const int nb = i / MB, mb = i % MB;
    const u32x4 b = {bf[s][nb][0].x, bf[s][nb][0].y, bf[s][nb][1].x, bf[s][nb][1].y};
    mma16<T>(acc[mb][nb], b, af[s][mb]);
  };

#pragma unroll
  for (int s = 0; s < NST - 1; ++s) {
#pragma unroll
    for (int j = 0; j < PER; ++j) load_one(lds0 + s * STAGE, j);
    if (s == 0 && ends_first) {  // on to block 0, kt_hi - 1 blocks
      a_voff -= (uint32_t)(n_kt * AROW);
      a_left += (kt_hi - 1) * BK - (p.k - n_kt * BK);
      b_soff = b_left > 0 ? 0 : b_end;
    }
  }
  // While the first stages are on their way.  Not by an MFMA: where the accumulators
  // fill every AGPR the register allocator may move one aside here, and would read it
  // before the MFMA has written it.
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) mma_zero(acc[i][j]);
  wait_vmcnt<(NST - 2) * PER>();
  lds_barrier();
  if (ends_first) {
    const int row = threadIdx.x, left = p.k & 7;
    if (row < TM) {
      lds_u32x4* const at = (lds_u32x4*)(lds + row * AROW + (((p.k % BK / 8) ^ ((row >> 2) & 3)) << 4));
      u32x4 w = *at;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (e >= left) w[e / 2] &= e & 1 ? 0x0000ffffu : 0xffff0000u;
      *at = w;
    }
    lds_barrier();
  }
#pragma unroll
  for (int i = 0; i < NRD; ++i) read_one(0, 0, i);

  constexpr int NM = MB * NB;
  constexpr int NJ = NRD + PER;      // reads and loads of a stage, dealt over its
  constexpr int NS = NM - NM / 8;    // first MFMAs: the last reads land under the rest
  uint32_t nxt = STAGE;               // byte base of the buffer of stage kt + 1
  uint32_t fill = (NST - 1) * STAGE;  // of the one to fill: stage kt + NST - 1
  // Stage kt (its operands in set s): its MFMAs, with the next stage's operand
  // reads and the loads of stage kt + NST - 1 between them.
  auto stage = [&](int s) __attribute__((always_inline)) {
    // stage kt + 1 has landed (this wave's part; the barrier covers the others')
    // and every wave holds stage kt's operands and has left kt - 1's buffer
    wait_vmcnt<(NST - 3) * PER>();
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      mfma_one(s, i);
#pragma unroll
      for (int j = i * NJ / NS; j < (i + 1) * NJ / NS && j < NJ; ++j) {
        if ((j + 1) * PER / NJ != j * PER / NJ) load_one(lds0 + fill, j * PER / NJ);
        else read_one(nxt, s ^ 1, j - j * PER / NJ);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    nxt = nxt + STAGE == NST * STAGE ? 0 : nxt + STAGE;
    fill = fill + STAGE == NST * STAGE ? 0 : fill + STAGE;
  };
  // by twos: with an odd count the last stage is all zeros
  for (int kt = kt_lo; kt < kt_hi; kt += 2) {
    stage(0);
    stage(1);
  }
  mma_drain();
  wait_vmcnt<0>();
  lds_barrier();

  // Lane (lc, g) holds row 16 mb + lc of the wave's block and columns 16 nb +
  // 4 g + 0..3.  The scheduling barriers keep the accumulators in AGPRs until
  // each is used.
  const int mw = m_tile + 16 * MB * wm, nw = n_tile + 16 * NB * wn;  // the wave's corner
  if (p.ksplit > 1) {
    // fp32 partials of this K-slice; n_g is a multiple of 4 here
    float* wsb = p.ws + p.ws_off[grp] + (int64_t)ks * p.m * pn;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = mw + 16 * mb + lc;
      float* row = wsb + (int64_t)m * pn;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int n = nw + 16 * nb + 4 * g;
        if (m < p.m && n < pn) *(f32x4*)(row + n) = mma_take(acc[mb][nb]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
  Bits* cbase = (Bits*)p.G.c[grp];
  const int64_t pldc = p.G.ldc[grp];
  if ((p.vec_store >> grp) & 1) {
    // Through LDS, 32 rows at a time, so that a store instruction writes whole
    // row pieces: 16 NB columns, 16 bytes a lane.
    constexpr int CH = 2 * NB;               // 16-byte chunks of a row piece
    constexpr int STRIDE = 32 * NB + 16;     // bytes; the pad spreads the rows over the banks
    constexpr int RB = 2;                    // row blocks a pass
    static_assert(4 * 16 * RB * STRIDE <= NST * STAGE, "the staging rows fit");
    __attribute__((address_space(3))) char* const mine = lds + wave * (16 * RB * STRIDE);
#pragma unroll
    for (int m2 = 0; m2 < MB / RB; ++m2) {
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const f32x4 v = mma_take(acc[RB * m2 + r][nb]);
          const float x0[2] = {v[0], v[1]}, x1[2] = {v[2], v[3]};
          *(lds_u32x2*)(mine + (16 * r + lc) * STRIDE + 32 * nb + 8 * g) = u32x2{pack2<T>(x0), pack2<T>(x1)};
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int i = 0; i < 16 * RB * CH / 64; ++i) {
        const int at = 64 * i + lane;
        const int r = at / CH, c = at % CH;
        const u32x4 w = *(lds_u32x4*)(mine + r * STRIDE + 16 * c);
        const int m = mw + 16 * RB * m2 + r, n = nw + 8 * c;
        if (m < p.m && n < pn) *(u32x4*)(cbase + (int64_t)m * pldc + n) = w;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_sched_barrier(0);
    }
    return;
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int m = mw + 16 * mb + lc;
    Bits* row = cbase + (int64_t)m * pldc;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const f32x4 v = mma_take(acc[mb][nb]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = nw + 16 * nb + 4 * g + r;
        if (m < p.m && n < pn) row[n] = from_f32<T>(v[r]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace

WidePlan gemm_wide_plan(int m, int k, const GemmGroups& G, int min_split, int max_split) {
  WidePlan best{};
  const int cus = tl_device_cus();
  const int stages = (k + 31) / 32;
  int64_t ncols = 0;
  for (int g = 0; g < G.count; ++g) ncols += G.n[g];
  double t_best = 0;
  for (WidePlan c : kWidePlans) {
    int64_t tiles = 0;
    for (int g = 0; g < G.count; ++g) tiles += (int64_t)((m + c.tm - 1) / c.tm) * ((G.n[g] + c.tn - 1) / c.tn);
    for (int S = min_split; S <= max_split && (S == min_split || stages >= 4 * S); ++S) {
      c.ksplit = S;
      c.kt_per = (stages + S - 1) / S;
      const double reduce = S > 1 ? (8.0 * S + 2) * m * (double)ncols / 8.0e6 + 2.5 + 0.2 * S : 0.0;
      const double t = (double)((tiles * S + cus - 1) / cus) * (c.tile_us + c.kt_per * c.stage_us) + reduce;
      if (best.tm == 0 || t < t_best) {
        best = c;
        t_best = t;
      }
    }
  }
  return best;
}

namespace {
template <typename T>
void launch(const GemmParams& p, const WidePlan& w, hipStream_t st) {
  const dim3 grid((unsigned)(8 * p.per_xcd)), block(256);
  if (w.tm == 256)
    hipLaunchKernelGGL((gemm_wide_kernel<T, 8, 8, 5>), grid, block, 0, st, p);
  else if (w.tm == 192)
    hipLaunchKernelGGL((gemm_wide_kernel<T, 6, 8, 5>), grid, block, 0, st, p);
  else if (w.tm == 64)
    hipLaunchKernelGGL((gemm_wide_kernel<T, 2, 4, 12>), grid, block, 0, st, p);
  else if (w.tn == 256)
    hipLaunchKernelGGL((gemm_wide_kernel<T, 4, 8, 6>), grid, block, 0, st, p);
  else if (w.tn == 192)
    hipLaunchKernelGGL((gemm_wide_kernel<T, 4, 6, 8>), grid, block, 0, st, p);
  else
    hipLaunchKernelGGL((gemm_wide_kernel<T, 4, 4, 8>), grid, block, 0, st, p);
}
}  // namespace

int launch_gemm_wide(const GemmParams& p, const WidePlan& w, int dtype, hipStream_t st) {
  if (dtype == TL_DTYPE_BF16)
    launch<BF16>(p, w, st);
  else
    launch<F16>(p, w, st);
  return tl_launch_status();
}

}  // namespace tlg
