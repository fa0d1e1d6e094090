// The model step's elementwise and row-reduction layers around the
// projections: RMSNorm, residual add + RMSNorm fused, SwiGLU, add.
//
// Reference behaviour being replaced:
//   * rms_norm (triton_llm/kernels/rms_norm.py:21-116): one program per row,
//     rms = sqrt(sum(x^2) / N + eps), y = (x / rms) * w (:47-56);
//   * swiglu (swiglu.py:21-125): silu(x) * y with the single-exp stable
//     sigmoid, exp(-|x|) (:46-54);
//   * add (add.py:14-104): z = x + y.
// In the model every RMSNorm after the first of a layer reads the sum the
// residual add just wrote (smollm2_triton/model.py:352-357 and the next
// layer's :279-280); tl_add_rms_norm does both in one pass over the row,
// writing the sum (the next residual) and the normalised row.
//
// All are HBM-bound (or launch-bound at decode sizes): 16 bytes a lane, lanes
// contiguous, fp32 arithmetic whatever the storage type.
#include "tl_common.h"

#include <math.h>

namespace {

constexpr int kRowThreads = 256;
constexpr int kEltThreads = 256;

template <typename T>
__device__ __forceinline__ float ld(const void* p, int64_t i) {
  return to_f32<T>(((const typename T::bits*)p)[i]);
}
template <typename T>
__device__ __forceinline__ void st(void* p, int64_t i, float x) {
  ((typename T::bits*)p)[i] = from_f32<T>(x);
}

__device__ __forceinline__ float block_sum(float v, float* s_red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_red[wave] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < kRowThreads / 64; ++w) t += s_red[w];
  return t;
}

// 16 bytes of T <-> fp32 (4 or 8 elements); the rounding is from_f32's.
template <typename T>
constexpr int kVec = 16 / T::size;

template <typename T>
__device__ __forceinline__ void unpack16(const u32x4& w, float (&f)[kVec<T>]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (T::size == 4) f[i] = __uint_as_float(w[i]);
    else unpack2<T>(w[i], f[2 * i], f[2 * i + 1]);
  }
}
template <typename T>
__device__ __forceinline__ u32x4 pack16(const float (&f)[kVec<T>]) {
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (T::size == 4) w[i] = __float_as_uint(f[i]);
    else w[i] = (uint32_t)from_f32<T>(f[2 * i]) | (uint32_t)from_f32<T>(f[2 * i + 1]) << 16;
  }
  return w;
}

// Rows of whole 16-byte chunks on 16-byte aligned pointers: one workgroup per
// row, CH chunks per thread (chunk tid + 256 j) in registers, so the row is
// read once; w's chunks are loaded with it, so that their latency does not
// follow the reduction's.  HBM-bound for a prompt: add + RMSNorm of 2048 x
// 3072 bf16 rows (50 MB) 21.8 -> 14.5 us, of 64 rows 5.2 -> 4.9, one fp32 row
// of 960 3.3 -> 2.0 us (the chain of dependent loads), against two- or
// four-byte accesses, one element a lane.  With b != nullptr the row is a + b,
// written to h and normalised as stored, i.e. after rounding to T.
template <typename T, int CH>
__global__ __launch_bounds__(kRowThreads) void rms_norm_vec_kernel(const void* a, const void* b, void* h, const void* w,
                                                                   void* y, int n, float eps) {
  __shared__ float s_red[kRowThreads / 64];
  constexpr int V = kVec<T>;
  const int chunks = n / V;
  const int64_t row = (int64_t)blockIdx.x * chunks;
  float x[CH][V];
  u32x4 av[CH], bv[CH], wv[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {  // every load of the row in flight before the first is used
    const int i = threadIdx.x + kRowThreads * j;
    av[j] = bv[j] = wv[j] = u32x4{0, 0, 0, 0};
    if (i < chunks) {
      av[j] = ((const u32x4*)a)[row + i];
      if (b) bv[j] = ((const u32x4*)b)[row + i];
      wv[j] = ((const u32x4*)w)[i];
    }
  }
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    unpack16<T>(av[j], x[j]);
    if (b) {
      const int i = threadIdx.x + kRowThreads * j;
      float s[V];
      unpack16<T>(bv[j], s);
#pragma unroll
      for (int e = 0; e < V; ++e) s[e] += x[j][e];
      const u32x4 r = pack16<T>(s);
      if (i < chunks) ((u32x4*)h)[row + i] = r;
      unpack16<T>(r, x[j]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < CH; ++j)
#pragma unroll
    for (int e = 0; e < V; e += 4)  // fours, so that no sum is a longer chain than the scalar kernel's
      ss += (x[j][e] * x[j][e] + x[j][e + 1] * x[j][e + 1]) + (x[j][e + 2] * x[j][e + 2] + x[j][e + 3] * x[j][e + 3]);
  const float rms = sqrtf(block_sum(ss, s_red) / (float)n + eps);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    const int i = threadIdx.x + kRowThreads * j;
    if (i < chunks) {
      float wf[V], o[V];
      unpack16<T>(wv[j], wf);
#pragma unroll
      for (int e = 0; e < V; ++e) o[e] = (x[j][e] / rms) * wf[e];
      ((u32x4*)y)[row + i] = pack16<T>(o);
    }
  }
}

// Rows of any length and alignment, up to 256 * VPT elements.
// One workgroup per row, the row held in registers (VPT elements per
// thread, element tid + 256 j), so it is read from memory once.  With
// b != nullptr the row is a + b, written to h (the residual for the next add)
// and normalised as stored, i.e. after rounding to T, as a separate add then
// RMSNorm would.  Rows longer than 256 * 32 take rms_norm_kernel below.
template <typename T, int VPT>
__global__ __launch_bounds__(kRowThreads) void rms_norm_row_kernel(const void* a, const void* b, void* h, const void* w,
                                                                   void* y, int n, float eps) {
  __shared__ float s_red[kRowThreads / 64];
  const int64_t row = (int64_t)blockIdx.x * n;
  float x[VPT];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int i = threadIdx.x + kRowThreads * j;
    float v = 0.f;
    if (i < n) {
      v = ld<T>(a, row + i);
      if (b) {
        const typename T::bits r = from_f32<T>(v + ld<T>(b, row + i));
        ((typename T::bits*)h)[row + i] = r;
        v = to_f32<T>(r);
      }
    }
    x[j] = v;
    ss += v * v;
  }
  const float rms = sqrtf(block_sum(ss, s_red) / (float)n + eps);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    const int i = threadIdx.x + kRowThreads * j;
    if (i < n) st<T>(y, row + i, (x[j] / rms) * ld<T>(w, i));
  }
}

// Any row length: two passes over the row (the second mostly from L2).
template <typename T>
// No __restrict__: callers may update the residual in place (h == a) or
// normalise in place (y == x); every element is read before it is written by
// the same thread.
__global__ __launch_bounds__(kRowThreads) void rms_norm_kernel(const void* a, const void* b, void* h, const void* w,
                                                               void* y, int n, float eps) {
  __shared__ float s_red[kRowThreads / 64];
  const int64_t row = (int64_t)blockIdx.x * n;
  float ss = 0.f;
  for (int i = threadIdx.x; i < n; i += kRowThreads) {
    float x = ld<T>(a, row + i);
    if (b) {
      x += ld<T>(b, row + i);
      st<T>(h, row + i, x);
      x = ld<T>(h, row + i);  // normalise the stored (rounded) sum, as a separate add then RMSNorm would
    }
    ss += x * x;
  }
  const float rms = sqrtf(block_sum(ss, s_red) / (float)n + eps);
  const void* src = b ? (const void*)h : a;
  for (int i = threadIdx.x; i < n; i += kRowThreads) st<T>(y, row + i, (ld<T>(src, row + i) / rms) * ld<T>(w, i));
}

// n / d for d in [1, 2] and n in [0, 1], bit for bit what the IEEE division
// gives: its reciprocal, Newton step and two residual corrections, without the
// scaling and special cases that no such operand needs (every n below 2^-25
// comes with d == 1 here, where each step is exact).
__device__ __forceinline__ float div_unit(float n, float d) {
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.f), r, r);
  float q = n * r;
  q = fmaf(fmaf(-d, q, n), r, q);
  return fmaf(fmaf(-d, q, n), r, q);
}

// silu(x) * u with the single-exp stable sigmoid: exp(-|x|) <= 1 never
// overflows, and one division serves both signs.
struct SwigluOp {
  template <typename T>
  static __device__ __forceinline__ float apply(float x, float u) {
    const float e = expf(-fabsf(x));
    return x * div_unit(x >= 0.f ? 1.f : e, 1.f + e) * u;
  }
};
struct AddOp {
  template <typename T>
  static __device__ __forceinline__ float apply(float x, float y) { return x + y; }
};

// out[i] = Op(x[i], y[i]), HBM-bound: 2048 x 8192 bf16 SwiGLU (100 MB) 38.9 ->
// 18.9 us (5.3 TB/s), 2048 x 3072 add (38 MB) 17.8 -> 8.4 us against one
// element a lane.  VEC: 16-byte aligned operands, 16 bytes a lane,
// the last count % kVec elements by the lanes after them; otherwise one
// element a lane.  In place (out == x or y) is fine: a lane reads what it
// writes first.
template <typename T, typename Op, bool VEC>
__global__ __launch_bounds__(kEltThreads) void binary_kernel(const void* x, const void* y, void* out, int64_t count) {
  const int64_t step = (int64_t)gridDim.x * kEltThreads;
  const int64_t t0 = (int64_t)blockIdx.x * kEltThreads + threadIdx.x;
  if constexpr (VEC) {
    constexpr int V = kVec<T>;
    const int64_t nv = count / V;
    const int tail = (int)(count - nv * V);
    for (int64_t i = t0; i < nv + tail; i += step) {
      if (i < nv) {
        float a[V], b[V], o[V];
        unpack16<T>(((const u32x4*)x)[i], a);
        unpack16<T>(((const u32x4*)y)[i], b);
#pragma unroll
        for (int e = 0; e < V; ++e) o[e] = Op::template apply<T>(a[e], b[e]);
        ((u32x4*)out)[i] = pack16<T>(o);
      } else {
        const int64_t k = nv * V + (i - nv);
        st<T>(out, k, Op::template apply<T>(ld<T>(x, k), ld<T>(y, k)));
      }
    }
  } else {
    for (int64_t i = t0; i < count; i += step) st<T>(out, i, Op::template apply<T>(ld<T>(x, i), ld<T>(y, i)));
  }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

bool dtype_ok(int dtype) { return dtype == TL_DTYPE_F32 || dtype == TL_DTYPE_F16 || dtype == TL_DTYPE_BF16; }

template <template <typename> class Launch, typename... Args>
int by_dtype(int dtype, Args... args) {
  switch (dtype) {
    case TL_DTYPE_F32: return Launch<F32>::run(args...);
    case TL_DTYPE_F16: return Launch<F16>::run(args...);
    default: return Launch<BF16>::run(args...);
  }
}

template <typename T>
struct RmsLaunch {
  static int run(const void* a, const void* b, void* h, const void* w, void* y, int m, int n, float eps, hipStream_t st) {
    const dim3 grid((unsigned)m), block(kRowThreads);
    constexpr int V = kVec<T>;
    const int per = kRowThreads * V;  // elements of one chunk a thread
    if (n % V == 0 && n <= 8 * per && aligned16(a) && aligned16(w) && aligned16(y) &&
        (!b || (aligned16(b) && aligned16(h)))) {
      if (n <= per)
        hipLaunchKernelGGL((rms_norm_vec_kernel<T, 1>), grid, block, 0, st, a, b, h, w, y, n, eps);
      else if (n <= 2 * per)
        hipLaunchKernelGGL((rms_norm_vec_kernel<T, 2>), grid, block, 0, st, a, b, h, w, y, n, eps);
      else if (n <= 4 * per)
        hipLaunchKernelGGL((rms_norm_vec_kernel<T, 4>), grid, block, 0, st, a, b, h, w, y, n, eps);
      else
        hipLaunchKernelGGL((rms_norm_vec_kernel<T, 8>), grid, block, 0, st, a, b, h, w, y, n, eps);
    } else if (n <= kRowThreads * 4)
      hipLaunchKernelGGL((rms_norm_row_kernel<T, 4>), grid, block, 0, st, a, b, h, w, y, n, eps);
    else if (n <= kRowThreads * 8)
      hipLaunchKernelGGL((rms_norm_row_kernel<T, 8>), grid, block, 0, st, a, b, h, w, y, n, eps);
    else if (n <= kRowThreads * 16)
      hipLaunchKernelGGL((rms_norm_row_kernel<T, 16>), grid, block, 0, st, a, b, h, w, y, n, eps);
    else if (n <= kRowThreads * 32)
      hipLaunchKernelGGL((rms_norm_row_kernel<T, 32>), grid, block, 0, st, a, b, h, w, y, n, eps);
    else
      hipLaunchKernelGGL((rms_norm_kernel<T>), grid, block, 0, st, a, b, h, w, y, n, eps);
    return tl_launch_status();
  }
};
template <typename T, typename Op>
int launch_binary(const void* x, const void* y, void* out, int64_t count, hipStream_t st) {
  const bool vec = aligned16(x) && aligned16(y) && aligned16(out);
  const int64_t items = vec ? count / kVec<T> + count % kVec<T> : count;
  const int64_t b = (items + kEltThreads - 1) / kEltThreads;
  const dim3 grid((unsigned)(b < 65536 ? b : 65536));
  if (vec)
    hipLaunchKernelGGL((binary_kernel<T, Op, true>), grid, dim3(kEltThreads), 0, st, x, y, out, count);
  else
    hipLaunchKernelGGL((binary_kernel<T, Op, false>), grid, dim3(kEltThreads), 0, st, x, y, out, count);
  return tl_launch_status();
}
template <typename T>
struct SwigluLaunch {
  static int run(const void* g, const void* u, void* o, int64_t count, hipStream_t st) {
    return launch_binary<T, SwigluOp>(g, u, o, count, st);
  }
};
template <typename T>
struct AddLaunch {
  static int run(const void* x, const void* y, void* z, int64_t count, hipStream_t st) {
    return launch_binary<T, AddOp>(x, y, z, count, st);
  }
};

}  // namespace

extern "C" {

int tl_rms_norm(const void* x, const void* w, void* y, int m, int n, float eps, int dtype, void* stream) {
  if (m < 0 || n < 0 || !dtype_ok(dtype)) return TL_ERR_INVALID;
  if (m == 0) return 0;
  if (n == 0 || !x || !w || !y) return TL_ERR_INVALID;
  return by_dtype<RmsLaunch>(dtype, x, (const void*)nullptr, (void*)nullptr, w, y, m, n, eps, tl_resolve_stream(stream));
}

int tl_add_rms_norm(const void* a, const void* b, void* h, const void* w, void* y, int m, int n, float eps, int dtype,
                    void* stream) {
  if (m < 0 || n < 0 || !dtype_ok(dtype)) return TL_ERR_INVALID;
  if (m == 0) return 0;
  if (n == 0 || !a || !b || !h || !w || !y) return TL_ERR_INVALID;
  return by_dtype<RmsLaunch>(dtype, a, b, h, w, y, m, n, eps, tl_resolve_stream(stream));
}

int tl_swiglu(const void* gate, const void* up, void* out, int64_t count, int dtype, void* stream) {
  if (count < 0 || !dtype_ok(dtype)) return TL_ERR_INVALID;
  if (count == 0) return 0;
  if (!gate || !up || !out) return TL_ERR_INVALID;
  return by_dtype<SwigluLaunch>(dtype, gate, up, out, count, tl_resolve_stream(stream));
}

int tl_add(const void* x, const void* y, void* z, int64_t count, int dtype, void* stream) {
  if (count < 0 || !dtype_ok(dtype)) return TL_ERR_INVALID;
  if (count == 0) return 0;
  if (!x || !y || !z) return TL_ERR_INVALID;
  return by_dtype<AddLaunch>(dtype, x, y, z, count, tl_resolve_stream(stream));
}

}  // extern "C"
