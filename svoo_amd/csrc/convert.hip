// Element-type conversion at the operator boundary.  The hot path computes in bf16 (the MFMA operand type of
// every kernel here) on rows of 128 elements; fp16 and fp32 inputs are rounded to bf16 (to nearest even, through
// fp32, which holds both exactly), rows of a smaller head dim are padded with zeros, and results go back to the
// caller's type and row width.  Memory-bound: each lane moves 8 consecutive elements (16 or 32 bytes) where the
// buffers start at 16-byte addresses and the row widths are multiples of 8; other buffers go one element per lane.
// Measured on fp16 rows of 64 to bf16 rows of 128, 80056 rows (31 MB): 22.3 us one element per lane (a 64-bit division
// each), 8.2 here; fp32 to bf16 at 1.2 million elements 4.5 us either way (the launch).
#include "svoo_common.h"

namespace svoo {

enum ElemType { kElemBf16 = 0, kElemF16 = 1, kElemF32 = 2 };

template <int S>
__device__ __forceinline__ float load_elem(const void* __restrict__ p, long long i) {
  if (S == kElemBf16) return bf16_to_f32(((const uint16_t*)p)[i]);
  if (S == kElemF16) return (float)__builtin_bit_cast(_Float16, ((const uint16_t*)p)[i]);
  return ((const float*)p)[i];
}

template <int D>
__device__ __forceinline__ void store_elem(void* __restrict__ p, long long i, float v) {
  if (D == kElemBf16) ((uint16_t*)p)[i] = f32_to_bf16(v);
  else if (D == kElemF16) ((uint16_t*)p)[i] = __builtin_bit_cast(uint16_t, (_Float16)v);
  else ((float*)p)[i] = v;
}

template <int S>
__device__ __forceinline__ void load8(const void* __restrict__ p, long long v, float (&f)[8]) {
  if (S == kElemF32) {
    const f32x4_t a = ((const f32x4_t*)p)[2 * v], b = ((const f32x4_t*)p)[2 * v + 1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = a[e];
      f[4 + e] = b[e];
    }
  } else {
    const u32x4_t w = ((const u32x4_t*)p)[v];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint16_t b = (uint16_t)(w[e / 2] >> (16 * (e & 1)));
      f[e] = S == kElemBf16 ? bf16_to_f32(b) : (float)__builtin_bit_cast(_Float16, b);
    }
  }
}

template <int D>
__device__ __forceinline__ void store8(void* __restrict__ p, long long v, const float (&f)[8]) {
  if (D == kElemF32) {
    ((f32x4_t*)p)[2 * v] = f32x4_t{f[0], f[1], f[2], f[3]};
    ((f32x4_t*)p)[2 * v + 1] = f32x4_t{f[4], f[5], f[6], f[7]};
  } else {
    u32x4_t w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint16_t lo = D == kElemBf16 ? f32_to_bf16(f[2 * e]) : __builtin_bit_cast(uint16_t, (_Float16)f[2 * e]);
      const uint16_t hi = D == kElemBf16 ? f32_to_bf16(f[2 * e + 1]) : __builtin_bit_cast(uint16_t, (_Float16)f[2 * e + 1]);
      w[e] = (uint32_t)lo | ((uint32_t)hi << 16);
    }
    ((u32x4_t*)p)[v] = w;
  }
}

// n / 8 vectors, the last n % 8 elements one per lane.
template <int S, int D>
__global__ void __launch_bounds__(256) convert8_kernel(const void* __restrict__ src, void* __restrict__ dst,
                                                       long long n) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x, stride = (long long)gridDim.x * blockDim.x;
  for (long long v = t; v < n / 8; v += stride) {
    float f[8];
    load8<S>(src, v, f);
    store8<D>(dst, v, f);
  }
  if (t < n % 8) store_elem<D>(dst, n - 1 - t, load_elem<S>(src, n - 1 - t));
}

// Rows of vs vectors to rows of vd vectors, nv vectors in all (nv < 2^31).
template <int S, int D>
__global__ void __launch_bounds__(256) convert_rows8_kernel(const void* __restrict__ src, uint32_t vs,
                                                            void* __restrict__ dst, uint32_t vd, uint32_t nv) {
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += stride) {
    const uint32_t r = v / vd, c = v - r * vd;
    float f[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (c < vs) load8<S>(src, (long long)r * vs + c, f);
    store8<D>(dst, v, f);
  }
}

template <int S, int D>
__global__ void __launch_bounds__(256) convert_kernel(const void* __restrict__ src, void* __restrict__ dst,
                                                      long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    store_elem<D>(dst, i, load_elem<S>(src, i));
}

// Rows of src_cols elements to rows of dst_cols: the first min(src_cols, dst_cols) converted, the rest zero.
template <int S, int D>
__global__ void __launch_bounds__(256) convert_rows_kernel(const void* __restrict__ src, int src_cols,
                                                           void* __restrict__ dst, int dst_cols, long long n) {
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const long long r = i / dst_cols;
    const int c = (int)(i - r * dst_cols);
    store_elem<D>(dst, i, c < src_cols ? load_elem<S>(src, r * src_cols + c) : 0.0f);
  }
}

static unsigned blocks_for(long long threads) { return (unsigned)min(max((threads + 255) / 256, 1ll), 65536ll); }
static bool aligned16(const void* a, const void* b) { return (((uintptr_t)a | (uintptr_t)b) & 15) == 0; }

template <int S, int D>
static void launch_rows(const void* src, int src_cols, void* dst, int dst_cols, long long n, hipStream_t s) {
  if (aligned16(src, dst) && src_cols % 8 == 0 && dst_cols % 8 == 0 && n / 8 < (1ll << 31))
    hipLaunchKernelGGL((convert_rows8_kernel<S, D>), dim3(blocks_for(n / 8)), dim3(256), 0, s, src,
                       (uint32_t)src_cols / 8, dst, (uint32_t)dst_cols / 8, (uint32_t)(n / 8));
  else
    hipLaunchKernelGGL((convert_rows_kernel<S, D>), dim3(blocks_for(n)), dim3(256), 0, s, src, src_cols, dst,
                       dst_cols, n);
}

template <int S, int D>
static void launch_flat(const void* src, void* dst, long long n, hipStream_t s) {
  if (aligned16(src, dst))
    hipLaunchKernelGGL((convert8_kernel<S, D>), dim3(blocks_for(n / 8)), dim3(256), 0, s, src, dst, n);
  else
    hipLaunchKernelGGL((convert_kernel<S, D>), dim3(blocks_for(n)), dim3(256), 0, s, src, dst, n);
}

template <int S>
static void launch_rows_from(const void* src, int src_cols, int dst_type, void* dst, int dst_cols, long long n,
                             hipStream_t s) {
  if (dst_type == kElemBf16) launch_rows<S, kElemBf16>(src, src_cols, dst, dst_cols, n, s);
  else if (dst_type == kElemF16) launch_rows<S, kElemF16>(src, src_cols, dst, dst_cols, n, s);
  else launch_rows<S, kElemF32>(src, src_cols, dst, dst_cols, n, s);
}

template <int S>
static void launch_from(const void* src, int dst_type, void* dst, long long n, hipStream_t s) {
  if (dst_type == kElemBf16) launch_flat<S, kElemBf16>(src, dst, n, s);
  else if (dst_type == kElemF16) launch_flat<S, kElemF16>(src, dst, n, s);
  else launch_flat<S, kElemF32>(src, dst, n, s);
}

}  // namespace svoo

using namespace svoo;

extern "C" int svoo_convert(const void* src, int src_type, void* dst, int dst_type, long long n, void* stream) {
  SVOO_REQUIRE(src_type >= kElemBf16 && src_type <= kElemF32 && dst_type >= kElemBf16 && dst_type <= kElemF32,
               SVOO_ERR_INVALID_ARG, "svoo_convert: element types %d -> %d (0 bf16, 1 fp16, 2 fp32)", src_type,
               dst_type);
  SVOO_REQUIRE(n >= 0, SVOO_ERR_INVALID_ARG, "svoo_convert: n=%lld", n);
  if (n == 0) return SVOO_OK;
  SVOO_REQUIRE(src && dst, SVOO_ERR_INVALID_ARG, "svoo_convert: null pointer");
  hipStream_t s = (hipStream_t)stream;
  if (src_type == kElemBf16) launch_from<kElemBf16>(src, dst_type, dst, n, s);
  else if (src_type == kElemF16) launch_from<kElemF16>(src, dst_type, dst, n, s);
  else launch_from<kElemF32>(src, dst_type, dst, n, s);
  return check_launch("svoo_convert");
}

extern "C" int svoo_convert_rows(const void* src, int src_type, int src_cols, void* dst, int dst_type, int dst_cols,
                                 long long rows, void* stream) {
  SVOO_REQUIRE(src_type >= kElemBf16 && src_type <= kElemF32 && dst_type >= kElemBf16 && dst_type <= kElemF32,
               SVOO_ERR_INVALID_ARG, "svoo_convert_rows: element types %d -> %d (0 bf16, 1 fp16, 2 fp32)", src_type,
               dst_type);
  SVOO_REQUIRE(rows >= 0 && src_cols > 0 && dst_cols > 0, SVOO_ERR_INVALID_ARG,
               "svoo_convert_rows: rows=%lld src_cols=%d dst_cols=%d", rows, src_cols, dst_cols);
  const long long n = rows * dst_cols;
  if (n == 0) return SVOO_OK;
  SVOO_REQUIRE(src && dst, SVOO_ERR_INVALID_ARG, "svoo_convert_rows: null pointer");
  hipStream_t s = (hipStream_t)stream;
  if (src_type == kElemBf16) launch_rows_from<kElemBf16>(src, src_cols, dst_type, dst, dst_cols, n, s);
  else if (src_type == kElemF16) launch_rows_from<kElemF16>(src, src_cols, dst_type, dst, dst_cols, n, s);
  else launch_rows_from<kElemF32>(src, src_cols, dst_type, dst, dst_cols, n, s);
  return check_launch("svoo_convert_rows");
}
