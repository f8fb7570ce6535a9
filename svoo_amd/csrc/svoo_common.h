// Shared device helpers and host error plumbing for the SVOO HIP kernels (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/svoo_hip.h"

namespace svoo {

constexpr int kWave = 64;

// ---------------------------------------------------------------- bf16 <-> f32
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

// Round-to-nearest-even float32 -> bfloat16 bit pattern (NaN -> quiet NaN).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)0x7fc0u;
  uint32_t lsb = (u >> 16) & 1u;
  return (uint16_t)((u + 0x7fffu + lsb) >> 16);
}

__device__ __forceinline__ float bf16_round_f32(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// ---------------------------------------------------------------- vector types for MFMA
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16x8_t as_bf16x8(u32x4_t v) { return __builtin_bit_cast(bf16x8_t, v); }

// 32x32x16 bf16 MFMA, fp32 accumulate.  Operand layout (wave64):
//   A[m][k]: lane m + 32*(k/8), element k%8     B[k][n]: lane n + 32*(k/8), element k%8
//   C[m][n]: lane n + 32*((m/4)%2), element (m/8)*4 + m%4
__device__ __forceinline__ f32x16_t mfma32x32x16(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16x16x32 bf16 MFMA.  A[m][k]: lane m + 16*(k/8); C[m][n]: lane n + 16*(m/4), element m%4.
__device__ __forceinline__ f32x4_t mfma16x16x32(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 16x16x4 fp64 MFMA.  A[i][k]: lane i + 16 k; B[k][j]: lane j + 16 k; D[i][j]: lane j + 16 (i % 4),
// element i / 4 (measured by svoo_probe_mfma_f64_layout).
typedef double f64x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f64x4_t mfma16x16x4_f64(double a, double b, f64x4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return (uint32_t)f32_to_bf16(lo) | ((uint32_t)f32_to_bf16(hi) << 16);
}

// Two floats -> packed bf16 pair with the gfx950 conversion instruction (v_cvt_pk_bf16_f32,
// round to nearest even); same values as pack_bf16x2 for every non-NaN input.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){lo, hi}, bf16x2_t));
}

// gfx950 transposing LDS read (ds_read_b64_tr_b16).  Within each group of 16 lanes, lane i of the
// group receives element e (e = 0..3) = element i%4 of the 8 bytes read by group lane 4e + i/4.
// With group lane s addressing row (r0 + s/4), columns (c0 + 4*(s%4) .. +3) of a row-major bf16
// matrix, lane i receives rows r0..r0+3 of column c0 + i.
typedef short i16x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 ds_read_tr16_b64(const uint16_t* lds_ptr) {
  const i16x4_t r =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(lds_ptr));
  return __builtin_bit_cast(uint2, r);
}

// Physical 16-byte chunk of logical chunk c in row r of an LDS tile of unpadded 256-byte rows.  The
// XOR pattern makes both read patterns used here conflict-free: 16 consecutive rows at one chunk
// (MFMA A-operand rows via ds_read_b128) and 4 consecutive rows x 4 consecutive chunks (the
// transposing reads).
__device__ __forceinline__ int swz(int r, int c) { return c ^ (((r & 3) << 2) | ((r >> 2) & 3)); }

// Direct global -> LDS copy of 16 bytes per lane: lane i writes lds_base + 16 i (gfx950 LDS DMA,
// global_load_lds_dwordx4).  lds_base must be wave-uniform; completion is tracked by vmcnt.
__device__ __forceinline__ void lds_dma16(const void* src, uint16_t* lds_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)lds_base, 16, 0, 0);
}

// The same copy issued from inline assembly: 16 bytes per lane from sbase + voff (bytes) to LDS byte address
// lds + 16 * lane (sbase and lds wave-uniform).  The compiler neither sees nor counts it, so its waits for the
// kernel's own LDS reads stay exact (it treats a visible LDS DMA as an LDS event that may complete out of
// order and answers every later LDS read with lgkmcnt(0)).  The caller waits for completion explicitly
// (s_waitcnt vmcnt) before the barrier that publishes the data.  M0 needs one wait state after its write.
__device__ __forceinline__ void lds_dma16_asm(const void* sbase, uint32_t voff, uint32_t lds) {
  __asm__ volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds)
                   : "memory", "m0");
}
// LDS byte address of a __shared__ object, wave-uniform.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p);
}

// Max / sum of a value and its partner lane (lane ^ 32), in both lanes: one v_permlane32_swap (a VALU
// op) instead of a ds_bpermute round trip through LDS.  The swap returns {lanes 0-31 of the first operand
// with lanes 0-31 of the second in the upper half, lanes 32-63 of the first in the lower half with lanes
// 32-63 of the second}; with both operands x, each lane sees x of itself and of its partner.
__device__ __forceinline__ float xhalf_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// ---------------------------------------------------------------- float64 exponential from a table
// 2^(i / 64), i = 0 .. 63, as the nearest double and the nearest to what that leaves; kernels keep a copy in LDS.
static __device__ const double2 kExp2Table[64] = {
    {0x1.0000000000000p+0, 0.0}, {0x1.02c9a3e778061p+0, -0x1.19083535b085dp-56},
    {0x1.059b0d3158574p+0, 0x1.d73e2a475b465p-55}, {0x1.0874518759bc8p+0, 0x1.186be4bb284ffp-57},
    {0x1.0b5586cf9890fp+0, 0x1.8a62e4adc610bp-54}, {0x1.0e3ec32d3d1a2p+0, 0x1.03a1727c57b53p-59},
    {0x1.11301d0125b51p+0, -0x1.6c51039449b3ap-54}, {0x1.1429aaea92de0p+0, -0x1.32fbf9af1369ep-54},
    {0x1.172b83c7d517bp+0, -0x1.19041b9d78a76p-55}, {0x1.1a35beb6fcb75p+0, 0x1.e5b4c7b4968e4p-55},
    {0x1.1d4873168b9aap+0, 0x1.e016e00a2643cp-54}, {0x1.2063b88628cd6p+0, 0x1.dc775814a8495p-55},
    {0x1.2387a6e756238p+0, 0x1.9b07eb6c70573p-54}, {0x1.26b4565e27cddp+0, 0x1.2bd339940e9d9p-55},
    {0x1.29e9df51fdee1p+0, 0x1.612e8afad1255p-55}, {0x1.2d285a6e4030bp+0, 0x1.0024754db41d5p-54},
    {0x1.306fe0a31b715p+0, 0x1.6f46ad23182e4p-55}, {0x1.33c08b26416ffp+0, 0x1.32721843659a6p-54},
    {0x1.371a7373aa9cbp+0, -0x1.63aeabf42eae2p-54}, {0x1.3a7db34e59ff7p+0, -0x1.5e436d661f5e3p-56},
    {0x1.3dea64c123422p+0, 0x1.ada0911f09ebcp-55}, {0x1.4160a21f72e2ap+0, -0x1.ef3691c309278p-58},
    {0x1.44e086061892dp+0, 0x1.89b7a04ef80d0p-59}, {0x1.486a2b5c13cd0p+0, 0x1.3c1a3b69062f0p-56},
    {0x1.4bfdad5362a27p+0, 0x1.d4397afec42e2p-56}, {0x1.4f9b2769d2ca7p+0, -0x1.4b309d25957e3p-54},
    {0x1.5342b569d4f82p+0, -0x1.07abe1db13cadp-55}, {0x1.56f4736b527dap+0, 0x1.9bb2c011d93adp-54},
    {0x1.5ab07dd485429p+0, 0x1.6324c054647adp-54}, {0x1.5e76f15ad2148p+0, 0x1.ba6f93080e65ep-54},
    {0x1.6247eb03a5585p+0, -0x1.383c17e40b497p-54}, {0x1.6623882552225p+0, -0x1.bb60987591c34p-54},
    {0x1.6a09e667f3bcdp+0, -0x1.bdd3413b26456p-54}, {0x1.6dfb23c651a2fp+0, -0x1.bbe3a683c88abp-57},
    {0x1.71f75e8ec5f74p+0, -0x1.16e4786887a99p-55}, {0x1.75feb564267c9p+0, -0x1.0245957316dd3p-54},
    {0x1.7a11473eb0187p+0, -0x1.41577ee04992fp-55}, {0x1.7e2f336cf4e62p+0, 0x1.05d02ba15797ep-56},
    {0x1.82589994cce13p+0, -0x1.d4c1dd41532d8p-54}, {0x1.868d99b4492edp+0, -0x1.fc6f89bd4f6bap-54},
    {0x1.8ace5422aa0dbp+0, 0x1.6e9f156864b27p-54}, {0x1.8f1ae99157736p+0, 0x1.5cc13a2e3976cp-55},
    {0x1.93737b0cdc5e5p+0, -0x1.75fc781b57ebcp-57}, {0x1.97d829fde4e50p+0, -0x1.d185b7c1b85d1p-54},
    {0x1.9c49182a3f090p+0, 0x1.c7c46b071f2bep-56}, {0x1.a0c667b5de565p+0, -0x1.359495d1cd533p-54},
    {0x1.a5503b23e255dp+0, -0x1.d2f6edb8d41e1p-54}, {0x1.a9e6b5579fdbfp+0, 0x1.0fac90ef7fd31p-54},
    {0x1.ae89f995ad3adp+0, 0x1.7a1cd345dcc81p-54}, {0x1.b33a2b84f15fbp+0, -0x1.2805e3084d708p-57},
    {0x1.b7f76f2fb5e47p+0, -0x1.5584f7e54ac3bp-56}, {0x1.bcc1e904bc1d2p+0, 0x1.23dd07a2d9e84p-55},
    {0x1.c199bdd85529cp+0, 0x1.11065895048ddp-55}, {0x1.c67f12e57d14bp+0, 0x1.2884dff483cadp-54},
    {0x1.cb720dcef9069p+0, 0x1.503cbd1e949dbp-56}, {0x1.d072d4a07897cp+0, -0x1.cbc3743797a9cp-54},
    {0x1.d5818dcfba487p+0, 0x1.2ed02d75b3707p-55}, {0x1.da9e603db3285p+0, 0x1.c2300696db532p-54},
    {0x1.dfc97337b9b5fp+0, -0x1.1a5cd4f184b5cp-54}, {0x1.e502ee78b3ff6p+0, 0x1.39e8980a9cc8fp-55},
    {0x1.ea4afa2a490dap+0, -0x1.e9c23179c2893p-54}, {0x1.efa1bee615a27p+0, 0x1.dc7f486a4b6b0p-54},
    {0x1.f50765b6e4540p+0, 0x1.9d3e12dd8a18bp-54}, {0x1.fa7c1819e90d8p+0, 0x1.74853f3a5931ep-55}
};
// exp(x) for x <= 0 (or NaN): 2^(n / 64) from the table times the degree-6 series in |r| <= ln2 / 128 with r^6 replaced
// by the r^4 and r^2 of its Chebyshev expansion (what is dropped is 2^-60).  Within 0.54 units of the last place
// (0.530 over 2x10^7 points; the library's exp is within 0.88 here, and a table of single doubles gives 1.27 with the
// plain degree-5 series; the second double costs the sparsity counts 1%, the block mask nothing).  x below -200 counts
// as -200 (its result is 0 in bf16 and fp32).
__device__ __forceinline__ double exp_tab(const double2* exp2_tab, double x) {
  x = x < -200.0 ? -200.0 : x;  // a NaN stays
  const double nd = __builtin_rint(x * 0x1.71547652b82fep+6);
  const int n = (int)nd;
  double r = fma(nd, -0x1.62e42fefa39efp-7, x);
  r = fma(nd, -0x1.abc9e3b39803fp-62, r);
  double p = fma(r, 1.0 / 120.0, 0x1.55557621dbbb3p-5);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0x1.fffffffffd0bap-2);
  p = fma(p * r, r, r);
  const double2 t = exp2_tab[n & 63];
  return __builtin_ldexp(t.x + fma(t.x, p, t.y), n >> 6);
}

// ---------------------------------------------------------------- wave scans and sums
// Inclusive scan over the wave in the VALU (DPP row shifts and broadcasts; lanes without a source add 0).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add_f64(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, ROWS, 0xf, false);
  return v + __builtin_bit_cast(double, ((unsigned long long)(uint32_t)hi << 32) | (uint32_t)lo);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add_i32(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);
}
// The same within each row of 16 lanes.
__device__ __forceinline__ double row_scan_f64(double v) {
  v = dpp_add_f64<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_add_f64<0x112, 0xf>(v);
  v = dpp_add_f64<0x114, 0xf>(v);
  return dpp_add_f64<0x118, 0xf>(v);
}
__device__ __forceinline__ int row_scan_i32(int v) {
  v = dpp_add_i32<0x111, 0xf>(v);
  v = dpp_add_i32<0x112, 0xf>(v);
  v = dpp_add_i32<0x114, 0xf>(v);
  return dpp_add_i32<0x118, 0xf>(v);
}
__device__ __forceinline__ double wave_scan_f64(double v) {
  v = dpp_add_f64<0x142, 0xa>(row_scan_f64(v));  // row_bcast:15 into rows 1 and 3
  return dpp_add_f64<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
}
__device__ __forceinline__ int wave_scan_i32(int v) {
  v = dpp_add_i32<0x142, 0xa>(row_scan_i32(v));
  return dpp_add_i32<0x143, 0xc>(v);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ long long dpp_add_i64(long long v) {
  const unsigned long long u = (unsigned long long)v;
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, ROWS, 0xf, false);
  return v + (long long)(((unsigned long long)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ long long wave_scan_i64(long long v) {
  v = dpp_add_i64<0x111, 0xf>(v);
  v = dpp_add_i64<0x112, 0xf>(v);
  v = dpp_add_i64<0x114, 0xf>(v);
  v = dpp_add_i64<0x118, 0xf>(v);
  v = dpp_add_i64<0x142, 0xa>(v);
  return dpp_add_i64<0x143, 0xc>(v);
}
// A lane's value in every lane (the lane uniform).
__device__ __forceinline__ long long lane_i64(long long v, int lane) {
  const unsigned long long u = (unsigned long long)v;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return (long long)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// ---------------------------------------------------------------- block reductions
template <int kThreads>
__device__ __forceinline__ double block_sum_f64(double v, double* scratch) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
  __syncthreads();
  if (l == 0) scratch[w] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int i = 0; i < kThreads / kWave; ++i) t += scratch[i];
  return t;
}

template <int kThreads>
__device__ __forceinline__ float block_max_f32(float v, float* scratch) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
  __syncthreads();
  if (l == 0) scratch[w] = v;
  __syncthreads();
  float t = scratch[0];
#pragma unroll
  for (int i = 1; i < kThreads / kWave; ++i) t = fmaxf(t, scratch[i]);
  return t;
}

template <int kThreads>
__device__ __forceinline__ int block_sum_i32(int v, int* scratch) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
  __syncthreads();
  if (l == 0) scratch[w] = v;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int i = 0; i < kThreads / kWave; ++i) t += scratch[i];
  return t;
}

// Exclusive prefix sum over the block (int64); returns this thread's exclusive prefix and writes the total.
template <int kThreads>
__device__ __forceinline__ long long block_exclusive_scan_i64(long long v, long long* scratch, long long* total) {
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
  long long inc = v;
  for (int o = 1; o < kWave; o <<= 1) {
    long long n = __shfl_up(inc, o);
    if (l >= o) inc += n;
  }
  __syncthreads();
  if (l == kWave - 1) scratch[w] = inc;
  __syncthreads();
  long long base = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kThreads / kWave; ++i) {
    if (i < w) base += scratch[i];
    tot += scratch[i];
  }
  *total = tot;
  return base + inc - v;
}

// ---------------------------------------------------------------- host side
void set_error(const char* fmt, ...);
int check_launch(const char* what);

}  // namespace svoo

#define SVOO_REQUIRE(cond, code, ...)     \
  do {                                    \
    if (!(cond)) {                        \
      ::svoo::set_error(__VA_ARGS__);     \
      return (code);                      \
    }                                     \
  } while (0)

// Head dims: rows always hold 128 elements; d (1..128) is the head dim, elements d..127 of every row are zero.
#define SVOO_REQUIRE_HEAD_DIM(d, name)                                                                    \
  SVOO_REQUIRE((d) >= 1 && (d) <= 128, SVOO_ERR_UNSUPPORTED, "%s: D=%d (head dims 1..128, rows of 128)", \
               name, (d))
