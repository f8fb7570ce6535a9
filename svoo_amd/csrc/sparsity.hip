// Exact attention sparsity of one query row (the offline profile producer).
//
// For a row of scaled scores s_j (bf16 scores times scale, as the reference's fp32 softmax input)
// the count is the smallest c such that the c largest softmax weights hold at least `threshold` of
// the row's mass.  Softmax weights are exp(s_j - m) / Z with m the row max, so the count is the same
// for the unnormalised weights e_j = exp(s_j - m), computed here as float(exp(double(s_j - m))).
//
// Scores are bf16, so a row holds at most 65536 distinct values, and equal values have equal weights: the row is
// first counted into a histogram of the 65536 bit patterns (16-bit counts, 128 KB of LDS, one LDS atomic per score),
// and everything after that works on the distinct values, in descending order of value:
//   1. the non-empty groups of 64 patterns are listed (about 130 of 1024 for scores of one scale);
//   2. per listed group the wave's 64 lanes weigh the 64 counts and sum them (fp64);
//   3. one wave scans the group masses to the group where the mass from the top first reaches threshold * total,
//      and the 64 values of that group to the crossing value, whose multiplicity is exact.
// All masses are fp64 sums of fp32 weights times counts, so the count does not depend on summation order beyond
// 2^-53 of the mass.
//
// What bounds it: the LDS atomics (one row of n scores is n / 64 wave instructions on one CU) next to the read of the
// row.  One 1024-thread block per CU (the histogram takes most of the LDS) walks rows, the next row's scores already
// in registers while the current one is counted and scanned, so memory and LDS work overlap.  Measured on 12288 rows of
// 32760 scores (805 MB): 9.28 ms with a fp64 exp and a wave-combined LDS update per score (three passes, 256 threads),
// 0.34 ms here (2.3 TB/s); a row costs about 17 thousand cycles, 9 thousand of them independent of its length (9608
// rows of 2402 scores: 0.56 -> 0.16 ms).
#include "svoo_common.h"

namespace svoo {

constexpr int kSpThreads = 1024;
constexpr int kSpWaves = kSpThreads / kWave;
constexpr int kSpGroups = 1024;          // groups of 64 bit patterns
constexpr int kSpSingle = 65535;         // longest row whose 16-bit counts cannot overflow
constexpr int kSpMultiVecs = 4;          // longer rows: segments of 4 * 1024 vectors of 8 scores

// Bit pattern of order o: o = 0 is the largest value (patterns 0x7fff .. 0x0000, then 0x8000 .. 0xffff), so the
// patterns of one 64-group of o are one aligned 64-group of patterns, reversed for the non-negative half.
__device__ __forceinline__ uint32_t sp_order(uint32_t b) { return (b & 0x8000u) ? b : 0x7fffu - b; }
__device__ __forceinline__ uint32_t sp_raw(uint32_t o) { return o < 0x8000u ? 0x7fffu - o : o; }
// First pattern of wave w's 64 groups (orders 4096 w ..).
__device__ __forceinline__ int sp_base(int w) { return (int)sp_raw((uint32_t)w * 4096) & ~4095; }

// 2^(i / 64), i = 0 .. 63, correctly rounded; the kernels keep a copy in LDS.
__device__ const double kSpExp2[64] = {
    0x1.0000000000000p+0, 0x1.02c9a3e778061p+0, 0x1.059b0d3158574p+0, 0x1.0874518759bc8p+0,
    0x1.0b5586cf9890fp+0, 0x1.0e3ec32d3d1a2p+0, 0x1.11301d0125b51p+0, 0x1.1429aaea92de0p+0,
    0x1.172b83c7d517bp+0, 0x1.1a35beb6fcb75p+0, 0x1.1d4873168b9aap+0, 0x1.2063b88628cd6p+0,
    0x1.2387a6e756238p+0, 0x1.26b4565e27cddp+0, 0x1.29e9df51fdee1p+0, 0x1.2d285a6e4030bp+0,
    0x1.306fe0a31b715p+0, 0x1.33c08b26416ffp+0, 0x1.371a7373aa9cbp+0, 0x1.3a7db34e59ff7p+0,
    0x1.3dea64c123422p+0, 0x1.4160a21f72e2ap+0, 0x1.44e086061892dp+0, 0x1.486a2b5c13cd0p+0,
    0x1.4bfdad5362a27p+0, 0x1.4f9b2769d2ca7p+0, 0x1.5342b569d4f82p+0, 0x1.56f4736b527dap+0,
    0x1.5ab07dd485429p+0, 0x1.5e76f15ad2148p+0, 0x1.6247eb03a5585p+0, 0x1.6623882552225p+0,
    0x1.6a09e667f3bcdp+0, 0x1.6dfb23c651a2fp+0, 0x1.71f75e8ec5f74p+0, 0x1.75feb564267c9p+0,
    0x1.7a11473eb0187p+0, 0x1.7e2f336cf4e62p+0, 0x1.82589994cce13p+0, 0x1.868d99b4492edp+0,
    0x1.8ace5422aa0dbp+0, 0x1.8f1ae99157736p+0, 0x1.93737b0cdc5e5p+0, 0x1.97d829fde4e50p+0,
    0x1.9c49182a3f090p+0, 0x1.a0c667b5de565p+0, 0x1.a5503b23e255dp+0, 0x1.a9e6b5579fdbfp+0,
    0x1.ae89f995ad3adp+0, 0x1.b33a2b84f15fbp+0, 0x1.b7f76f2fb5e47p+0, 0x1.bcc1e904bc1d2p+0,
    0x1.c199bdd85529cp+0, 0x1.c67f12e57d14bp+0, 0x1.cb720dcef9069p+0, 0x1.d072d4a07897cp+0,
    0x1.d5818dcfba487p+0, 0x1.da9e603db3285p+0, 0x1.dfc97337b9b5fp+0, 0x1.e502ee78b3ff6p+0,
    0x1.ea4afa2a490dap+0, 0x1.efa1bee615a27p+0, 0x1.f50765b6e4540p+0, 0x1.fa7c1819e90d8p+0
};
// float(exp(double(s - m))): 2^(n / 64) from the table times a polynomial in |r| <= ln2 / 128 (its next term is below
// 2^-54), within one unit of the last place of the float64 exponential.  The library's exp costs about three times
// the instructions, and its constants, kept in registers over the loop, spilled.  s <= m, or NaN.
__device__ __forceinline__ float sp_weight(const double* exp2_tab, uint32_t raw, float scale, float m) {
  const float s = __uint_as_float(raw << 16) * scale;
  double x = (double)(s - m);
  x = x < -200.0 ? -200.0 : x;  // 0 as a float well before; a NaN stays
  const double nd = __builtin_rint(x * 0x1.71547652b82fep+6);
  const int n = (int)nd;
  double r = fma(nd, -0x1.62e42fefa39efp-7, x);
  r = fma(nd, -0x1.abc9e3b39803fp-62, r);
  double p = fma(r, 1.0 / 120.0, 1.0 / 24.0);
  p = fma(p, r, 1.0 / 6.0);
  p = fma(p, r, 0.5);
  p = fma(p * r, r, r);
  const double t = exp2_tab[n & 63];
  const double y = fma(t, p, t);
  return (float)__builtin_ldexp(y, n >> 6);
}

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
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), lane);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// The wave's number, and a value that is the same in its lanes, in scalar registers.
__device__ __forceinline__ int sp_wave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave); }
__device__ __forceinline__ unsigned long long uniform_u64(unsigned long long v) {
  return ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32) |
         (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
}

struct SpShared {
  uint32_t hist[32768];                // pattern b: 16 bits at half b & 1 of word b >> 1
  double mass[kSpGroups];              // per group of orders: the mass of its scores
  int32_t cnt[kSpGroups];              // and their number
  double exp2_tab[64];                 // kSpExp2
  double wmass[kSpWaves];              // the same per wave's 64 groups
  int32_t wcnt[kSpWaves];
  uint16_t list[kSpGroups];            // non-empty groups, from the top
  unsigned long long mask[kSpWaves];   // wave w's 64 groups (from the top): non-empty ones
  unsigned long long any[kSpWaves];    // long rows: the union of the masks over the segments
  uint32_t fine[kWave];                // long rows: the counts of the crossing group
  uint32_t wmax[kSpWaves];
  int cross;
};

__device__ __forceinline__ void sp_count(uint32_t* hist, uint32_t b) {
  atomicAdd(&hist[b >> 1], 1u << ((b & 1u) * 16));
}
__device__ __forceinline__ uint32_t sp_get(const uint32_t* hist, uint32_t b) {
  return (hist[b >> 1] >> ((b & 1u) * 16)) & 0xffffu;
}

// A row's scores as 16-byte vectors from its first aligned address, up to 7 scores before and after them.
struct SpRow {
  const uint16_t* p;
  int head, nvec, tail;
};
__device__ __forceinline__ SpRow sp_row(const uint16_t* scores, size_t row, int n) {
  SpRow r;
  r.p = scores + row * (size_t)n;
  r.head = min(n, (int)(((16 - ((uintptr_t)r.p & 15)) & 15) / 2));
  r.nvec = (n - r.head) / 8;
  r.tail = n - r.head - 8 * r.nvec;
  return r;
}
// The single scores of a row: thread t < head holds score t, thread 8 <= t < 8 + tail one of the last.
__device__ __forceinline__ bool sp_has_edge(const SpRow& r, int tid) {
  return tid < r.head || (tid >= 8 && tid < 8 + r.tail);
}
__device__ __forceinline__ uint16_t sp_edge(const SpRow& r, int tid) {
  return r.p[tid < r.head ? tid : r.head + 8 * r.nvec + tid - 8];
}

// Lists the non-empty groups and weighs them into sh.mass / sh.cnt (added with ACC).  The
// histogram is complete and visible on entry; on return the sums are not yet (the caller's barrier).
template <bool ACC>
__device__ __forceinline__ void sp_groups(SpShared& sh, float scale, float& m) {
  const int wave = sp_wave(), lane = threadIdx.x % kWave;
  const int base = sp_base(wave);
  bool full = false;                             // pattern group `lane` of them is non-empty
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const u32x4_t w = *(const u32x4_t*)(sh.hist + base / 2 + s * 256 + lane * 4);
    const unsigned long long b = __ballot((w[0] | w[1] | w[2] | w[3]) != 0u);
    if ((lane >> 3) == s) full = ((b >> (8 * (lane & 7))) & 0xffull) != 0ull;
  }
  unsigned long long mk = __ballot(full);
  if (wave < kSpWaves / 2) mk = __brevll(mk);  // the non-negative half runs downwards
  if (lane == 0) sh.mask[wave] = mk;
  __syncthreads();
  // the waves' numbers of groups, scanned by every row of 16 lanes
  const int inc = row_scan_i32((int)__popcll(sh.mask[lane % 16]));
  const int total = __builtin_amdgcn_readlane(inc, 15);
  const int off = __builtin_amdgcn_readlane(inc, wave) - (int)__popcll(mk);
  if ((mk >> lane) & 1ull) sh.list[off + (int)__popcll(mk & ((1ull << lane) - 1ull))] = (uint16_t)(wave * 64 + lane);
  __syncthreads();
  if (!ACC) {  // the largest value: first non-empty pattern of the first group
    const uint32_t o = (uint32_t)sh.list[0] * 64;
    const unsigned long long b = __ballot(sp_get(sh.hist, sp_raw(o + lane)) != 0u);
    m = __uint_as_float(sp_raw(o + (uint32_t)__ffsll((long long)b) - 1u) << 16) * scale;
  }
  // four groups at a time, 16 lanes of 4 patterns each
  for (int i0 = 4 * wave; i0 < total; i0 += 4 * kSpWaves) {
    const int i = i0 + lane / 16;
    const int g = sh.list[min(i, total - 1)];
    const uint32_t raw = (sp_raw((uint32_t)g * 64) & ~63u) + (uint32_t)(lane % 16) * 4;
    const uint2 w = *(const uint2*)(sh.hist + raw / 2);
    const uint32_t c[4] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16};
    double v = 0.0;
    int cs = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v += c[e] ? (double)c[e] * (double)sp_weight(sh.exp2_tab, raw + e, scale, m) : 0.0;
      cs += (int)c[e];
    }
    v = row_scan_f64(v);
    cs = row_scan_i32(cs);
    if (lane % 16 == 15 && i < total) {
      sh.mass[g] = ACC ? sh.mass[g] + v : v;
      sh.cnt[g] = ACC ? sh.cnt[g] + cs : cs;
    }
  }
}

// Every wave clears the counts of its own 64 groups (those that hold any), two per store.
__device__ __forceinline__ void sp_clear(SpShared& sh) {
  const int wave = sp_wave(), lane = threadIdx.x % kWave;
  unsigned long long mk = uniform_u64(sh.mask[wave]);
  if (wave < kSpWaves / 2) mk = __brevll(mk);  // by pattern
  uint32_t* h = sh.hist + sp_base(wave) / 2 + lane;
  while (mk != 0ull) {
    const int l = (__ffsll((long long)mk) - 1) & ~1;
    h[l * 32] = 0u;
    mk &= ~(3ull << l);
  }
}

// The group where the mass from the top first reaches threshold * total (the last one when rounding leaves the total
// below it): every wave scans its own 64 groups (those in `mask`), and the waves' totals place them.  Returns the group
// in the wave that holds it, -1 in the others; `rem` is what its values must reach, `above` the scores above it.
__device__ __forceinline__ int sp_cross(SpShared& sh, const unsigned long long* mask, float threshold, double* rem,
                                        long long* above) {
  const int wave = sp_wave(), lane = threadIdx.x % kWave;
  const unsigned long long mk = uniform_u64(mask[wave]);
  const bool in = (mk >> lane) & 1ull;
  const double vs = wave_scan_f64(in ? sh.mass[wave * 64 + lane] : 0.0);
  const int cs = wave_scan_i32(in ? sh.cnt[wave * 64 + lane] : 0);
  if (lane == kWave - 1) {
    sh.wmass[wave] = vs;
    sh.wcnt[wave] = cs;
  }
  __syncthreads();
  // the waves' totals, scanned by every row of 16 lanes
  const double run = row_scan_f64(sh.wmass[lane % 16]);
  const int crun = row_scan_i32(sh.wcnt[lane % 16]);
  const double target = (double)threshold * lane_f64(run, 15);
  const uint32_t reach = (uint32_t)__ballot(run >= target) & 0xffffu;
  const uint32_t some = (uint32_t)__ballot(mask[lane % 16] != 0ull) & 0xffffu;
  const uint32_t hit = reach & some;
  const int at = hit != 0u ? __ffs((int)hit) - 1 : 31 - __clz((int)some);
  if (at != wave) return -1;
  const double base = wave > 0 ? lane_f64(run, max(wave - 1, 0)) : 0.0;
  const double v = base + vs;
  const unsigned long long up = (unsigned long long)__ballot(v >= target) & mk;
  // rounding can leave the wave's last group below what its total reached: the last group then
  const int l = (hit == 0u || up == 0ull) ? 63 - (int)__clzll((long long)mk) : __ffsll((long long)up) - 1;
  *rem = target - (l > 0 ? lane_f64(v, max(l - 1, 0)) : base);
  *above = (wave > 0 ? __builtin_amdgcn_readlane(crun, max(wave - 1, 0)) : 0) +
           (l > 0 ? __builtin_amdgcn_readlane(cs, max(l - 1, 0)) : 0);
  return wave * 64 + l;
}

// One wave: the count of a row whose crossing group holds c[lane] scores of its 64 values.
__device__ __forceinline__ void sp_finish(const SpShared& sh, int g, int c, double rem, long long above, float scale, float m,
                                          int32_t* out) {
  const int lane = threadIdx.x % kWave;
  const float w = sp_weight(sh.exp2_tab, sp_raw((uint32_t)g * 64 + lane), scale, m);
  const double v = wave_scan_f64(c ? (double)c * (double)w : 0.0);
  const int cs = wave_scan_i32(c);
  const double ab = __shfl_up(v, 1);
  const double before = lane > 0 ? ab : 0.0;
  const unsigned long long some = __ballot(c > 0);
  const unsigned long long hit = __ballot(c > 0 && before < rem && v >= rem);
  const int l = hit != 0ull ? __ffsll((long long)hit) - 1 : 63 - (int)__clzll((long long)some);
  if (lane == l) {
    const double need = rem - before, wd = (double)w;
    long long k = 1;
    if (wd > 0.0 && need > 0.0) {
      k = (long long)ceil(need / wd);
      // the smallest k with k * w >= need (the division may round either way)
      while (k > 1 && (double)(k - 1) * wd >= need) --k;
      while (k < c && (double)k * wd < need) ++k;
    }
    k = k < 1 ? 1 : (k > c ? c : k);
    *out = (int32_t)(above + (long long)(cs - c) + k);
  }
}

// Rows of at most kSpSingle scores: NV vectors of 8 scores per thread, loaded one row ahead.
template <int NV>
__global__ void __launch_bounds__(kSpThreads) exact_count_kernel(const uint16_t* __restrict__ scores, uint32_t rows, int n,
                                                                 float scale, float threshold,
                                                                 int32_t* __restrict__ counts) {
  __shared__ __attribute__((aligned(16))) SpShared sh;
  const int tid = threadIdx.x, lane = tid % kWave;
  for (int i = tid; i < 32768 / 4; i += kSpThreads) ((u32x4_t*)sh.hist)[i] = u32x4_t{0u, 0u, 0u, 0u};
  if (tid < 64) sh.exp2_tab[tid] = kSpExp2[tid];
  u32x4_t v[NV];
  uint16_t edge = 0;
  auto load = [&](uint32_t row) {
    const SpRow r = sp_row(scores, row, n);
    const u32x4_t* src = (const u32x4_t*)(r.p + r.head);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (i * kSpThreads + tid < r.nvec) v[i] = src[i * kSpThreads + tid];
    if (sp_has_edge(r, tid)) edge = sp_edge(r, tid);
  };
  if (blockIdx.x < rows) load(blockIdx.x);
  __syncthreads();
  for (uint32_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const SpRow r = sp_row(scores, row, n);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (i * kSpThreads + tid < r.nvec) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sp_count(sh.hist, v[i][e] & 0xffffu);
          sp_count(sh.hist, v[i][e] >> 16);
        }
      }
    if (sp_has_edge(r, tid)) sp_count(sh.hist, edge);
    if (row + gridDim.x < rows) load(row + gridDim.x);
    __syncthreads();
    float m = 0.0f;
    sp_groups<false>(sh, scale, m);
    __syncthreads();
    double rem;
    long long above;
    const int g = sp_cross(sh, sh.mask, threshold, &rem, &above);
    const int c = g >= 0 ? (int)sp_get(sh.hist, sp_raw((uint32_t)g * 64 + lane)) : 0;
    sp_clear(sh);
    __syncthreads();
    // the other waves go on to the next row meanwhile
    if (g >= 0) sp_finish(sh, g, c, rem, above, scale, m, counts + row);
  }
}

// Longer rows: the maximum first, then the histogram segment by segment (each at most 32782 scores) with the group
// masses added up, and the crossing group counted again over the row in 32 bits.
__global__ void __launch_bounds__(kSpThreads) exact_count_long_kernel(const uint16_t* __restrict__ scores, uint32_t rows,
                                                                      int n, float scale, float threshold,
                                                                      int32_t* __restrict__ counts) {
  __shared__ __attribute__((aligned(16))) SpShared sh;
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  for (int i = tid; i < 32768 / 4; i += kSpThreads) ((u32x4_t*)sh.hist)[i] = u32x4_t{0u, 0u, 0u, 0u};
  if (tid < 64) sh.exp2_tab[tid] = kSpExp2[tid];
  for (uint32_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const SpRow r = sp_row(scores, row, n);
    const u32x4_t* src = (const u32x4_t*)(r.p + r.head);
    uint32_t omin = 0xffffu;
    for (int i = tid; i < r.nvec; i += kSpThreads) {
      const u32x4_t w = src[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) omin = min(omin, min(sp_order(w[e] & 0xffffu), sp_order(w[e] >> 16)));
    }
    if (sp_has_edge(r, tid)) omin = min(omin, sp_order(sp_edge(r, tid)));
    for (int o = 32; o > 0; o >>= 1) omin = min(omin, (uint32_t)__shfl_xor((int)omin, o));
    sh.mass[tid] = 0.0;
    sh.cnt[tid] = 0;
    if (lane == 0) sh.wmax[wave] = omin;
    if (tid < kSpWaves) sh.any[tid] = 0ull;
    if (tid < kWave) sh.fine[tid] = 0u;
    __syncthreads();
    for (int w = 0; w < kSpWaves; ++w) omin = min(omin, sh.wmax[w]);
    float m = __uint_as_float(sp_raw(omin) << 16) * scale;
    for (int v0 = 0; v0 < r.nvec; v0 += kSpMultiVecs * kSpThreads) {
#pragma unroll
      for (int i = 0; i < kSpMultiVecs; ++i) {
        const int at = v0 + i * kSpThreads + tid;
        if (at < r.nvec) {
          const u32x4_t w = src[at];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            sp_count(sh.hist, w[e] & 0xffffu);
            sp_count(sh.hist, w[e] >> 16);
          }
        }
      }
      if (v0 == 0 && sp_has_edge(r, tid)) sp_count(sh.hist, sp_edge(r, tid));
      __syncthreads();
      sp_groups<true>(sh, scale, m);
      if (tid < kSpWaves) sh.any[tid] |= sh.mask[tid];
      __syncthreads();
      sp_clear(sh);
      __syncthreads();
    }
    double rem = 0.0;
    long long above = 0;
    const int mine = sp_cross(sh, sh.any, threshold, &rem, &above);
    if (mine >= 0 && lane == 0) sh.cross = mine;
    __syncthreads();
    const uint32_t g = (uint32_t)sh.cross;
    auto again = [&](uint32_t b) {
      const uint32_t o = sp_order(b);
      if ((o >> 6) == g) atomicAdd(&sh.fine[o & 63u], 1u);
    };
    for (int i = tid; i < r.nvec; i += kSpThreads) {
      const u32x4_t w = src[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        again(w[e] & 0xffffu);
        again(w[e] >> 16);
      }
    }
    if (sp_has_edge(r, tid)) again(sp_edge(r, tid));
    __syncthreads();
    if (mine >= 0) sp_finish(sh, (int)g, (int)sh.fine[lane], rem, above, scale, m, counts + row);
    __syncthreads();
  }
}

}  // namespace svoo

using namespace svoo;

extern "C" int svoo_exact_sparsity_counts(const uint16_t* scores, long long rows, int n, float scale, float threshold,
                                          int32_t* counts, void* stream) {
  SVOO_REQUIRE(scores && counts, SVOO_ERR_INVALID_ARG, "svoo_exact_sparsity_counts: null pointer");
  SVOO_REQUIRE(rows > 0 && rows < (1ll << 31) && n > 0, SVOO_ERR_INVALID_ARG,
               "svoo_exact_sparsity_counts: bad dims rows=%lld n=%d", rows, n);
  SVOO_REQUIRE(threshold > 0.0f && threshold <= 1.0f, SVOO_ERR_INVALID_ARG,
               "svoo_exact_sparsity_counts: threshold %g outside (0, 1]", (double)threshold);
  // One block per CU (256 on MI355X): the histogram fills the LDS, and the rows are dealt round robin.
  const dim3 grid((unsigned)(rows < 256 ? rows : 256)), block(kSpThreads);
  hipStream_t s = (hipStream_t)stream;
#define SVOO_COUNT(K) hipLaunchKernelGGL(K, grid, block, 0, s, scores, (uint32_t)rows, n, scale, threshold, counts)
  if (n > kSpSingle) SVOO_COUNT(exact_count_long_kernel);
  else if (n <= 8 * kSpThreads) SVOO_COUNT(exact_count_kernel<1>);
  else if (n <= 32 * kSpThreads) SVOO_COUNT(exact_count_kernel<4>);
  else SVOO_COUNT(exact_count_kernel<8>);
#undef SVOO_COUNT
  return check_launch("svoo_exact_sparsity_counts");
}
