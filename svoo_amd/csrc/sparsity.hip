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
//   2. 16 lanes per listed group weigh its 64 counts and sum them (fp64);
//   3. every wave scans the masses of its 64 groups, the waves' totals find the group where the mass from the top first
//      reaches threshold * total, and its wave the crossing value among the group's 64, whose multiplicity is exact.
// All masses are fp64 sums of fp32 weights times counts, so the count does not depend on summation order beyond
// 2^-53 of the mass.
//
// What bounds it: the LDS atomics (one row of n scores is n / 64 wave instructions on one CU) next to the read of the
// row.  One 1024-thread block per CU (the histogram takes most of the LDS) walks rows, the next row's scores already
// in registers while the current one is counted and scanned, so memory and LDS work overlap.  Measured on 12288 rows of
// 32760 scores (805 MB): 9.28 ms with a fp64 exp and a wave-combined LDS update per score (three passes, 256 threads),
// 0.34 ms here (2.3 TB/s); a row costs about 17 thousand cycles, 9 thousand of them independent of its length (9608
// rows of 2402 scores: 0.56 -> 0.16 ms).  Many short rows take exact_count_short_kernel (the rule of short_rows).
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

// float(exp(double(s - m))).  The library's exp costs about three times the instructions of exp_tab, and its constants,
// kept in registers over the loop, spilled.  s <= m, or NaN.
__device__ __forceinline__ float sp_weight(const double2* exp2_tab, uint32_t raw, float scale, float m) {
  const float s = __uint_as_float(raw << 16) * scale;
  return (float)exp_tab(exp2_tab, (double)(s - m));
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
  double2 exp2_tab[64];                 // kExp2Table
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
  if (tid < 64) sh.exp2_tab[tid] = kExp2Table[tid];
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
  if (tid < 64) sh.exp2_tab[tid] = kExp2Table[tid];
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

// ---------------------------------------------------------------- short rows
// One block of 256 threads per row, several per CU, without the table of all patterns: the largest score; a 256-bin
// histogram over the high byte of the key (counts and masses), whose scan finds the bin where the mass from the top
// reaches threshold * total; counts over the low byte inside that bin, each sub-bin one exact value.
constexpr int kShortThreads = 256;

// Bit pattern -> key whose unsigned order is the numeric order.
__device__ __forceinline__ uint32_t short_key(uint16_t b) { return 0xffffu - sp_order(b); }

__device__ __forceinline__ float short_weight(uint32_t raw, float scale, float m) {
  const float s = __uint_as_float(raw << 16) * scale;
  return (float)exp((double)(s - m));
}

// Lanes of a wave with the same bin combine their (count, weight) before one LDS atomic per
// distinct bin: scores concentrate in a few binades, and plain per-lane atomics would serialise.
__device__ __forceinline__ double wave_sum_f64(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ void hist_add(int32_t* cnt, double* mass, int bin, double w, bool valid) {
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long todo = __ballot(valid);
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const int lb = __shfl(bin, leader);
    const bool mine = valid && bin == lb;
    const unsigned long long mm = __ballot(mine);
    const double sum = wave_sum_f64(mine ? w : 0.0);
    if (lane == leader) {
      atomicAdd(&cnt[lb], (int)__popcll(mm));
      atomicAdd(&mass[lb], sum);
    }
    todo &= ~mm;
  }
}
__device__ __forceinline__ void count_add(int32_t* cnt, int bin, bool valid) {
  const int lane = threadIdx.x & (kWave - 1);
  unsigned long long todo = __ballot(valid);
  while (todo) {
    const int leader = __ffsll((long long)todo) - 1;
    const int lb = __shfl(bin, leader);
    const unsigned long long mm = __ballot(valid && bin == lb);
    if (lane == leader) atomicAdd(&cnt[lb], (int)__popcll(mm));
    todo &= ~mm;
  }
}

// Inclusive prefix, from the top bin down, of the 256 bins' masses and counts (thread t holds bin
// 255 - t); a fixed summation order.
__device__ void short_scan(const int32_t* cnt, const double* mass, double* dsc, long long* isc) {
  const int tid = threadIdx.x;
  dsc[tid] = mass[255 - tid];
  isc[tid] = cnt[255 - tid];
  __syncthreads();
  for (int off = 1; off < kShortThreads; off <<= 1) {
    const double dv = tid >= off ? dsc[tid - off] : 0.0;
    const long long iv = tid >= off ? isc[tid - off] : 0;
    __syncthreads();
    dsc[tid] += dv;
    isc[tid] += iv;
    __syncthreads();
  }
}

// The bin (scanned from the top) at which the scanned mass first reaches `target`, with the mass
// and count strictly above it; the lowest non-empty bin when rounding leaves the total below the
// target.  Call after sp_scan.
struct ShortCross {
  int bin;
  double mass_above;
  long long cnt_above;
};
__device__ ShortCross short_find(const int32_t* cnt, double target, const double* dsc, const long long* isc, int* found) {
  const int tid = threadIdx.x;
  if (tid == 0) *found = -1;
  __syncthreads();
  const double above = tid > 0 ? dsc[tid - 1] : 0.0;
  if (cnt[255 - tid] > 0 && above < target && dsc[tid] >= target) *found = tid;
  __syncthreads();
  if (*found < 0) {
    __syncthreads();
    if (tid == 0) {
      int last = 0;
      for (int i = 0; i < kShortThreads; ++i)
        if (cnt[255 - i] > 0) last = i;
      *found = last;
    }
    __syncthreads();
  }
  const int t = *found;
  ShortCross r;
  r.bin = 255 - t;
  r.mass_above = t > 0 ? dsc[t - 1] : 0.0;
  r.cnt_above = t > 0 ? isc[t - 1] : 0;
  __syncthreads();
  return r;
}

__global__ void __launch_bounds__(kShortThreads) exact_count_short_kernel(const uint16_t* __restrict__ scores, int n,
                                                                   float scale, float threshold,
                                                                   int32_t* __restrict__ counts) {
  __shared__ int32_t cnt[256];
  __shared__ double mass[256];
  __shared__ double dsc[kShortThreads];
  __shared__ long long isc[kShortThreads];
  __shared__ int found;
  __shared__ uint32_t kmax_s;
  const size_t row = blockIdx.x;
  const int tid = threadIdx.x;
  const uint16_t* sr = scores + row * (size_t)n;

  // 1. row max as a key
  uint32_t kmax = 0;
  for (int j = tid; j < n; j += kShortThreads) kmax = max(kmax, short_key(sr[j]));
  for (int o = 32; o > 0; o >>= 1) kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o));
  if (tid == 0) kmax_s = 0;
  cnt[tid] = 0;
  mass[tid] = 0.0;
  __syncthreads();
  if ((tid & (kWave - 1)) == 0) atomicMax(&kmax_s, kmax);
  __syncthreads();
  const float m = bf16_to_f32((uint16_t)sp_raw(0xffffu - kmax_s)) * scale;

  // 2. high-byte histogram of counts and weights (whole-wave iterations: every lane takes part)
  for (int j0 = 0; j0 < n; j0 += kShortThreads) {
    const int j = j0 + tid;
    const bool valid = j < n;
    const uint16_t b = valid ? sr[j] : (uint16_t)0;
    const uint32_t k = short_key(b);
    hist_add(cnt, mass, (int)(k >> 8), valid ? (double)short_weight(b, scale, m) : 0.0, valid);
  }
  __syncthreads();
  short_scan(cnt, mass, dsc, isc);
  const double total = dsc[kShortThreads - 1];
  const double target = (double)threshold * total;
  const ShortCross c1 = short_find(cnt, target, dsc, isc, &found);

  // 3. low-byte counts inside the crossing bin; each sub-bin is one exact value
  cnt[tid] = 0;
  __syncthreads();
  for (int j0 = 0; j0 < n; j0 += kShortThreads) {
    const int j = j0 + tid;
    const uint32_t k = j < n ? short_key(sr[j]) : 0u;
    count_add(cnt, (int)(k & 255), j < n && (int)(k >> 8) == c1.bin);
  }
  __syncthreads();
  {
    const int sb = 255 - tid;
    mass[sb] = (double)cnt[sb] * (double)short_weight(sp_raw(0xffffu - (((uint32_t)c1.bin << 8) | (uint32_t)sb)), scale, m);
  }
  __syncthreads();
  short_scan(cnt, mass, dsc, isc);
  const double rem = target - c1.mass_above;
  const ShortCross c2 = short_find(cnt, rem, dsc, isc, &found);
  if (tid == 0) {
    const double v = (double)short_weight(sp_raw(0xffffu - (((uint32_t)c1.bin << 8) | (uint32_t)c2.bin)), scale, m);
    const int mult = cnt[c2.bin];
    const double need = rem - c2.mass_above;
    long long k = 1;
    if (v > 0.0 && need > 0.0) {
      k = (long long)ceil(need / v);
      // the smallest k with k * v >= need (the division may round either way)
      while (k > 1 && (double)(k - 1) * v >= need) --k;
      while (k < mult && (double)k * v < need) ++k;
    }
    k = k < 1 ? 1 : (k > mult ? mult : k);
    counts[row] = (int32_t)(c1.cnt_above + c2.cnt_above + k);
  }
}

}  // namespace svoo

using namespace svoo;

// Short rows go to the kernel of several small blocks per CU once there are rows enough: the histogram's rows cost one
// CU about 3.7 us each whatever their length, in rounds of 256 rows, the small blocks' 9-15 us in all plus a share that
// grows with the length.  Histogram -> small blocks: 64 scores 6.3 -> 10.5 us at 256 rows, 13.3 -> 10.8 at 513, 178 ->
// 75 at 12288; 257 scores 10.5 -> 12.2 at 500, 17.7 -> 15.2 at 769; 385 scores 18.7 -> 20.8 at 1024, 36.7 -> 34.8 at
// 2049; 513 scores 193 -> 186 at 12288; 600 scores 194 -> 216 at 12288, and always behind from there on.
static bool short_rows(long long rows, int n) {
  if (n > 544) return false;
  return rows > 256 * (n <= 32 ? 1 : n <= 256 ? 2 : n <= 288 ? 3 : n <= 448 ? 8 : n <= 512 ? 16 : 32);
}

extern "C" int svoo_exact_sparsity_counts(const uint16_t* scores, long long rows, int n, float scale, float threshold,
                                          int32_t* counts, void* stream) {
  SVOO_REQUIRE(scores && counts, SVOO_ERR_INVALID_ARG, "svoo_exact_sparsity_counts: null pointer");
  SVOO_REQUIRE(rows > 0 && rows < (1ll << 31) && n > 0, SVOO_ERR_INVALID_ARG,
               "svoo_exact_sparsity_counts: bad dims rows=%lld n=%d", rows, n);
  SVOO_REQUIRE(threshold > 0.0f && threshold <= 1.0f, SVOO_ERR_INVALID_ARG,
               "svoo_exact_sparsity_counts: threshold %g outside (0, 1]", (double)threshold);
  hipStream_t s = (hipStream_t)stream;
  if (short_rows(rows, n)) {
    hipLaunchKernelGGL(exact_count_short_kernel, dim3((unsigned)rows), dim3(kShortThreads), 0, s, scores, n, scale,
                       threshold, counts);
    return check_launch("svoo_exact_sparsity_counts");
  }
  // One block per CU (256 on MI355X): the histogram fills the LDS, and the rows are dealt round robin.
  const dim3 grid((unsigned)(rows < 256 ? rows : 256)), block(kSpThreads);
#define SVOO_COUNT(K) hipLaunchKernelGGL(K, grid, block, 0, s, scores, (uint32_t)rows, n, scale, threshold, counts)
  if (n > kSpSingle) SVOO_COUNT(exact_count_long_kernel);
  else if (n <= 8 * kSpThreads) SVOO_COUNT(exact_count_kernel<1>);
  else if (n <= 32 * kSpThreads) SVOO_COUNT(exact_count_kernel<4>);
  else SVOO_COUNT(exact_count_kernel<8>);
#undef SVOO_COUNT
  return check_launch("svoo_exact_sparsity_counts");
}
