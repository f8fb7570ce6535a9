// Centroid scores and the block-mask builder.
//
// centroid_scores_kernel (one 4-wave block per 32 key centroids of a head):
//   t_ij = bf16(f32(bf16(Qc_i . Kc_j)) * f32(1/sqrt(D)))   the reference's bf16 matmul, then "/ D**0.5"
//   The dot runs on the bf16 MFMA, one k-step (16 exact products) per accumulator, and the eight partial
//   sums are added in fp64; a second MFMA over |Qc| and |Kc| gives a = sum |q_d k_d|.  Each partial is
//   the fp32 rounding of at most 16 additions, so |r - s| <= 16 * 2^-24 * a; with e = 2^-19 a (twice that,
//   which also covers the fp32 error of a itself and the rounding of the fp64 sum to fp32) every value in
//   [r - e, r + e] rounds (via fp32) to the same bf16 as the exact dot s when its two ends do.  The entries
//   that fail this test (2-3% of them on centroid data), or whose rows hold bf16 subnormals (which the MFMA
//   may flush), are computed exactly in fp64: by their lane, or (for the mask) by the mask kernel.
//
// block_mask_kernel (one 256-thread block per (b, h, q-cluster) row) and block_mask_wave_kernel (one wave per row, for
// many rows of at most 1024 clusters):
//   p_j  = bf16(f32(w_j e^(t_j - max) / max(sum, 1e-12)))   weighted softmax, evaluated in fp64
//   order (p desc, j asc), found by two-level histograms of the bf16 bits of p (no sort)
//   prefix_t = sum_{u<=t} floor(p_u * 2^60)  (exact int64) -> bf16 -> compared with bf16(top_p)
//   kept length L = max(1 + #{t <= Kc-2 : prefix_t <= p}, preserve_h), capped by cap_h
// and the first L clusters of that order are written back as 1 in the bool map.
#include "svoo_common.h"

namespace svoo {

constexpr int kMaskThreads = 256;
constexpr int kWaveRows = 2048;  // rows from which a wave each is faster than a block each (svoo_block_mask)

constexpr int kScoreThreads = 256;

// Dot of two bf16 rows of 128 in fp64 by 16 lanes (aligned groups of 16; lane c of the group takes the
// 16-byte chunk c of both rows): the products are exact in fp64, and so is their sum while the products'
// exponents span less than 2^30 (beyond that the sum is rounded in a fixed order).  Every lane of the group
// returns the dot.  `valid` may differ between groups; all 64 lanes must call it together.
__device__ __forceinline__ double group16_dot128(const uint16_t* __restrict__ x, const uint16_t* __restrict__ y,
                                                 bool valid) {
  const int c = threadIdx.x % 16;
  double acc = 0.0;
  if (valid) {
    const u32x4_t a = ((const u32x4_t*)x)[c], b = ((const u32x4_t*)y)[c];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc = fma((double)bf16_to_f32((uint16_t)(a[e] & 0xffffu)), (double)bf16_to_f32((uint16_t)(b[e] & 0xffffu)), acc);
      acc = fma((double)bf16_to_f32((uint16_t)(a[e] >> 16)), (double)bf16_to_f32((uint16_t)(b[e] >> 16)), acc);
    }
  }
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  return acc;
}

// Folds 8 bf16 values, signs cleared, into a running minimum of (bits - 1): one of them was subnormal (exponent 0,
// mantissa not 0) when a half ends below 0x7f.
typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void fold_subnormal(u16x2_t& lowest, u32x4_t mag) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    lowest = __builtin_elementwise_min(lowest, (u16x2_t)(__builtin_bit_cast(u16x2_t, mag[e]) - (u16x2_t){1, 1}));
}
__device__ __forceinline__ bool found_subnormal(u16x2_t lowest) { return lowest.x < 0x7f || lowest.y < 0x7f; }

// Marks an entry whose certificate failed when the exact dot is left to the mask kernel (not a value
// f32_to_bf16 produces: its NaNs are 0x7fc0).
constexpr uint16_t kDeferredScore = 0xffffu;
// The certificate's half-width is kHalfWidth a: twice the worst-case fp32 rounding of a partial of one k-step (16
// products; the partials are added in fp64), which also covers the fp32 error of a itself and the final rounding.
constexpr float kHalfWidth = 0x1p-24f * 32.0f;

// Lane layout (v_mfma_f32_32x32x16_bf16, keys on M, query centroids on N): lane (l32, h) supplies key
// row kt*32 + l32 and query row qt*32 + l32, the 8 values at d = 16s + 8h in k-step s, and receives entry r at key (r/4)*8 + 4h + r%4,
// query l32.  DEFER writes kDeferredScore for the entries that fail the certificate instead of
// recomputing them.
// Bound by the VALU (a tile is 256 float64 operations per lane, the certificate of 16 entries and the subnormal test
// beside 16 MFMAs), so the test is three packed 16-bit operations per two values and the rounding the conversion
// instruction.  The key tile is staged and tested once per block; registers for four waves per SIMD.  40 heads x 100
// queries x 1000 keys: 26.6 us with 12 operations a word and 240 registers (two waves), 14.5 us now; 12 x 100 x 500:
// 9.4 -> 6.2 us.  Five waves per SIMD spill (17.9 us).
template <bool DEFER>
__global__ void __launch_bounds__(kScoreThreads, DEFER ? 4 : 3)
centroid_scores_kernel(const uint16_t* __restrict__ qc, const uint16_t* __restrict__ kc, int qn, int kn,
                       float inv_sqrt_d, uint16_t* __restrict__ out) {
  const int b = blockIdx.y, kt = blockIdx.x;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, h = lane / 32, l32 = lane % 32;
  const int qtiles = (qn + 31) / 32;
  const uint16_t* kbase = kc + (size_t)b * kn * 128;
  const uint16_t* qbase = qc + (size_t)b * qn * 128;
  const u32x4_t absm = {0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu, 0x7fff7fffu};
  // the key tile in LDS, 16-byte chunk c of row l at l * 16 + (c ^ l % 16); its rows holding a subnormal as bits
  __shared__ u32x4_t ktile[32 * 16];
  __shared__ uint32_t kmask_s;
  if (threadIdx.x == 0) kmask_s = 0;
  __syncthreads();
#pragma unroll
  for (int c = threadIdx.x; c < 32 * 16; c += kScoreThreads) {
    const int l = c / 16;
    const u32x4_t w = ((const u32x4_t*)(kbase + (size_t)min(kt * 32 + l, kn - 1) * 128))[c % 16];
    u16x2_t kmin = {0xffff, 0xffff};
    fold_subnormal(kmin, w & absm);
    if (found_subnormal(kmin)) atomicOr(&kmask_s, 1u << l);
    ktile[l * 16 + ((c ^ l) % 16)] = w;
  }
  __syncthreads();
  const uint32_t kmask = kmask_s;
  for (int qt = wave; qt < qtiles; qt += kScoreThreads / kWave) {
    const int i = qt * 32 + l32, irow = min(i, qn - 1);
    u32x4_t qb[8];
    {
      const u32x4_t* src = (const u32x4_t*)(qbase + (size_t)irow * 128) + h;
#pragma unroll
      for (int st = 0; st < 8; ++st) qb[st] = src[2 * st];
    }
    asm volatile("" ::: "memory");  // (the key tile is read again for each query tile, not kept in registers)
    // partials of one k-step each, summed in fp64 as they come
    u16x2_t qmin = {0xffff, 0xffff};
    double sd[16];
    f32x16_t asum = f32x16_t{};
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      const u32x4_t ka = ktile[l32 * 16 + ((2 * st + h) ^ (l32 % 16))];
      const f32x16_t part = mfma32x32x16(as_bf16x8(ka), as_bf16x8(qb[st]), f32x16_t{});
      const u32x4_t qm = qb[st] & absm;
      asum = mfma32x32x16(as_bf16x8(ka & absm), as_bf16x8(qm), asum);
      fold_subnormal(qmin, qm);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sd[r] = st == 0 ? (double)part[r] : sd[r] + (double)part[r];
        asm volatile("" : "+v"(sd[r]));  // (the sums are formed here: deferred to their use, all partials stay live)
      }
    }
    // this lane's query row holds a subnormal (either half)
    const uint32_t qsub = found_subnormal(qmin) ? 1u : 0u;
    const auto qsw = __builtin_amdgcn_permlane32_swap(qsub, qsub, false, false);
    const uint32_t subs = (qsw[0] | qsw[1]) != 0 ? 0xffffffffu : kmask >> (4 * h);
    // entries whose certificate fails: bit r of `redo`
    uint32_t redo = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint32_t packed[2] = {0u, 0u};
      const int j0 = kt * 32 + g * 8 + 4 * h;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = 4 * g + e;
        const float rs = (float)sd[r];
        const float a = asum[r];
        const float err = fmaf(a, kHalfWidth, 0x1p-118f);
        const uint32_t both = cvt_pk_bf16(rs - err, rs + err);  // (a NaN comes with a > 3e38)
        const bool sub = ((subs >> (g * 8 + e)) & 1u) != 0;
        uint32_t tb = cvt_pk_bf16(__uint_as_float(both << 16) * inv_sqrt_d, 0.0f) & 0xffffu;
        if (sub || !(a <= 3.0e38f) || (both & 0xffffu) != both >> 16) {
          redo |= 1u << r;
          if (DEFER) tb = kDeferredScore;
        }
        packed[e / 2] |= tb << (16 * (e % 2));
      }
      if (i < qn) {
        uint16_t* dst = out + ((size_t)b * qn + i) * kn + j0;
        if (j0 + 3 < kn && (kn % 4) == 0)
          *(uint2*)dst = make_uint2(packed[0], packed[1]);
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (j0 + e < kn) dst[e] = (uint16_t)(packed[e / 2] >> (16 * (e % 2)));
      }
    }
    // The failed entries again, exactly in fp64, four at a time by groups of 16 lanes (listed in this wave's
    // LDS slice as lane << 4 | r); their stores come after the first ones, in the same wave.
    if constexpr (!DEFER) {
      if (i >= qn) redo = 0;
      const int nmine = __builtin_popcount(redo);
      int pos = nmine;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int n = __shfl_up(pos, o);
        if (lane >= o) pos += n;
      }
      const int total = __shfl(pos, kWave - 1);
      pos -= nmine;
      __shared__ uint16_t redo_list[kScoreThreads / kWave][kWave * 16];
      uint16_t* list = redo_list[wave];
      while (redo) {
        const int r = __builtin_ctz(redo);
        redo &= redo - 1;
        list[pos++] = (uint16_t)((lane << 4) | r);
      }
      __builtin_amdgcn_wave_barrier();
      for (int base = 0; base < total; base += 4) {
        const int slot = base + lane / 16;
        const bool valid = slot < total;
        int ii = 0, jj = 0;
        if (valid) {
          const int ent = list[slot], ln = ent >> 4, r = ent & 15;
          ii = qt * 32 + (ln % 32);
          jj = kt * 32 + (r / 4) * 8 + 4 * (ln / 32) + (r % 4);
        }
        const bool ok = valid && jj < kn;
        const double dot = group16_dot128(qbase + (size_t)ii * 128, kbase + (size_t)min(jj, kn - 1) * 128, ok);
        if (ok && lane % 16 == 0)
          out[((size_t)b * qn + ii) * kn + jj] = f32_to_bf16(bf16_to_f32(f32_to_bf16((float)dot)) * inv_sqrt_d);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// ------------------------------------------------------------------------------------------ block mask
// The sort keys are the bf16 bits of p (p >= 0, so they order as unsigned integers like the values):
// bin = key >> 7 (the exponent), sub-bin = key & 127 (the mantissa), so a sub-bin holds one value.
// A NaN or +inf score, or only -inf ones, makes the row's sum NaN: there is no order then, and every key is 0, so that
// the row keeps its first clusters up to the cap, all without one (the reference's comparisons with NaN remove nothing).
constexpr int kBins = 128;

// bf16(f32(x * 2^-60)) <= p_st for a fixed-point prefix x (monotone in x)
__device__ __forceinline__ bool prefix_within(long long x, float p_st) {
  return bf16_round_f32((float)((double)x * 0x1p-60)) <= p_st;
}

// floor(p * 2^60) of a bf16 probability key
__device__ __forceinline__ long long fixed60(uint32_t key) {
  const float p = bf16_to_f32((uint16_t)key);
  return p > 0.0f ? (long long)ldexp((double)p, 60) : 0ll;
}

// The softmax's divisor: at least 1e-12; infinite for a NaN sum, which makes every key 0.
__device__ __forceinline__ double softmax_divisor(double sum) { return sum != sum ? INFINITY : fmax(sum, 1e-12); }
// The key of a probability (0 for a NaN).
__device__ __forceinline__ uint32_t probability_key(double p) { return f32_to_bf16(fmaxf((float)p, 0.0f)); }

// Inclusive scans over the 64 lanes of a wave.
__device__ __forceinline__ long long wave_incl_scan_i64(long long v) {
  const int l = threadIdx.x % kWave;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const long long n = __shfl_up(v, o);
    if (l >= o) v += n;
  }
  return v;
}
__device__ __forceinline__ int wave_incl_scan_i32(int v) {
  const int l = threadIdx.x % kWave;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int n = __shfl_up(v, o);
    if (l >= o) v += n;
  }
  return v;
}

// Thread t owns entries j = E t .. E t + E - 1.  The kept set is the first L clusters in the order (p desc,
// j asc); instead of sorting, the kernel finds where that order crosses the top-p threshold and where it
// reaches L from histograms of the keys:
//   level 1: count and fixed-point mass per exponent bin; a scan over the bins (descending) finds the bin in
//            which the prefix first leaves the threshold;
//   level 2: counts per mantissa (one value each, so its mass is count * fx) inside that bin; a scan finds
//            the value, and within it (equal values, index order) the crossing position follows from
//            base + (r + 1) * fx by a binary search;
// the same two levels by count find the key and the rank among equal keys of position L - 1, and a scan of
// the equal-key indicator in index order gives each entry its rank.
template <int KP>
__global__ void __launch_bounds__(kMaskThreads) block_mask_kernel(uint16_t* __restrict__ scores,
                                                                  const uint16_t* __restrict__ qc,
                                                                  const uint16_t* __restrict__ kc,
                                                                  const int32_t* __restrict__ ksz,
                                                                  const int32_t* __restrict__ preserve,
                                                                  const int32_t* __restrict__ cap, int h, int qn,
                                                                  int kn, float inv_sqrt_d, float p_st,
                                                                  uint8_t* __restrict__ map,
                                                                  int32_t* __restrict__ lengths) {
  constexpr int E = KP / kMaskThreads;  // entries per thread
  __shared__ uint32_t cnt1[kBins], ccum1[kBins], cnt2[kBins];
  __shared__ unsigned long long mass1[kBins];
  __shared__ double red_d[kMaskThreads / kWave];
  __shared__ float red_f[kMaskThreads / kWave];
  __shared__ long long red_l[kMaskThreads / kWave];
  __shared__ long long bc[4];  // broadcast slots
  __shared__ uint16_t dlist[KP], tfix[KP];
  __shared__ int ndef;

  const int bh = blockIdx.y, i = blockIdx.x, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int head = bh % h;
  const size_t row = (size_t)bh * qn + i;
  uint8_t* mrow = map + row * kn;
  uint16_t* trow = scores + row * kn;
  const uint16_t* qrow = qc + row * 128;
  const uint16_t* kb = kc + (size_t)bh * kn * 128;

  // Scores.  The entries the score kernel could not certify are listed, computed exactly here (16 at a time,
  // 16 lanes each) and written back; then the row max.
  if (tid == 0) ndef = 0;
  __syncthreads();
  uint16_t tb[E];
  uint32_t deferred = 0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = tid * E + u;
    tb[u] = j < kn ? trow[j] : 0;
    if (j < kn && tb[u] == kDeferredScore) {
      deferred |= 1u << u;
      dlist[atomicAdd(&ndef, 1)] = (uint16_t)j;
    }
  }
  __syncthreads();
  const int nd = ndef;
  if (nd > 0) {
    for (int base = 0; base < nd; base += kMaskThreads / 16) {
      const int slot = base + tid / 16;
      const bool valid = slot < nd;
      const int j = valid ? dlist[slot] : 0;
      const double dot = group16_dot128(qrow, kb + (size_t)j * 128, valid);
      if (valid && tid % 16 == 0) {
        const uint16_t bits = f32_to_bf16(bf16_to_f32(f32_to_bf16((float)dot)) * inv_sqrt_d);
        tfix[j] = bits;
        trow[j] = bits;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (deferred & (1u << u)) tb[u] = tfix[tid * E + u];
  }
  float tv[E];
  float lmax = -INFINITY;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    tv[u] = tid * E + u < kn ? bf16_to_f32(tb[u]) : -INFINITY;
    lmax = fmaxf(lmax, tv[u]);
  }
  const float m = block_max_f32<kMaskThreads>(lmax, red_f);

  // Weighted softmax in fp64 -> bf16 probability keys.
  const int32_t* wrow = ksz + (size_t)bh * kn;
  double we[E];
  double lsum = 0.0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = tid * E + u;
    we[u] = 0.0;
    if (j < kn) {
      we[u] = (double)wrow[j] * exp((double)tv[u] - (double)m);
      lsum += we[u];
    }
  }
  const double den = softmax_divisor(block_sum_f64<kMaskThreads>(lsum, red_d));
  uint32_t key[E];
#pragma unroll
  for (int u = 0; u < E; ++u) key[u] = probability_key(we[u] / den);

  // Level 1: counts and masses per exponent bin.
  if (tid < kBins) {
    cnt1[tid] = 0;
    mass1[tid] = 0;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < E; ++u) {
    if (tid * E + u < kn) {
      atomicAdd(&cnt1[(key[u] >> 7) & (kBins - 1)], 1u);
      atomicAdd(&mass1[(key[u] >> 7) & (kBins - 1)], (unsigned long long)fixed60(key[u]));
    }
  }
  __syncthreads();
  // Wave 0 scans the bins in descending order (lane l: positions 2l, 2l + 1 = bins 127 - 2l, 126 - 2l) and
  // finds the first bin whose inclusive prefix leaves the threshold.
  if (wave == 0) {
    const int b0 = kBins - 1 - 2 * lane, b1 = b0 - 1;
    const int c0 = (int)cnt1[b0], c1 = (int)cnt1[b1];
    const long long m0 = (long long)mass1[b0], m1 = (long long)mass1[b1];
    const int ci = wave_incl_scan_i32(c0 + c1);
    const long long mi = wave_incl_scan_i64(m0 + m1);
    const int ce = ci - c0 - c1;
    const long long me = mi - m0 - m1;
    ccum1[2 * lane] = (uint32_t)(ce + c0);
    ccum1[2 * lane + 1] = (uint32_t)ci;
    const bool out0 = !prefix_within(me + m0, p_st), out1 = !prefix_within(mi, p_st);
    const uint64_t any = __ballot(out0 || out1);
    if (any == 0) {
      if (lane == 0) bc[0] = -1;
    } else if (lane == __builtin_ctzll(any)) {
      const bool first = out0;
      bc[0] = first ? 2 * lane : 2 * lane + 1;   // position of the bin
      bc[1] = first ? me : me + m0;              // mass before it
      bc[2] = first ? ce : ce + c0;              // entries before it
    }
  }
  __syncthreads();
  const int dstar = (int)bc[0];
  long long T = kn;  // leading positions whose prefix stays within the threshold
  if (dstar >= 0) {
    const int bstar = kBins - 1 - dstar;
    // Level 2 inside that bin: counts per mantissa.
    if (tid < kBins) cnt2[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (tid * E + u < kn && (int)((key[u] >> 7) & (kBins - 1)) == bstar) atomicAdd(&cnt2[key[u] & 127], 1u);
    __syncthreads();
    if (wave == 0) {
      const long long base_m = bc[1], base_c = bc[2];
      const int s0 = kBins - 1 - 2 * lane, s1 = s0 - 1;
      const uint32_t k0 = ((uint32_t)bstar << 7) | (uint32_t)s0, k1 = ((uint32_t)bstar << 7) | (uint32_t)s1;
      const int c0 = (int)cnt2[s0], c1 = (int)cnt2[s1];
      const long long f0 = fixed60(k0), f1 = fixed60(k1);
      const long long m0 = (long long)c0 * f0, m1 = (long long)c1 * f1;
      const int ci = wave_incl_scan_i32(c0 + c1);
      const long long mi = wave_incl_scan_i64(m0 + m1);
      const int ce = ci - c0 - c1;
      const long long me = mi - m0 - m1;
      const bool out0 = !prefix_within(base_m + me + m0, p_st), out1 = !prefix_within(base_m + mi, p_st);
      const uint64_t any = __ballot(out0 || out1);
      if (any != 0 && lane == __builtin_ctzll(any)) {
        const bool first = out0;
        const long long mb = base_m + (first ? me : me + m0);
        const long long fx = first ? f0 : f1;
        const int cnt = first ? c0 : c1;
        // smallest r in [0, cnt) with the prefix mb + (r + 1) fx outside the threshold
        int lo = 0, hi = cnt - 1;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (!prefix_within(mb + (long long)(mid + 1) * fx, p_st))
            hi = mid;
          else
            lo = mid + 1;
        }
        bc[3] = base_c + (first ? ce : ce + c0) + lo;
      }
    }
    __syncthreads();
    T = bc[3];
  }
  int len = 1 + (int)min(T, (long long)(kn - 1));
  len = max(len, (int)preserve[head]);
  if (cap[head] > 0) len = min(len, (int)cap[head]);
  len = min(len, kn);

  // The key and the rank among equal keys of position len - 1.
  uint32_t key_l = 0;
  int rank_l = 0;
  if (len < kn) {
    __syncthreads();  // bc and cnt2 are read above
    if (wave == 0) {
      const bool r0 = (int)ccum1[2 * lane] >= len, r1 = (int)ccum1[2 * lane + 1] >= len;
      const uint64_t any = __ballot(r0 || r1);
      if (lane == __builtin_ctzll(any)) {
        const int d = r0 ? 2 * lane : 2 * lane + 1;
        bc[0] = d;
        bc[1] = d > 0 ? (long long)ccum1[d - 1] : 0;
      }
    }
    __syncthreads();
    const int dl = (int)bc[0];
    const int bl = kBins - 1 - dl;
    if (dl != dstar) {  // block-uniform: rebuild the level-2 counts for this bin
      if (tid < kBins) cnt2[tid] = 0;
      __syncthreads();
#pragma unroll
      for (int u = 0; u < E; ++u)
        if (tid * E + u < kn && (int)((key[u] >> 7) & (kBins - 1)) == bl) atomicAdd(&cnt2[key[u] & 127], 1u);
      __syncthreads();
    }
    if (wave == 0) {
      const long long base_c = bc[1];
      const int s0 = kBins - 1 - 2 * lane, s1 = s0 - 1;
      const int c0 = (int)cnt2[s0], c1 = (int)cnt2[s1];
      const int ci = wave_incl_scan_i32(c0 + c1);
      const int ce = ci - c0 - c1;
      const bool r0 = base_c + ce + c0 >= len, r1 = base_c + ci >= len;
      const uint64_t any = __ballot(r0 || r1);
      if (lane == __builtin_ctzll(any)) {
        const bool first = r0;
        bc[2] = ((long long)bl << 7) | (first ? s0 : s1);
        bc[3] = len - 1 - (base_c + (first ? ce : ce + c0));
      }
    }
    __syncthreads();
    key_l = (uint32_t)bc[2];
    rank_l = (int)bc[3];
  }

  // Rank of each entry among the entries with key key_l, in index order; kept = ahead of position len - 1.
  int eq = 0;
#pragma unroll
  for (int u = 0; u < E; ++u) eq += (tid * E + u < kn && key[u] == key_l) ? 1 : 0;
  long long tot;
  int rank = (int)block_exclusive_scan_i64<kMaskThreads>(eq, red_l, &tot);
  uint32_t word = 0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    bool keep = true;
    if (len < kn) {
      keep = key[u] > key_l;
      if (key[u] == key_l) keep = rank++ <= rank_l;
    }
    if (tid * E + u < kn && keep) word |= 1u << (8 * (u % 4));
    if (u % 4 == 3 || u == E - 1) {
      const int j0 = tid * E + (u / 4) * 4;
      if ((kn & 3) == 0 && E >= 4) {
        if (j0 < kn) *(uint32_t*)(mrow + j0) = word;
      } else {
        for (int e = 0; e <= u % 4; ++e)
          if (j0 + e < kn) mrow[j0 + e] = (uint8_t)(word >> (8 * e));
      }
      word = 0;
    }
  }
  if (tid == 0 && lengths) lengths[row] = len;
}

// The same row by one wave, E entries per lane (entry u * 64 + lane), without block barriers: a block of 256 threads per
// row spent most of its time at some 17 of them and in wave 0's scans.  Differences from the block's kernel, none in a
// result: the exponential comes from a table (within 0.54 units of the last place of float64, the library's within 0.88)
// and the quotient from one reciprocal with a correction step (the residual is exact and the reciprocal within 2^-53 of
// itself, so it is within 0.5 + 2^-51 units; a division takes 1.8 us more at 4800 rows of 1000), and a bin's count and
// mass share one 32-bit LDS counter: a key of exponent e holds (128 + mantissa) 2^(e - 74) of the 2^60, so a bin's mass is a sum of
// integers below 2^18 times a power of two (below e = 74 each entry is rounded down on its own, as the mass demands).
// The score and size loads are issued together on clamped indexes (a guarded load waits for the one before it: 11.7k of
// a row's 46k cycles, then 1.7k).  What is left is the exact dots of the deferred scores (a third of a row: 25 of 1000
// entries) and the softmax.  Measured on 4000 rows of 1000: 33 us by blocks, 24.9 us by waves; eight gathered rows in
// flight per group instead of four: 25.6 us (134 registers, fewer waves).
template <int E>
__global__ void __launch_bounds__(kMaskThreads) block_mask_wave_kernel(uint16_t* __restrict__ scores,
                                                                       const uint16_t* __restrict__ qc,
                                                                       const uint16_t* __restrict__ kc,
                                                                       const int32_t* __restrict__ ksz,
                                                                       const int32_t* __restrict__ preserve,
                                                                       const int32_t* __restrict__ cap, int h, int qn,
                                                                       int kn, long long rows, float inv_sqrt_d,
                                                                       float p_st, uint8_t* __restrict__ map,
                                                                       int32_t* __restrict__ lengths) {
  constexpr int kW = kMaskThreads / kWave;
  __shared__ double2 tab[64];
  __shared__ uint32_t hist_s[kW][2][kBins];
  __shared__ uint16_t dlist_s[kW][E * kWave], tfix_s[kW][E * kWave];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  if (tid < 64) tab[tid] = kExp2Table[tid];
  __syncthreads();
  const long long row = (long long)blockIdx.x * kW + wave;
  if (row >= rows) return;
  const int bh = (int)(row / qn), head = bh % h;
  uint32_t* h1 = hist_s[wave][0];
  uint32_t* h2 = hist_s[wave][1];
  uint16_t* dlist = dlist_s[wave];
  uint16_t* tfix = tfix_s[wave];
  uint8_t* mrow = map + row * kn;
  uint16_t* trow = scores + row * kn;
  const uint16_t* kb = kc + (size_t)bh * kn * 128;
  const int32_t* wrow = ksz + (size_t)bh * kn;

  // Scores, and the entries left to be computed exactly: 16 at a time, four per group of 16 lanes.
  uint16_t tb[E];
  int wt[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = min(u * kWave + lane, kn - 1);  // (conditional loads would each wait for the one before)
    tb[u] = trow[j];
    wt[u] = wrow[j];
  }
  int nd = 0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = u * kWave + lane;
    const bool def = j < kn && tb[u] == kDeferredScore;
    const uint64_t b = __ballot(def);
    if (def) dlist[nd + (int)__popcll(b & ((1ull << lane) - 1ull))] = (uint16_t)j;
    nd += (int)__popcll(b);
  }
  if (nd > 0) {
    const u32x4_t qw = ((const u32x4_t*)(qc + row * 128))[lane % 16];
    constexpr int kR = 4;  // rows in flight per group
    for (int base = 0; base < nd; base += 4 * kR) {
      int jj[kR];
      u32x4_t kw[kR];
#pragma unroll
      for (int t = 0; t < kR; ++t) {
        const int slot = base + 4 * t + lane / 16;
        jj[t] = slot < nd ? dlist[slot] : -1;
        kw[t] = ((const u32x4_t*)(kb + (size_t)max(jj[t], 0) * 128))[lane % 16];
      }
#pragma unroll
      for (int t = 0; t < kR; ++t) {
        double acc = 0.0;  // the sum of group16_dot128
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc = fma((double)bf16_to_f32((uint16_t)(qw[e] & 0xffffu)), (double)bf16_to_f32((uint16_t)(kw[t][e] & 0xffffu)), acc);
          acc = fma((double)bf16_to_f32((uint16_t)(qw[e] >> 16)), (double)bf16_to_f32((uint16_t)(kw[t][e] >> 16)), acc);
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
        if (jj[t] >= 0 && lane % 16 == 0) {
          const uint16_t bits = f32_to_bf16(bf16_to_f32(f32_to_bf16((float)acc)) * inv_sqrt_d);
          tfix[jj[t]] = bits;
          trow[jj[t]] = bits;
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (u * kWave + lane < kn && tb[u] == kDeferredScore) tb[u] = tfix[u * kWave + lane];
  }
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < E; ++u) m = fmaxf(m, u * kWave + lane < kn ? bf16_to_f32(tb[u]) : -INFINITY);
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));

  // Weighted softmax in fp64 -> bf16 probability keys.
  double we[E];
  double lsum = 0.0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    we[u] = 0.0;
    if (u * kWave + lane < kn) {
      we[u] = (double)wt[u] * exp_tab(tab, (double)bf16_to_f32(tb[u]) - (double)m);
      lsum += we[u];
    }
  }
  const double den = softmax_divisor(lane_f64(wave_scan_f64(lsum), kWave - 1));
  const double rden = 1.0 / den;
  uint32_t key[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const double q = we[u] * rden;
    key[u] = probability_key(fma(fma(-q, den, we[u]), rden, q));
  }

  // Level 1: per exponent bin count << 20 | sum of (128 + mantissa).
  h1[lane] = 0;
  h1[lane + kWave] = 0;
  h2[lane] = 0;
  h2[lane + kWave] = 0;
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int u = 0; u < E; ++u) {
    if (u * kWave + lane < kn) {
      const int e = (int)(key[u] >> 7);
      uint32_t c = 128u + (key[u] & 127u);
      if (e < 74) c = e > 66 ? c >> (74 - e) : 0u;
      atomicAdd(&h1[e & (kBins - 1)], (1u << 20) | c);
    }
  }
  __builtin_amdgcn_wave_barrier();
  // Lane l: positions 2l, 2l + 1 = bins 127 - 2l, 126 - 2l; the first bin whose prefix leaves the threshold.
  const int b0 = kBins - 1 - 2 * lane, b1 = b0 - 1;
  const uint32_t w0 = h1[b0], w1 = h1[b1];
  const int c0 = (int)(w0 >> 20), c1 = (int)(w1 >> 20);
  const long long m0 = (long long)(w0 & 0xfffffu) << max(b0 - 74, 0), m1 = (long long)(w1 & 0xfffffu) << max(b1 - 74, 0);
  const int ci = wave_scan_i32(c0 + c1), ce = ci - c0 - c1;
  const long long mi = wave_scan_i64(m0 + m1), me = mi - m0 - m1;
  // Counts per mantissa of one bin (its values, one each) into h2.
  auto level2 = [&](int bin) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < E; ++u)
      if (u * kWave + lane < kn && (int)((key[u] >> 7) & (kBins - 1)) == bin) atomicAdd(&h2[key[u] & 127u], 1u);
    __builtin_amdgcn_wave_barrier();
  };
  long long T = kn;  // leading positions whose prefix stays within the threshold
  int dstar = -1;
  {
    const bool out0 = !prefix_within(me + m0, p_st), out1 = !prefix_within(mi, p_st);
    const uint64_t any = __ballot(out0 || out1);
    if (any != 0) {
      const int l = __builtin_ctzll(any);
      const bool first = (__ballot(out0) >> l) & 1;
      dstar = first ? 2 * l : 2 * l + 1;
      const long long base_m = lane_i64(first ? me : me + m0, l);
      const int base_c = __builtin_amdgcn_readlane(first ? ce : ce + c0, l);
      const int bstar = kBins - 1 - dstar;
      level2(bstar);
      const uint32_t k0 = ((uint32_t)bstar << 7) | (uint32_t)b0, k1 = ((uint32_t)bstar << 7) | (uint32_t)b1;
      const int d0 = (int)h2[b0], d1 = (int)h2[b1];
      const long long f0 = fixed60(k0), f1 = fixed60(k1);
      const long long n0 = (long long)d0 * f0, n1 = (long long)d1 * f1;
      const int di = wave_scan_i32(d0 + d1), de = di - d0 - d1;
      const long long ni = wave_scan_i64(n0 + n1), ne = ni - n0 - n1;
      const bool o0 = !prefix_within(base_m + ne + n0, p_st), o1 = !prefix_within(base_m + ni, p_st);
      const uint64_t any2 = __ballot(o0 || o1);
      const int l2 = __builtin_ctzll(any2 | (1ull << 63));
      const bool f2 = (__ballot(o0) >> l2) & 1;
      const long long mb = base_m + lane_i64(f2 ? ne : ne + n0, l2);
      const long long fx = lane_i64(f2 ? f0 : f1, l2);
      // smallest r in [0, cnt) with the prefix mb + (r + 1) fx outside the threshold
      int lo = 0, hi = __builtin_amdgcn_readlane(f2 ? d0 : d1, l2) - 1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (!prefix_within(mb + (long long)(mid + 1) * fx, p_st))
          hi = mid;
        else
          lo = mid + 1;
      }
      T = base_c + __builtin_amdgcn_readlane(f2 ? de : de + d0, l2) + lo;
    }
  }
  int len = 1 + (int)min(T, (long long)(kn - 1));
  len = max(len, (int)preserve[head]);
  if (cap[head] > 0) len = min(len, (int)cap[head]);
  len = min(len, kn);

  // The key and the rank among equal keys of position len - 1.
  uint32_t key_l = 0;
  int rank_l = 0;
  if (len < kn) {
    const bool r0 = ce + c0 >= len, r1 = ci >= len;
    const int l = __builtin_ctzll(__ballot(r0 || r1));
    const bool first = (__ballot(r0) >> l) & 1;
    const int dl = first ? 2 * l : 2 * l + 1;
    const int base_c = __builtin_amdgcn_readlane(first ? ce : ce + c0, l);
    const int bl = kBins - 1 - dl;
    if (dl != dstar) {
      h2[lane] = 0;
      h2[lane + kWave] = 0;
      __builtin_amdgcn_wave_barrier();
      level2(bl);
    }
    const int d0 = (int)h2[b0], d1 = (int)h2[b1];
    const int di = wave_scan_i32(d0 + d1), de = di - d0 - d1;
    const bool q0 = base_c + de + d0 >= len, q1 = base_c + di >= len;
    const int l2 = __builtin_ctzll(__ballot(q0 || q1) | (1ull << 63));
    const bool f2 = (__ballot(q0) >> l2) & 1;
    key_l = ((uint32_t)bl << 7) | (uint32_t)(kBins - 1 - 2 * l2 - (f2 ? 0 : 1));
    rank_l = len - 1 - (base_c + __builtin_amdgcn_readlane(f2 ? de : de + d0, l2));
  }

  // Kept: ahead of position len - 1 in (key desc, index asc).
  int run = 0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = u * kWave + lane;
    const uint64_t eq = __ballot(j < kn && key[u] == key_l);
    const int rank = run + (int)__popcll(eq & ((1ull << lane) - 1ull));
    run += (int)__popcll(eq);
    const bool keep = len >= kn || key[u] > key_l || (key[u] == key_l && rank <= rank_l);
    if (j < kn) mrow[j] = keep ? 1 : 0;
  }
  if (lane == 0 && lengths) lengths[row] = len;
}

// All-true map rows (top_p >= 1, svoo/co_clustering.py:575-576).
__global__ void __launch_bounds__(kMaskThreads) full_mask_kernel(uint8_t* __restrict__ map, int qn, int kn,
                                                                 int32_t* __restrict__ lengths) {
  const size_t row = (size_t)blockIdx.y * qn + blockIdx.x;
  uint8_t* mrow = map + row * kn;
  for (int j = threadIdx.x; j < kn; j += kMaskThreads) mrow[j] = 1;
  if (threadIdx.x == 0 && lengths) lengths[row] = kn;
}

// Standalone weighted softmax (one block per row).
template <int KP>
__global__ void __launch_bounds__(kMaskThreads) weighted_softmax_kernel(const uint16_t* __restrict__ scores,
                                                                        const float* __restrict__ weights,
                                                                        long long wstride, uint16_t* __restrict__ out,
                                                                        int cols) {
  constexpr int E = KP / kMaskThreads;
  __shared__ double red_d[kMaskThreads / kWave];
  __shared__ float red_f[kMaskThreads / kWave];
  const long long r = blockIdx.x;
  const uint16_t* srow = scores + r * cols;
  const float* wrow = weights + r * wstride;
  float lmax = -INFINITY;
  float sv[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = threadIdx.x + u * kMaskThreads;
    sv[u] = j < cols ? bf16_to_f32(srow[j]) : -INFINITY;
    lmax = fmaxf(lmax, sv[u]);
  }
  const float m = block_max_f32<kMaskThreads>(lmax, red_f);
  double we[E];
  double lsum = 0.0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = threadIdx.x + u * kMaskThreads;
    we[u] = j < cols ? (double)wrow[j] * exp((double)sv[u] - (double)m) : 0.0;
    lsum += we[u];
  }
  const double den = fmax(block_sum_f64<kMaskThreads>(lsum, red_d), 1e-12);
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int j = threadIdx.x + u * kMaskThreads;
    if (j < cols) out[r * cols + j] = f32_to_bf16((float)(we[u] / den));
  }
}

}  // namespace svoo

using namespace svoo;

extern "C" int svoo_centroid_scores(const uint16_t* qc, const uint16_t* kc, int bh, int qn, int kn, int d,
                                    uint16_t* scores, void* stream) {
  SVOO_REQUIRE(qc && kc && scores, SVOO_ERR_INVALID_ARG, "svoo_centroid_scores: null pointer");
  SVOO_REQUIRE(bh > 0 && qn > 0 && kn > 0, SVOO_ERR_INVALID_ARG, "svoo_centroid_scores: bad dims");
  SVOO_REQUIRE_HEAD_DIM(d, "svoo_centroid_scores");
  SVOO_REQUIRE(bh <= 65535 && kn <= (1 << 26), SVOO_ERR_UNSUPPORTED, "svoo_centroid_scores: grid too large");
  const float inv = 1.0f / (float)sqrt((double)d);
  hipLaunchKernelGGL(centroid_scores_kernel<false>, dim3((kn + 31) / 32, bh), dim3(kScoreThreads), 0, (hipStream_t)stream,
                     qc, kc, qn, kn, inv, scores);
  return check_launch("svoo_centroid_scores");
}

extern "C" int svoo_block_mask(const uint16_t* qc, const uint16_t* kc, const int32_t* k_sizes,
                               const int32_t* preserve, const int32_t* cap, int b, int h, int qn, int kn, int d,
                               float p_storage, int full, uint8_t* map, int32_t* lengths, uint16_t* scores,
                               void* stream) {
  SVOO_REQUIRE(map && (full || (qc && kc && k_sizes && preserve && cap && scores)), SVOO_ERR_INVALID_ARG,
               "svoo_block_mask: null pointer");
  SVOO_REQUIRE(b > 0 && h > 0 && qn > 0 && kn > 0, SVOO_ERR_INVALID_ARG, "svoo_block_mask: bad dims");
  SVOO_REQUIRE_HEAD_DIM(d, "svoo_block_mask");
  SVOO_REQUIRE(kn <= 4096, SVOO_ERR_UNSUPPORTED, "svoo_block_mask: Kc=%d exceeds 4096", kn);
  SVOO_REQUIRE(qn <= 65535 && (long long)b * h <= 65535, SVOO_ERR_UNSUPPORTED, "svoo_block_mask: grid too large");
  dim3 grid(qn, b * h);
  hipStream_t s = (hipStream_t)stream;
  if (full) {
    hipLaunchKernelGGL(full_mask_kernel, grid, dim3(kMaskThreads), 0, s, map, qn, kn, lengths);
    return check_launch("svoo_block_mask");
  }
  const float inv = 1.0f / (float)sqrt((double)d);
  // scores with the uncertified entries deferred to the mask kernel, which computes them exactly
  hipLaunchKernelGGL(centroid_scores_kernel<true>, dim3((kn + 31) / 32, b * h), dim3(kScoreThreads), 0, s, qc, kc, qn, kn,
                     inv, scores);
  if (int rc = check_launch("svoo_block_mask (scores)")) return rc;
#define SVOO_MASK_LAUNCH(KP)                                                                                     \
  hipLaunchKernelGGL(block_mask_kernel<KP>, grid, dim3(kMaskThreads), 0, s, scores, qc, kc, k_sizes, preserve, cap, \
                     h, qn, kn, inv, p_storage, map, lengths)
#define SVOO_MASK_WAVES(E)                                                                                       \
  hipLaunchKernelGGL(block_mask_wave_kernel<E>, wgrid, dim3(kMaskThreads), 0, s, scores, qc, kc, k_sizes, preserve, cap, \
                     h, qn, kn, rows, inv, p_storage, map, lengths)
  // A row per wave or per block. A wave's row has no barriers and leaves room for many rows on a CU, a block's row is
  // done sooner; the wave is ahead once there are some eight rows per CU, and always where a lane holds four entries.
  // Block -> wave, Gaussian centroids, d 128: 200 clusters 6.4 -> 6.4 us at 200 rows, 43.6 -> 20.9 at 10240;
  // 500 clusters 8.8 -> 9.5 at 600 rows, 11.0 -> 10.7 at 1200, 17.6 -> 12.9 at 2400, 55.4 -> 30.3 at 10240;
  // 1000 clusters 14.9 -> 16.5 at 1200 rows, 24.4 -> 20.3 at 2400, 77.6 -> 49.4 at 10240.
  const long long rows = (long long)b * h * qn;
  const bool waves = rows >= kWaveRows;
  const dim3 wgrid((unsigned)((rows + kMaskThreads / kWave - 1) / (kMaskThreads / kWave)));
  if (kn <= 256)
    SVOO_MASK_WAVES(4);
  else if (kn <= 512 && waves)
    SVOO_MASK_WAVES(8);
  else if (kn <= 512)
    SVOO_MASK_LAUNCH(512);
  else if (kn <= 1024 && waves)
    SVOO_MASK_WAVES(16);
  else if (kn <= 1024)
    SVOO_MASK_LAUNCH(1024);
  else if (kn <= 2048)
    SVOO_MASK_LAUNCH(2048);
  else
    SVOO_MASK_LAUNCH(4096);
#undef SVOO_MASK_LAUNCH
#undef SVOO_MASK_WAVES
  return check_launch("svoo_block_mask");
}

extern "C" int svoo_weighted_softmax(const uint16_t* scores, const float* weights, long long weight_row_stride,
                                     uint16_t* out, long long rows, int cols, void* stream) {
  SVOO_REQUIRE(scores && weights && out, SVOO_ERR_INVALID_ARG, "svoo_weighted_softmax: null pointer");
  SVOO_REQUIRE(rows > 0 && cols > 0 && rows <= 2147483647ll, SVOO_ERR_INVALID_ARG, "svoo_weighted_softmax: bad dims");
  SVOO_REQUIRE(cols <= 4096, SVOO_ERR_UNSUPPORTED, "svoo_weighted_softmax: cols=%d exceeds 4096", cols);
  hipStream_t s = (hipStream_t)stream;
  dim3 grid((unsigned)rows);
#define SVOO_WS_LAUNCH(KP) \
  hipLaunchKernelGGL(weighted_softmax_kernel<KP>, grid, dim3(kMaskThreads), 0, s, scores, weights, weight_row_stride, out, cols)
  if (cols <= 256)
    SVOO_WS_LAUNCH(256);
  else if (cols <= 1024)
    SVOO_WS_LAUNCH(1024);
  else
    SVOO_WS_LAUNCH(4096);
#undef SVOO_WS_LAUNCH
  return check_launch("svoo_weighted_softmax");
}
