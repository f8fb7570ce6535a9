// Projected rows to attention heads: the norm of Q and K, rotary embedding and the [S, H*D] -> [H, S, D] transposition
// of Q, K and V in one pass over each tensor.
//
// What bounds it: memory (each element read and written once).  One wave holds one token's row, 8 elements per lane and
// 512-element chunk, so a norm over the whole row is one wave reduction and a norm per head one over d / 8 lanes; a row
// leaves as d-element pieces, one per head, whole cache lines each.  A lane's place within the head is the same in
// every chunk (512 is a multiple of d), so its rotary angles are loaded once per row.
// Measured: 32760 tokens of 12 heads (604 MB read and written), norm over the row: 0.12 ms (4.95 TB/s) against 1.13 ms
// in 21 launches of the tensor operations; 32656 tokens of 24 heads (1.2 GB), norm per head: 0.23 ms against 4.3 ms.
#include "svoo_common.h"

namespace svoo {

constexpr int kHeadsThreads = 256;

struct HeadsArgs {
  const uint16_t* src[3];      // Q, K, V rows
  uint16_t* dst[3];            // [H][out_rows][d]
  long long stride[3];         // elements between source rows
  const uint16_t* weight[2];   // norm weights of Q and K (bf16) or null
  float eps[2];
  const float* cosp;           // [rope_rows][d] or null
  const float* sinp;
  int rows, heads, d, out_rows, out_row0, norm, rope_rows, form;
};

// y0 = x0 c0 - x1 s0, y1 = x1 c1 + x0 s1 with every product rounded to fp32, as the tensor operations round it: the
// empty asm keeps the compiler from fusing them into the sums.
__device__ __forceinline__ void rotate(float& x0, float& x1, float c0, float s0, float c1, float s1) {
  float a = x0 * c0, b = x1 * s0, c = x1 * c1, e = x0 * s1;
  __asm__("" : "+v"(a), "+v"(b), "+v"(c), "+v"(e));
  x0 = a - b;
  x1 = c + e;
}

template <int NC>
__global__ void __launch_bounds__(kHeadsThreads) qkv_heads_kernel(HeadsArgs a) {
  const int which = blockIdx.y;
  const int lane = threadIdx.x % kWave;
  const int row = blockIdx.x * (kHeadsThreads / kWave) + threadIdx.x / kWave;
  if (row >= a.rows) return;
  const int dim = a.heads * a.d;
  const uint16_t* src = a.src[which] + (long long)row * a.stride[which];
  u32x4_t x[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
    if (c * 512 + lane * 8 < dim) x[c] = *(const u32x4_t*)(src + c * 512 + lane * 8);
  const int d0 = (lane * 8) & (a.d - 1);  // d is 64 or 128
  if (which < 2) {
    const bool rope = a.cosp != nullptr && row < a.rope_rows;
    float cs[8], sn[8];
    if (rope) {
      const f32x4_t* cp = (const f32x4_t*)(a.cosp + (size_t)row * a.d + d0);
      const f32x4_t* sp = (const f32x4_t*)(a.sinp + (size_t)row * a.d + d0);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        cs[e] = cp[e / 4][e % 4];
        sn[e] = sp[e / 4][e % 4];
      }
      if (a.form == 0) {  // both elements of a pair take the even cosine and the odd sine
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          cs[e + 1] = cs[e];
          sn[e] = sn[e + 1];
        }
      }
    }
    float total = 0.0f;  // norm over the row
    if (a.norm == 1) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (c * 512 + lane * 8 < dim) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float u = bf16_to_f32((uint16_t)(x[c][e] & 0xffffu)), w = bf16_to_f32((uint16_t)(x[c][e] >> 16));
            total = fmaf(u, u, total);
            total = fmaf(w, w, total);
          }
        }
      for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o);
    }
    const float rstd_row = rsqrtf(total / (float)dim + a.eps[which]);
    const uint16_t* wt = a.weight[which];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (c * 512 >= dim) break;  // wave-uniform: the shuffles below need every lane of a head
      const bool in = c * 512 + lane * 8 < dim;
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[2 * e] = in ? bf16_to_f32((uint16_t)(x[c][e] & 0xffffu)) : 0.0f;
        v[2 * e + 1] = in ? bf16_to_f32((uint16_t)(x[c][e] >> 16)) : 0.0f;
      }
      if (a.norm != 0) {
        float rstd = rstd_row;
        if (a.norm == 2) {
          float sq = 0.0f;
#pragma unroll
          for (int e = 0; e < 8; ++e) sq = fmaf(v[e], v[e], sq);
          for (int o = 1; o < a.d / 8; o <<= 1) sq += __shfl_xor(sq, o);
          rstd = rsqrtf(sq / (float)a.d + a.eps[which]);
        }
        u32x4_t w4 = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // ones
        if (wt != nullptr && in) w4 = *(const u32x4_t*)(wt + (a.norm == 2 ? d0 : c * 512 + lane * 8));
        // the norm's result is a bf16 tensor, rounded before the rotation
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[2 * e] = bf16_round_f32(bf16_to_f32((uint16_t)(w4[e] & 0xffffu)) * (rstd * v[2 * e]));
          v[2 * e + 1] = bf16_round_f32(bf16_to_f32((uint16_t)(w4[e] >> 16)) * (rstd * v[2 * e + 1]));
        }
      }
      if (rope) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) rotate(v[e], v[e + 1], cs[e], sn[e], cs[e + 1], sn[e + 1]);
      }
      if (a.norm != 0 || rope) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c][e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
      }
    }
  }
  uint16_t* dst = a.dst[which] + ((size_t)a.out_row0 + row) * a.d + d0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int col = c * 512 + lane * 8;
    if (col < dim) *(u32x4_t*)(dst + (size_t)(col / a.d) * a.out_rows * a.d) = x[c];
  }
}

}  // namespace svoo

using namespace svoo;

extern "C" int svoo_qkv_heads(const uint16_t* q, const uint16_t* k, const uint16_t* v, long long q_stride,
                              long long k_stride, long long v_stride, uint16_t* q_out, uint16_t* k_out,
                              uint16_t* v_out, int rows, int heads, int d, int out_rows, int out_row0, int norm,
                              const uint16_t* q_weight, const uint16_t* k_weight, float q_eps, float k_eps,
                              const float* cos_table, const float* sin_table, int rope_rows, int rope_form,
                              void* stream) {
  static const char* name = "svoo_qkv_heads";
  SVOO_REQUIRE(q && k && v && q_out && k_out && v_out, SVOO_ERR_INVALID_ARG, "%s: null pointer", name);
  SVOO_REQUIRE(d == 64 || d == 128, SVOO_ERR_UNSUPPORTED, "%s: D=%d (64 or 128)", name, d);
  SVOO_REQUIRE(heads > 0 && (long long)heads * d <= 8192, SVOO_ERR_UNSUPPORTED, "%s: H=%d x D=%d above 8192", name,
               heads, d);
  SVOO_REQUIRE(rows > 0 && out_row0 >= 0 && (long long)out_row0 + rows <= out_rows, SVOO_ERR_INVALID_ARG,
               "%s: rows=%d at %d of %d", name, rows, out_row0, out_rows);
  SVOO_REQUIRE(norm >= 0 && norm <= 2 && (rope_form == 0 || rope_form == 1), SVOO_ERR_INVALID_ARG,
               "%s: norm=%d rope_form=%d", name, norm, rope_form);
  SVOO_REQUIRE((cos_table == nullptr) == (sin_table == nullptr) && rope_rows >= 0 && rope_rows <= rows,
               SVOO_ERR_INVALID_ARG, "%s: rope tables of %d rows", name, rope_rows);
  const uintptr_t bits = (uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)q_out | (uintptr_t)k_out |
                         (uintptr_t)v_out | (uintptr_t)q_weight | (uintptr_t)k_weight | (uintptr_t)cos_table |
                         (uintptr_t)sin_table;
  SVOO_REQUIRE(bits % 16 == 0 && (q_stride | k_stride | v_stride) % 8 == 0, SVOO_ERR_INVALID_ARG,
               "%s: rows must start at 16-byte addresses", name);
  const HeadsArgs a = {{q, k, v},         {q_out, k_out, v_out}, {q_stride, k_stride, v_stride},
                       {q_weight, k_weight}, {q_eps, k_eps},     cos_table,
                       sin_table,         rows,                  heads,
                       d,                 out_rows,              out_row0,
                       norm,              rope_rows,             rope_form};
  const dim3 grid((rows + kHeadsThreads / kWave - 1) / (kHeadsThreads / kWave), 3), block(kHeadsThreads);
  hipStream_t s = (hipStream_t)stream;
  // the row in registers: 4 per 512-element chunk; widths of the Wan (1536, 5120) and HunyuanVideo (3072) models
  const int dim = heads * d;
  if (dim <= 3 * 512) hipLaunchKernelGGL(qkv_heads_kernel<3>, grid, block, 0, s, a);
  else if (dim <= 6 * 512) hipLaunchKernelGGL(qkv_heads_kernel<6>, grid, block, 0, s, a);
  else if (dim <= 10 * 512) hipLaunchKernelGGL(qkv_heads_kernel<10>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(qkv_heads_kernel<16>, grid, block, 0, s, a);
  return check_launch(name);
}
