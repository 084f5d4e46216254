// The step before the attention operator in one launch: per-head RMSNorm of
// the projected queries and keys, rotary position embedding, the query written
// in the [B, Hq, T, D] layout the attention operators read, and the key and
// value appended to the KV cache in place.
//
// Replaces the eager sequence of compiler/qwen3/adapters/attention.py:44-51:
//   q = q_norm(q_proj(x).view(B, T, Hq, D)).transpose(1, 2)
//   k = k_norm(k_proj(x).view(B, T, Hkv, D)).transpose(1, 2)
//   v = v_proj(x).view(B, T, Hkv, D).transpose(1, 2)
//   q, k = apply_rotary_pos_emb(q, k, cos, sin)
//   append_kv_batched(k, v, positions, cu_query, cache_key, cache_value)
// with the arithmetic and bf16 rounding points of those modules
// (transformers Qwen3RMSNorm and apply_rotary_pos_emb):
//   y  = bf16(x * rsqrt(mean(x^2) + eps))        mean, rsqrt in fp32
//   xn = bf16(w * y)
//   out_i = bf16(bf16(xn_i * cos_i) + bf16(rot_i * sin_i)),
//   rot_i = -xn_{i + D/2} for i < D/2, xn_{i - D/2} otherwise.
// Products of two bf16 values are exact in fp32, so every bf16 result above is
// the rounding of the same fp32 value the eager modules round; only mean(x^2),
// a sum whose order differs between implementations, may differ in its last
// bit.
//
// A row is a (token, projected head): the Hq query heads, then the Hkv key
// heads, then the Hkv value heads of each token.  LPR = D/8 lanes hold a row,
// 8 features (16 bytes) each; a wave takes 64/LPR heads of one kind at a time (a
// task), a block one token's tasks or some of them.  The partner of lane c for
// the rotation is lane c ^ LPR/2 (the other half of the row).  A key or value row
// is written to the cache only for a real token (t < count_r) whose position lies
// in [0, C); query rows are written for every token, as the eager sequence
// computes them.
//
// What bounds it: latency for a few tokens; for many the vector arithmetic and
// the waves' start (a row is 256 bytes at D = 128, and its rounding points take
// some 120 instructions).  So a task's kind, its addresses and its token's count
// and position are scalar work without a division, value rows are copied,
// roundings and the partner's exchange go two features at a time, and with many
// tokens the key and value rows of padded ones are not read.  Against one row per
// lane group with all of that per lane (16 query and 8 KV heads, D = 128, in
// graph replays): 8 x 384 tokens of which 391 are real 17.1 -> 11.1 us, 8 x 512
// real ones 22.0 -> 17.7 us (69 MB: 3.9 TB/s), 512 tokens 4.4 -> 4.1 us, 8 tokens
// 3.02 -> 2.82 us.  It loses where a token's heads fill few of a wave's lanes (4 query heads
// and 1 KV head, D = 64: 8 x 512 tokens 4.3 -> 6.4 us).
#include <algorithm>

#include "device_common.h"
#include "kernel_args.h"

namespace xattn {

// Two floats rounded to bf16: a packed pair of bits.
__device__ __forceinline__ uint32_t round2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// The partner lane's word (the other half of the row): DPP row_ror:8 within a
// 16-lane row (LPR = 16), the permlane16 swap (LPR = 32); a shuffle through LDS
// for LPR = 8.
template <int LPR>
__device__ __forceinline__ uint32_t partner_word(uint32_t x, int dc) {
  if constexpr (LPR == 16) {
    return __float_as_uint(dpp_move<kDppRowRor8>(__uint_as_float(x)));
  } else if constexpr (LPR == 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return dc < 16 ? r[1] : r[0];
  } else {
    return (uint32_t)__shfl_xor((int)x, LPR / 2, LPR);
  }
}

// Eight floats of a packed bf16 chunk.
struct Floats8 {
  float f[8];
};
__device__ __forceinline__ Floats8 unpack8(const u32x4 &x) {
  Floats8 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    r.f[2 * e] = bf16_lo(x[e]);
    r.f[2 * e + 1] = bf16_hi(x[e]);
  }
  return r;
}

// The normalised and rotated row (x: 8 features of it, w the norm weights, cs and
// sn the rotary tables).  The LPR lanes of a row call it together.
template <int LPR>
__device__ __forceinline__ u32x4 norm_rope(const u32x4 &x, const Floats8 &w, const Floats8 &cs, const Floats8 &sn,
                                           float eps, int dc) {
  const Floats8 xf = unpack8(x);
  float ss = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(xf.f[e], xf.f[e], ss);  // x^2 is exact in fp32
  ss = group_sum<LPR>(ss);
  const float inv = rsqrtf(ss / (float)(LPR * 8) + eps);
  // The rotation's sign: rot = -partner in the lower half of the row.
  const uint32_t sign = dc < LPR / 2 ? 0x80008000u : 0u;
  u32x4 out;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t y = round2(xf.f[2 * e] * inv, xf.f[2 * e + 1] * inv);
    const uint32_t xn = round2(w.f[2 * e] * bf16_lo(y), w.f[2 * e + 1] * bf16_hi(y));
    const uint32_t rot = partner_word<LPR>(xn, dc) ^ sign;
    const uint32_t p = round2(bf16_lo(xn) * cs.f[2 * e], bf16_hi(xn) * cs.f[2 * e + 1]);
    const uint32_t q = round2(bf16_lo(rot) * sn.f[2 * e], bf16_hi(rot) * sn.f[2 * e + 1]);
    out[e] = round2(bf16_lo(p) + bf16_lo(q), bf16_hi(p) + bf16_hi(q));
  }
  return out;
}

// Blocks by the number of tokens and of a token's tasks.
//  kSpread, few tokens of more than 4 tasks: one task a wave in blocks of 4 waves.  A
//   block of more waves starts later, and one of fewer waves than tasks has them wait
//   for each other (in blocks of 8 waves -> spread: 16 / 4 heads, D = 256, 12 tasks, 1 token
//   3.15 -> 2.63 us, 77 tokens 3.53 -> 3.02, 255 3.99 -> 3.84; 16 / 8, D = 128, 8 tasks, 77
//   tokens 3.12 -> 2.99, 192 3.23 -> 3.25, 512 4.07 -> 4.12; 32 / 8, D = 128, 12 tasks, 255
//   tokens 3.86 -> 3.70, 512 5.46 -> 5.69).
//  kWhole: a block takes a token, with a wave per task up to 8.
//  kMany: up to 4 waves take the tasks in turn and skip padded keys and values; with
//   fewer waves to start they gain more than the loads, begun before the position arrives,
//   lose (kWhole / kMany: 512 tokens 5.5 / 5.8 us, 1024 tokens at D = 256 10.6 / 11.5; 2048
//   tokens 12.3 / 11.2, 8 x 384 14.5 / 11.6, 2048 tokens at D = 256 16.6 / 15.8).
constexpr int64_t kNormRopeWholeTokens = 384, kNormRopeManyTokens = 2048;
constexpr int kNormRopeGridRows = 65535;
enum NormRopeMode { kSpread, kWhole, kMany };
constexpr int norm_rope_waves(NormRopeMode mode) { return mode == kWhole ? 8 : 4; }  // at most

template <int LPR, NormRopeMode MODE>
__global__ void __launch_bounds__(64 * norm_rope_waves(MODE), MODE == kWhole ? 2 : 4) norm_rope_kernel(const NormRopeArgs a) {
  constexpr int HEADS = 64 / LPR;  // heads of a task
  constexpr int WAVES = norm_rope_waves(MODE);
  const int lane = threadIdx.x & 63, head = lane / LPR, dc = lane % LPR;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // blockIdx.z: further tasks of the token (kSpread), or further rows.
  const int b = (int)((MODE == kSpread ? 0 : blockIdx.z * kNormRopeGridRows) + blockIdx.y), t = (int)blockIdx.x;
  if (b >= a.B) return;
  // The row's count and the token's position are block-uniform scalar loads.
  typedef const __attribute__((address_space(4))) int32_t *counts_ptr;
  typedef const __attribute__((address_space(4))) int64_t *positions_ptr;
  const counts_ptr cu = (counts_ptr)a.cu_query;
  const int64_t pos = ((positions_ptr)a.positions)[b * a.pos_sb + t * a.pos_st];
  const int count = cu[b + 1] - cu[b];
  const int q_tasks = (a.Hq + HEADS - 1) / HEADS, kv_tasks = (a.Hkv + HEADS - 1) / HEADS;
  // A block of fewer waves than WAVES has one for each task.
  for (int task = (MODE == kSpread ? (int)blockIdx.z * WAVES : 0) + wave; task < q_tasks + 2 * kv_tasks;
       task += WAVES) {
    const bool query = task < q_tasks, value = task >= q_tasks + kv_tasks;
    const int h = (task - (query ? 0 : (value ? q_tasks + kv_tasks : q_tasks))) * HEADS + head;
    const int heads = query ? a.Hq : a.Hkv;
    const bool real = t < count && pos >= 0 && pos < a.C;
    if (MODE == kMany && !query && !real) break;
    const View &src = query ? a.q : (value ? a.v : a.k);
    // Lanes past the last head repeat it; they write nothing.
    u32x4 out = load16(src.p + b * src.sb + t * src.st + (int64_t)min(h, heads - 1) * src.sh + dc * 8);
    if (!value) {
      const u32x4 w = load16((query ? a.q_weight : a.k_weight) + dc * 8);
      const u32x4 cs = load16(a.cos.p + b * a.cos.sb + t * a.cos.st + dc * 8);
      const u32x4 sn = load16(a.sin.p + b * a.sin.sb + t * a.sin.st + dc * 8);
      out = norm_rope<LPR>(out, unpack8(w), unpack8(cs), unpack8(sn), a.eps, dc);
    }
    if (query) {
      if (h < heads) store16(a.q_out + (((int64_t)b * a.Hq + h) * a.T + t) * (LPR * 8) + dc * 8, out);
    } else if (real && h < heads) {
      store16((value ? a.cache_value : a.cache_key) + (((int64_t)b * a.Hkv + h) * a.C + pos) * (LPR * 8) + dc * 8, out);
    }
    if constexpr (MODE == kSpread) break;
  }
}

template <int LPR, NormRopeMode MODE>
static void launch_norm_rope_mode(const NormRopeArgs &a, int tasks, hipStream_t stream) {
  constexpr int WAVES = norm_rope_waves(MODE);
  // Tokens by rows (no division in the kernel); a grid takes 65535 rows in y.
  const int rows = std::min(a.B, kNormRopeGridRows);
  const dim3 grid(a.T, rows, MODE == kSpread ? (tasks + WAVES - 1) / WAVES : (a.B + rows - 1) / rows);
  hipLaunchKernelGGL((norm_rope_kernel<LPR, MODE>), grid, dim3(64 * std::min(tasks, WAVES)), 0, stream, a);
}

template <int LPR>
static void launch_norm_rope_d(const NormRopeArgs &a, hipStream_t stream) {
  constexpr int HEADS = 64 / LPR;
  const int tasks = (a.Hq + HEADS - 1) / HEADS + 2 * ((a.Hkv + HEADS - 1) / HEADS);
  const int64_t tokens = (int64_t)a.B * a.T;
  if (tokens < kNormRopeWholeTokens && tasks > norm_rope_waves(kSpread)) launch_norm_rope_mode<LPR, kSpread>(a, tasks, stream);
  else if (tokens < kNormRopeManyTokens) launch_norm_rope_mode<LPR, kWhole>(a, tasks, stream);
  else launch_norm_rope_mode<LPR, kMany>(a, tasks, stream);
}

hipError_t launch_norm_rope(const NormRopeArgs &a, hipStream_t stream) {
  switch (a.D) {
    case 64: launch_norm_rope_d<8>(a, stream); break;
    case 128: launch_norm_rope_d<16>(a, stream); break;
    default: launch_norm_rope_d<32>(a, stream); break;
  }
  return hipGetLastError();
}

}  // namespace xattn
