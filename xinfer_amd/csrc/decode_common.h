// A decode wave (decode.hip): its stream of K and V tiles through its LDS buffers,
// and the arithmetic on a tile.
//
// The path is bound by reading K and V from HBM once.  A wave takes tiles of
// 8 KB of K and 8 KB of V (64, 32 or 16 keys for head dims 64, 128, 256)
// through two LDS buffers of its own, with no barrier between the waves.  K
// and V travel HBM -> LDS without registers (buffer_load_dwordx4 ... lds); the
// K buffer is refilled as soon as the scores have read it, the V buffer as soon
// as the accumulation has, so a wave has loads in flight while it computes and
// no register holds data on its way.  The descriptors end at the last key of
// the run: loads past it write zeros without touching memory.
//
// The arithmetic is on the matrix cores (16x16 tiles), with the query vectors
// as columns:
//   S^T[key, c] = K[key, :] . Q[c, :]       A = K (LDS), B = Q^T (registers)
//   O^T[d, c]  += V^T[d, key] P^T[key, c]   A = V^T (LDS, transposing reads), B = P^T
// The S^T accumulator of keys 4g..4g+3 of two 16-key groups is, register by
// register, the B operand of the PV product (k = 32; k = 16 for head dim 256).
//
// A row with at most kExactVectors = 8 query vectors keeps the fp32 precision
// of its softmax weights: the query is repeated in columns qv.. and 2qv.., and
// the columns take the high, middle and low 8 mantissa bits of the weight as
// bf16, three exact products whose sums are added at the end.  Wider rows round
// the weights to bf16 once, and their normaliser sums the rounded weights, so
// that an output stays an exact convex combination of the values (as in
// prefill.hip).  NC column groups of 16 hold the vectors: one serves up to 5
// exact or 16 rounded ones, two up to 8 and 32.
//
// MFMA 16x16x32 lane layout (A: 16xK32, B: K32x16, C: 16x16; g = lane / 16):
//   A lane: row lane%16, k = 8g + 0..7      B lane: col lane%16, same k
//   C lane, reg r: row 4g + r, col lane%16  (16x16x16: k = 4g + 0..3)
#pragma once

#include "launch.h"
#include "prefill_common.h"

namespace xattn {

template <int DP, int NC>
struct DecodeShape {
  static constexpr int CHUNKS = DP / 8;          // 16-byte chunks of a key row
  static constexpr int LOADS = 8;                // 1 KB loads per wave tile and tensor
  static constexpr int RPL = 512 / DP;           // key rows per load
  static constexpr int KT = LOADS * RPL;         // keys per wave tile: 64, 32, 16
  static constexpr int KG = KT / 16;             // 16-key groups per wave tile
  static constexpr int KS = DP / 32;             // k-steps of the scores
  static constexpr int DT = DP / 16;             // 16-feature d tiles of the output
  static constexpr int COLS = 16 * NC;
  // Loads after which the swizzle pattern of the fetched chunks repeats.
  static constexpr int NVK = 16 / RPL, NVV = 8 / RPL;
  static constexpr int STAGE = 8192;             // bytes of a wave's K (or V) buffer
  static constexpr int QBYTES = COLS * DP * 2;   // the query tile
  static constexpr int NKO = KS < 4 ? KS : 4, NVO = DT < 8 ? DT : 8;  // distinct LDS read offsets
};

// XOR swizzles of the 16-byte chunks of a key row in LDS (chunk c of key k is
// stored at slot c ^ swz(k)).  K reads take one chunk of 16 consecutive keys,
// V reads two neighbouring chunks of 8 keys per LDS pass; with 8 chunks to a
// row two rows share the banks' width.
template <int CHUNKS>
__device__ __forceinline__ int stream_k_swizzle(int key) { return CHUNKS >= 16 ? (key & 15) : ((key >> 1) & 7); }
template <int CHUNKS>
__device__ __forceinline__ int stream_v_swizzle(int key) { return CHUNKS >= 16 ? 2 * (key & 7) : 2 * ((key >> 1) & 3); }

// One 16-byte-per-lane load into LDS as prefill_common.h's lds_load16, for code
// whose scalar operands may come from vector lanes (v_readlane, as spilled
// scalars and the capture row table do): the hardware wants five wait states between such a
// write and a vector-memory read of the register, and the compiler does not
// look into the asm.  STREAM: the non-temporal cache policy, for data read once.
template <bool STREAM>
__device__ __forceinline__ void lds_load16_lanes(u32x4 rsrc, uint32_t lds_byte, uint32_t voffset, uint32_t soffset) {
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_byte)), "v"(voffset), "s"(rsrc),
                   "s"(__builtin_amdgcn_readfirstlane(soffset))
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(__builtin_amdgcn_readfirstlane(lds_byte)), "v"(voffset), "s"(rsrc),
                   "s"(__builtin_amdgcn_readfirstlane(soffset))
                 : "memory", "m0");
}

// Wait until at most N of this wave's vector-memory operations are outstanding.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Wait for this wave's LDS reads: a buffer they came from may be refilled.
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16_k16(u32x2 a, u32x2 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(shortx4, a), __builtin_bit_cast(shortx4, b), c,
                                                   0, 0, 0);
}

// One wave's stream over a run of keys of a (row, kv head): its K and V buffers
// and the loads that fill them.
template <int DP, int NC>
struct KvStream {
  using S = DecodeShape<DP, NC>;
  u32x4 k_rsrc, v_rsrc;
  uint32_t k_row, v_row;       // bytes of a key row
  uint32_t k_voff[S::NVK], v_voff[S::NVV];
  uint32_t kbuf, vbuf;         // LDS byte addresses

  // Load i of a tile fills 16-byte slots 64i + lane: key (64i + lane) / CHUNKS,
  // slot (64i + lane) % CHUNKS, holding chunk slot ^ swizzle (clamped into the
  // row past D: finite values that only meet zero query features or unused
  // output rows).
  __device__ __forceinline__ void init(const View &k, const View &v, int D, uint32_t base, int lane) {
    k_row = (uint32_t)(k.st * 2);
    v_row = (uint32_t)(v.st * 2);
    kbuf = base;
    vbuf = base + S::STAGE;
    const int key = lane / S::CHUNKS, slot = lane % S::CHUNKS, last = D / 8 - 1;
#pragma unroll
    for (int i = 0; i < S::NVK; ++i) {
      const int kk = key + i * S::RPL;
      k_voff[i] = (uint32_t)kk * k_row + (uint32_t)min(slot ^ stream_k_swizzle<S::CHUNKS>(kk), last) * 16;
    }
#pragma unroll
    for (int i = 0; i < S::NVV; ++i) {
      const int kk = key + i * S::RPL;
      v_voff[i] = (uint32_t)kk * v_row + (uint32_t)min(slot ^ stream_v_swizzle<S::CHUNKS>(kk), last) * 16;
    }
  }
  // The run's keys end before t1 of cache row `row`, kv head h.
  __device__ __forceinline__ void open(const View &k, const View &v, int row, int h, int t1) {
    k_rsrc = buffer_words(k.p + row * k.sb + (int64_t)h * k.sh, (uint32_t)t1 * k_row);
    v_rsrc = buffer_words(v.p + row * v.sb + (int64_t)h * v.sh, (uint32_t)t1 * v_row);
  }
  // The K (V) tile of keys kb .. kb + KT - 1.
  __device__ __forceinline__ void issue_k(int kb) const {
#pragma unroll
    for (int i = 0; i < S::LOADS; ++i)
      lds_load16_lanes<true>(k_rsrc, kbuf + i * 1024, k_voff[i % S::NVK],
                        (uint32_t)(kb + i / S::NVK * S::NVK * S::RPL) * k_row);
  }
  __device__ __forceinline__ void issue_v(int kb) const {
#pragma unroll
    for (int i = 0; i < S::LOADS; ++i)
      lds_load16_lanes<true>(v_rsrc, vbuf + i * 1024, v_voff[i % S::NVV],
                        (uint32_t)(kb + i / S::NVV * S::NVV * S::RPL) * v_row);
  }
};

// Loads of the query tile by the WAVES waves of a block: row c holds column c's
// vector of (row b, kv head h); zeros for unused columns and past D.
template <int DP, int NC, int WAVES>
__device__ __forceinline__ void issue_query(const View &q, int b, int h, int G, int D, int qrows, uint32_t dst,
                                            int wave, int lane) {
  using S = DecodeShape<DP, NC>;
  constexpr int QL = S::QBYTES / 1024;  // 1 KB loads of the query tile
  const u32x4 q_rsrc = buffer_words(q.p + b * q.sb + (int64_t)(h * G) * q.sh, 0x7fffffffu);
#pragma unroll
  for (int i = 0; i < (QL + WAVES - 1) / WAVES; ++i) {
    const int ld = i * WAVES + wave;
    if (QL % WAVES == 0 || ld < QL) {
      const int slot = ld * 64 + lane;
      const int c = slot / S::CHUNKS, chunk = (slot % S::CHUNKS) ^ stream_k_swizzle<S::CHUNKS>(c);
      const int rep = qrows <= kExactVectors ? c / qrows : 0, j = c - rep * qrows;
      const uint32_t off = (rep < 3 && j < qrows && chunk * 8 < D)
                               ? (uint32_t)(((j % G) * q.sh + (j / G) * q.st) * 2 + chunk * 16)
                               : 0x80000000u;
      lds_load16_lanes<false>(q_rsrc, dst + ld * 1024, off, 0);
    }
  }
}

// One wave's attention state over the columns of a (row, kv head).
template <int DP, int NC>
struct WaveAttention {
  using S = DecodeShape<DP, NC>;
  int col, grp;                    // lane % 16, lane / 16
  int k_off[S::NKO], v_off[S::NVO];
  bf16x8 qf[NC][S::KS];            // Q^T B operands: column col, features 32ks + 8grp .. +7
  bool exact;
  int rep[NC], lim[NC];            // the column's part of the weight (0 high, 1 middle, 2 low), the last key it sees
  int first_lim, t1;               // last key of the first query, end of the run
  f32x4 acc[S::DT][NC];            // O^T[16dt + 4grp + r][column]
  float m_run[NC], l_run[NC];

  // LDS read offsets (elements).  K operand of k-step ks: key col (+16 per
  // group), chunk 4ks + grp.  V operand of d tile dt: 16-lane group grp, lane
  // col addresses key 4grp + col/4 (+16 per group) and features 16dt +
  // 4(col%4); the swizzle permutes the d tiles among eight slots.
  __device__ __forceinline__ void init(int lane) {
    col = lane & 15;
    grp = lane >> 4;
#pragma unroll
    for (int ks = 0; ks < S::NKO; ++ks)
      k_off[ks] = col * DP + ((4 * ks + grp) ^ stream_k_swizzle<S::CHUNKS>(col)) * 8;
    const int kk = 4 * grp + (col >> 2), swz = stream_v_swizzle<S::CHUNKS>(kk);
#pragma unroll
    for (int dt = 0; dt < S::NVO; ++dt)
      v_off[dt] = kk * DP + ((2 * dt + ((col & 3) >> 1)) ^ swz) * 8 + 4 * (col & 1);
  }

  // Start a run: qrows vectors of G heads, keys before run_end, the first query's
  // last key first_key_limit.
  __device__ __forceinline__ void begin(int qrows, int G, int first_key_limit, int run_end) {
    exact = qrows <= kExactVectors;
    first_lim = first_key_limit;
    t1 = run_end;
#pragma unroll
    for (int nc = 0; nc < NC; ++nc) {
      const int c = nc * 16 + col;
      rep[nc] = exact ? c / qrows : 0;
      const int j = c - rep[nc] * qrows;
      lim[nc] = j < qrows ? min(first_lim + j / G, t1 - 1) : t1 - 1;
      m_run[nc] = -INFINITY;
      l_run[nc] = 0.0f;
#pragma unroll
      for (int dt = 0; dt < S::DT; ++dt) acc[dt][nc] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  }

  // The query operands, once the query tile is in LDS.
  __device__ __forceinline__ void load_query(const uint16_t *qt) {
#pragma unroll
    for (int nc = 0; nc < NC; ++nc)
#pragma unroll
      for (int ks = 0; ks < S::KS; ++ks)
        qf[nc][ks] = as_bf16x8(*reinterpret_cast<const u32x4 *>(
            qt + (nc * 16 + col) * DP + ((4 * ks + grp) ^ stream_k_swizzle<S::CHUNKS>(col)) * 8));
  }

  // S^T of a tile: s[kg][nc][r] is key 16kg + 4grp + r against column nc*16 + col.
  __device__ __forceinline__ void scores(const uint16_t *Kt, f32x4 (&s)[S::KG][NC]) const {
#pragma unroll
    for (int kg = 0; kg < S::KG; ++kg)
#pragma unroll
      for (int nc = 0; nc < NC; ++nc) s[kg][nc] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int ks = 0; ks < S::KS; ++ks)
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg) {
        const bf16x8 ka = as_bf16x8(
            *reinterpret_cast<const u32x4 *>(Kt + k_off[ks % S::NKO] + ks / S::NKO * 128 + kg * 16 * DP));
#pragma unroll
        for (int nc = 0; nc < NC; ++nc) s[kg][nc] = mfma16(ka, qf[nc][ks], s[kg][nc]);
      }
  }

  // Online softmax of the tile of keys kb ..: pw are the P^T B operands, keys
  // 16kg + 4grp .. +3 of the column.
  __device__ __forceinline__ void weights(f32x4 (&s)[S::KG][NC], int kb, float c, uint32_t (&pw)[NC][S::KG][2]) {
    if (kb + S::KT > t1 || kb + S::KT - 1 > first_lim) {
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg)
#pragma unroll
        for (int nc = 0; nc < NC; ++nc)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[kg][nc][r] = kb + 16 * kg + 4 * grp + r > lim[nc] ? -INFINITY : s[kg][nc][r];
    }
#pragma unroll
    for (int nc = 0; nc < NC; ++nc) {
      float mx = -INFINITY;
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[kg][nc][r]);
      const float mt = pair_max32(pair_max16(mx)) * c;  // tile max of the column, log2 units
      if (__builtin_amdgcn_ballot_w64(mt > m_run[nc])) {
        const float m_new = fmaxf(m_run[nc], mt);
        const float alpha = fast_exp2(m_run[nc] - (m_new == -INFINITY ? 0.0f : m_new));
        l_run[nc] *= alpha;
#pragma unroll
        for (int dt = 0; dt < S::DT; ++dt) acc[dt][nc] *= alpha;
        m_run[nc] = m_new;
      }
      const float m_use = m_run[nc] == -INFINITY ? 0.0f : m_run[nc];
#pragma unroll
      for (int kg = 0; kg < S::KG; ++kg) {
        float w[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = fast_exp2(fmaf(s[kg][nc][r], c, -m_use));
          // p = high + middle + low, each a bf16 (8 mantissa bits) taken from
          // the remainder of the one before.
          const float high = __uint_as_float(f32_to_bf16_bits(p) << 16);
          const float rest = rep[nc] == 0 ? p : p - high;
          const float middle = __uint_as_float(f32_to_bf16_bits(rest) << 16);
          w[r] = rep[nc] == 2 ? rest - middle : rest;
          l_run[nc] += exact ? p : high;
        }
        pw[nc][kg][0] = pack_bf16x2(w[0], w[1]);
        pw[nc][kg][1] = pack_bf16x2(w[2], w[3]);
      }
    }
  }

  // O^T += V^T P^T of a tile.
  __device__ __forceinline__ void values(const uint16_t *Vt, const uint32_t (&pw)[NC][S::KG][2]) {
#pragma unroll
    for (int dt = 0; dt < S::DT; ++dt) {
      const uint16_t *vp = Vt + v_off[dt % S::NVO] + dt / S::NVO * 128;
      if constexpr (S::KG == 1) {
        const u32x2 va = lds_read_tr16(vp);
#pragma unroll
        for (int nc = 0; nc < NC; ++nc)
          acc[dt][nc] = mfma16_k16(va, u32x2{pw[nc][0][0], pw[nc][0][1]}, acc[dt][nc]);
      } else {
#pragma unroll
        for (int kg = 0; kg < S::KG; kg += 2) {
          const u32x2 lo = lds_read_tr16(vp + kg * 16 * DP), hi = lds_read_tr16(vp + (kg + 1) * 16 * DP);
          const bf16x8 va = as_bf16x8(u32x4{lo.x, lo.y, hi.x, hi.y});
#pragma unroll
          for (int nc = 0; nc < NC; ++nc)
            acc[dt][nc] = mfma16(
                va, as_bf16x8(u32x4{pw[nc][kg][0], pw[nc][kg][1], pw[nc][kg + 1][0], pw[nc][kg + 1][1]}), acc[dt][nc]);
        }
      }
    }
  }
};

// Passes of combine_waves, and its barriers: 2 * passes - 1.
template <int DP, int NC, int BYTES>
constexpr int combine_passes() {
  using S = DecodeShape<DP, NC>;
  return S::DT * NC * 1024 > BYTES ? S::DT * NC * 1024 / BYTES : 1;
}

// Combines the states of a block's WAVES waves and hands every query vector's
// quads of features to write(j, d, o, m, l) (features d .. d+3 of vector j, the
// unnormalised sum, the running max and the normaliser).  Wave w's state goes
// through the BYTES bytes at states + w * 2 * STAGE, in passes of DTP d tiles,
// laid out [d tile][column group][lane] quads; the columns of a quad are rotated
// so that both the writes and the reads of neighbouring quads spread over the
// banks.  red_ml holds [wave][column] (m, l).
template <int DP, int NC, int WAVES, int BYTES, typename Write>
__device__ __forceinline__ void combine_waves(const WaveAttention<DP, NC> &w, char *states, float2 *red_ml, int qrows,
                                              int D, int tid, int wave, Write &&write) {
  using S = DecodeShape<DP, NC>;
  constexpr int PASSES = combine_passes<DP, NC, BYTES>();
  constexpr int DTP = S::DT / PASSES, FQ = DTP * 4;  // d tiles and feature quads of a pass
  const int col = w.col, grp = w.grp;
#pragma unroll
  for (int pass = 0; pass < PASSES; ++pass) {
    if (pass > 0) __syncthreads();
#pragma unroll
    for (int dl = 0; dl < DTP; ++dl)
#pragma unroll
      for (int nc = 0; nc < NC; ++nc)
        *reinterpret_cast<f32x4 *>(states + wave * 2 * S::STAGE +
                                   ((dl * NC + nc) * 64 + grp * 16 + ((col + 4 * dl + grp) & 15)) * 16) =
            w.acc[pass * DTP + dl][nc];
    if (pass == 0) {
#pragma unroll
      for (int nc = 0; nc < NC; ++nc) {
        const float l = pair_sum32(pair_sum16(w.l_run[nc]));
        if (grp == 0) red_ml[wave * S::COLS + nc * 16 + col] = make_float2(w.m_run[nc], l);
      }
    }
    __syncthreads();
    for (int idx = tid; idx < qrows * FQ; idx += WAVES * 64) {
      const int j = idx / FQ, f = idx % FQ, dl = f / 4, g4 = f % 4;
      const int d = (pass * DTP + dl) * 16 + 4 * g4;
      if (d >= D) continue;
      float2 ml[WAVES];
      float mx = -INFINITY;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        ml[v] = red_ml[v * S::COLS + j];
        mx = fmaxf(mx, ml[v].x);
      }
      const float mu = mx == -INFINITY ? 0.0f : mx;
      auto state = [&](int v, int c) {
        return *reinterpret_cast<const f32x4 *>(
            states + v * 2 * S::STAGE + ((dl * NC + c / 16) * 64 + g4 * 16 + ((c + f) & 15)) * 16);
      };
      f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
      float lsum = 0.0f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        f32x4 ov = state(v, j);
        if (w.exact) {
          const f32x4 middle = state(v, j + qrows), low = state(v, j + 2 * qrows);
          // An infinite value times a zero remainder is not a number: keep the
          // high part alone then.
#pragma unroll
          for (int e = 0; e < 4; ++e) ov[e] = fabsf(ov[e]) < INFINITY ? ov[e] + (middle[e] + low[e]) : ov[e];
        }
        const float wt = fast_exp2(ml[v].x - mu);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = fmaf(wt, ov[e], o[e]);
        lsum = fmaf(wt, ml[v].y, lsum);
      }
      write(j, d, o, mx, lsum);
    }
  }
}

}  // namespace xattn
