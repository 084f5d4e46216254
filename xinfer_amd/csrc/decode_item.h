// A decode work item by four waves: its tiles, the combination of the waves, the
// output or record, and the merge in the launch (decode.hip has the overview).
#pragma once

#include "decode_common.h"
#include "launch.h"
#include "merge_common.h"

namespace xattn {

// LDS of an item block: the waves' buffers, then the query tile, whose place
// the waves' (m, l) take at the end.
constexpr int kItemWaves = kDecodeWaves, kItemThreads = kItemWaves * 64;
template <int DP, int NC>
struct ItemShared {
  using S = DecodeShape<DP, NC>;
  static constexpr int RING = kItemWaves * 2 * S::STAGE;
  static constexpr int BYTES = RING + S::QBYTES;
  static_assert(BYTES <= 80 * 1024, "two blocks per CU");
  // Barriers of an item with queries (process_item without a merge in the launch).
  static constexpr int BARRIERS = 2 + 2 * combine_passes<DP, NC, 2 * S::STAGE>() - 1;
  static_assert(kItemWaves * S::COLS * 8 <= S::QBYTES, "(m, l) of the waves");
};

struct DecodeItem {
  int b, h, split, nsplit, cnt, L, t0, t1;
  int kvb;      // cache row of the item's K/V: b, or b's page
  int counter;  // arrival counter of this (row, kv head)
  int64_t rec;  // first record of the item (its splits' records follow one another)
};

// The arguments a decode block uses (named as in AttnArgs), pinned in SGPRs by
// the kernel's prologue.
struct DecodeParams {
  View q, k, v;
  uint16_t *out;
  int64_t o_sb, o_sh, o_st;
  float *part_o, *part_ml;
  float scale_log2;
  int32_t D, G, T;
  uint64_t *arrive_ctr;  // in-launch merge (merge_in_launch), else null
  uint64_t tag;
};

// per: keys of one split; rec: the item's first record.
__device__ __forceinline__ DecodeItem make_item(int batch, int count, int length, int nsplit, int per, int h,
                                                int split, int counter, int64_t rec) {
  DecodeItem it;
  it.h = h;
  it.split = split;
  it.nsplit = nsplit;
  it.b = batch;
  it.kvb = batch;
  it.cnt = count;
  it.L = length;
  it.t0 = split * per;
  it.t1 = min(length, it.t0 + per);
  it.counter = counter;
  it.rec = rec;
  return it;
}

// Zero this item's share of out[b, h*G + g, t, :] for g < G and t in [count, T):
// the row's splits take equal runs of the padded tokens.
template <int DP>
__device__ __forceinline__ void zero_queries(const DecodeParams &a, const DecodeItem &it, int tid) {
  constexpr int CHUNKS = DP / 8, ROWS = kItemThreads / CHUNKS;
  const int n = a.T - it.cnt, D = a.D;
  const int t_begin = it.cnt + (int)((int64_t)n * it.split / it.nsplit);
  const int t_end = it.cnt + (int)((int64_t)n * (it.split + 1) / it.nsplit);
  const int c = tid % CHUNKS;
  if (c * 8 >= D) return;
  for (int g = 0; g < a.G; ++g) {
    uint16_t *const dst = a.out + it.b * a.o_sb + (int64_t)(it.h * a.G + g) * a.o_sh + c * 8;
    for (int t = t_begin + tid / CHUNKS; t < t_end; t += ROWS)
      store16(dst + (int64_t)t * a.o_st, u32x4{0, 0, 0, 0});
  }
}

// In-launch merge of one (row, kv head)'s split records, called by every
// thread of a block that has just written its records (AttnArgs::arrive_ctr
// set).  The planner takes this path only for launches whose split rows have
// at most kMergeSerialSplits splits and whose Hkv is a multiple of 8, and the
// kernel then runs every split of a (row, kv head) on one XCD (block b on XCD
// b % 8, which probe_xcd_dispatch checks once per device), so the records meet
// in that XCD's L2.  Each block, once its record stores are acknowledged,
// counts its arrival on the (row, kv head)'s counter; the last to arrive reads
// the records past its CU's L1 and folds them as merge.hip's one-thread-per-
// (vector, 4 features) layout does (merge_common.h: fold), splits in increasing
// order, so that both paths give the same bits, and resets the counter to zero.
//
// Counter word: arrivals (bits 0-11), XCC of the first arrival (12-15),
// arrivals from another XCC (16-27), the launch's tag (28-63).  The first
// arrival claims a word that does not carry this launch's tag (zero after the
// previous launch's reset, or whatever the workspace held) by compare-and-
// swap; every other arrival adds itself with one fetch-and-add, so no arrival
// waits behind another.  A (row, kv head) whose splits ran on more than one
// XCC gets NaN outputs rather than a fold of records another L2 may hold.
template <int DP>
__device__ void merge_in_launch(const DecodeParams &a, const DecodeItem &it, int qrows, char *smem) {
  uint32_t &arrival = *reinterpret_cast<uint32_t *>(smem);  // the block is done with its buffers
  const int tid = threadIdx.x;
  __builtin_amdgcn_s_waitcnt(0);  // this thread's record stores are acknowledged
  __syncthreads();
  if (tid == 0) {
    uint32_t xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    xcc &= 15u;
    uint64_t *const ctr = a.arrive_ctr + it.counter;
    const uint64_t tag = a.tag;
    uint64_t seen = 0;
    bool claimed = false;
    // Ends after at most two attempts: only this launch's first arrival
    // writes its tag, and no reset happens before every arrival is counted.
    while ((seen >> 28) != tag) {
      if (__hip_atomic_compare_exchange_strong(ctr, &seen, (tag << 28) | ((uint64_t)xcc << 12) | 1u,
                                               __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        claimed = true;
        break;
      }
    }
    uint32_t count = 1, mixed = 0;
    if (!claimed) {
      const bool other = ((seen >> 12) & 15u) != xcc;
      const uint64_t before = __hip_atomic_fetch_add(ctr, (uint64_t)1 + (other ? (uint64_t)1 << 16 : 0),
                                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      count = (uint32_t)(before & 0xfffu) + 1;
      mixed = (uint32_t)((before >> 16) & 0xfffu) + (other ? 1u : 0u);
    }
    const bool last = count == (uint32_t)it.nsplit;
    if (last) __hip_atomic_store(ctr, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    arrival = !last ? 0u : (mixed == 0 ? 1u : 2u);
  }
  __syncthreads();
  const uint32_t flag = arrival;
  if (flag == 0) return;

  constexpr int FQ = DP / 4;  // feature quads of a padded vector
  const int D = a.D, G = a.G, nsplit = it.nsplit;
  // Record (split s, vector j) of this (row, kv head): rec0 + s * qrows + j.
  const int64_t rec0 = it.rec - (int64_t)it.split * qrows;
  const __amdgpu_buffer_rsrc_t o_rsrc = buffer_rsrc(a.part_o + rec0 * D, (uint32_t)(nsplit * qrows * D * 4));
  const __amdgpu_buffer_rsrc_t ml_rsrc = buffer_rsrc(a.part_ml + 2 * rec0, (uint32_t)(nsplit * qrows * 8));
  for (int idx = tid; idx < qrows * FQ; idx += kItemThreads) {
    const int j = idx / FQ, f = idx - j * FQ;
    if (f * 4 >= D) continue;
    u32x2 ml[kMergeSerialSplits];
    u32x4 o[kMergeSerialSplits];
#pragma unroll
    for (int s = 0; s < kMergeSerialSplits; ++s)
      if (s < nsplit) {
        ml[s] = buffer_load8_l2(ml_rsrc, (uint32_t)((s * qrows + j) * 8));
        o[s] = buffer_load16_l2(o_rsrc, (uint32_t)(((s * qrows + j) * D + 4 * f) * 4));
      }
    MergeState st{-INFINITY, 0.0f, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int s = 0; s < kMergeSerialSplits; ++s) {
      if (s >= nsplit) break;
      fold(st, __uint_as_float(ml[s].x), __uint_as_float(ml[s].y), __builtin_bit_cast(f32x4, o[s]));
    }
    const float inv = 1.0f / st.l;
    uint16_t *dst = a.out + it.b * a.o_sb + (int64_t)(it.h * G + j % G) * a.o_sh + (int64_t)(j / G) * a.o_st + 4 * f;
    *as_global(reinterpret_cast<u32x2 *>(dst)) =
        flag == 1 ? u32x2{pack_bf16x2(st.o.x * inv, st.o.y * inv), pack_bf16x2(st.o.z * inv, st.o.w * inv)}
                  : u32x2{0x7fc07fc0u, 0x7fc07fc0u};
  }
}

// One work item; its four waves, of threads tid 0 .. 255, call it.  raw_page: the row's page
// table entry (read_page), awaited once the first loads are under way.
template <int DP, int NC>
__device__ __forceinline__ void process_item(const DecodeParams &a, DecodeItem &it, int raw_page, int kv_rows,
                                             char *smem, int tid) {
  using S = DecodeShape<DP, NC>;
  using M = ItemShared<DP, NC>;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.G, D = a.D;
  if (it.cnt == 0) {
    zero_queries<DP>(a, it, tid);
    return;
  }
  const int qrows = it.cnt * G;
  const int ntile = (it.t1 - it.t0 + S::KT - 1) / S::KT;

  // This wave's first K tile, the query tile, this wave's first V tile.
  KvStream<DP, NC> kv;
  const uint32_t ring = lds_address(smem);
  kv.init(a.k, a.v, D, ring + wave * 2 * S::STAGE, lane);
  kv.open(a.k, a.v, it.kvb, it.h, it.t1);
  const int first = it.t0 + wave * S::KT;
  if (wave < ntile) kv.issue_k(first);
  issue_query<DP, NC, kItemWaves>(a.q, it.b, it.h, G, D, qrows, ring + M::RING, wave, lane);
  if (wave < ntile) kv.issue_v(first);
  __builtin_amdgcn_sched_barrier(0);
  // Another page than row b (never with the identity table): drain and reload.
  const int page = page_in_range(raw_page, kv_rows);
  if (__builtin_expect(page != it.kvb, 0)) {
    wait_loads<0>();
    it.kvb = page;
    kv.open(a.k, a.v, page, it.h, it.t1);
    if (wave < ntile) {
      kv.issue_k(first);
      kv.issue_v(first);
    }
  }
  WaveAttention<DP, NC> w;
  w.init(lane);
  w.begin(qrows, G, it.L - it.cnt, it.t1);
  if (wave < ntile) wait_loads<S::LOADS>();
  else wait_loads<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  w.load_query(reinterpret_cast<const uint16_t *>(smem + M::RING));

  const uint16_t *const Kt = reinterpret_cast<const uint16_t *>(smem + wave * 2 * S::STAGE);
  const uint16_t *const Vt = Kt + S::STAGE / 2;
  for (int tile = wave; tile < ntile; tile += kItemWaves) {
    const bool next = tile + kItemWaves < ntile;
    const int kb = it.t0 + tile * S::KT, kb_next = kb + kItemWaves * S::KT;
    wait_loads<S::LOADS>();  // K of this tile (its V may still be on its way)
    f32x4 s[S::KG][NC];
    w.scores(Kt, s);
    wait_lds();
    if (next) kv.issue_k(kb_next);
    uint32_t pw[NC][S::KG][2];
    w.weights(s, kb, a.scale_log2, pw);
    if (next) wait_loads<S::LOADS>();  // V of this tile (the next tile's K may still be on its way)
    else wait_loads<0>();
    w.values(Vt, pw);
    wait_lds();
    if (next) kv.issue_v(kb_next);
  }
  if (it.cnt < a.T) zero_queries<DP>(a, it, tid);

  // Combine the four waves, then write the output or a partial record.
  __syncthreads();  // every wave has read the query tile
  combine_waves<DP, NC, kItemWaves, 2 * S::STAGE>(
      w, smem, reinterpret_cast<float2 *>(smem + M::RING), qrows, D, tid, wave,
      [&](int j, int d, const f32x4 &o, float m, float l) {
        if (it.nsplit == 1) {
          const int g = j % G, i = j / G;
          uint16_t *dst = a.out + it.b * a.o_sb + (int64_t)(it.h * G + g) * a.o_sh + (int64_t)i * a.o_st + d;
          *as_global(reinterpret_cast<u32x2 *>(dst)) =
              u32x2{pack_bf16x2(o[0] / l, o[1] / l), pack_bf16x2(o[2] / l, o[3] / l)};
        } else {
          const int64_t rec = it.rec + j;
          *as_global(reinterpret_cast<f32x4 *>(a.part_o + rec * D + d)) = o;
          if (d == 0)
            *as_global(reinterpret_cast<u32x2 *>(a.part_ml + 2 * rec)) =
                u32x2{__float_as_uint(m), __float_as_uint(l)};
        }
      });
  if (a.arrive_ctr != nullptr && it.nsplit > 1) merge_in_launch<DP>(a, it, qrows, smem);
}

// The arguments of a block of decode items, loaded in one round trip (see
// XATTN_PIN_VIEW).
struct DecodeLocals {
  RowLookup<RowSched> rows;
  int nrows;
  DecodeParams p;
  const int32_t *blocks;
  int64_t blocks_stride;
  int kv_rows;
  __device__ __forceinline__ explicit DecodeLocals(const AttnArgs &a)
      : nrows(a.nrows),
        p{a.q,          a.k, a.v, a.out, a.o_sb,       a.o_sh, a.o_st, a.part_o, a.part_ml,
          a.scale_log2, a.D, a.G, a.T,   a.arrive_ctr, a.tag},
        blocks(a.blocks), blocks_stride(a.blocks_stride), kv_rows(a.kv_rows) {
    rows.load(a.rows);
    asm volatile(""
                 : XATTN_PIN_BEGINS(rows), XATTN_PIN_ROWSCHED(rows.first), "+s"(nrows), XATTN_PIN_VIEW(p.q),
                   XATTN_PIN_VIEW(p.k), XATTN_PIN_VIEW(p.v), "+s"(p.out), "+s"(p.o_sb), "+s"(p.o_sh), "+s"(p.o_st),
                   "+s"(p.part_o), "+s"(p.part_ml), "+s"(p.scale_log2), "+s"(p.D), "+s"(p.G), "+s"(p.T),
                   "+s"(blocks), "+s"(blocks_stride), "+s"(kv_rows));
  }
};

// Item `item` of a launch: (row, kv head, split) in this order.
__device__ __forceinline__ DecodeItem launch_item(const AttnArgs &a, const DecodeLocals &l, int item) {
  const RowSched rs = l.rows.find(a.rows, l.nrows, item);
  const int local = item - rs.item_begin, h = local / rs.nsplit;
  return make_item(rs.batch, rs.count, rs.length, rs.nsplit, rs.ntiles, h, local - h * rs.nsplit, 0,
                   rs.rec_begin + (int64_t)local * (rs.count * l.p.G));
}

// A block of eight waves beside a prefill kernel's (attention_both_kernel): decode
// items 2 * block and 2 * block + 1 of the launch's total_items, four waves and half of
// the LDS each.  The two meet in every barrier, which an item has by its type
// alone; a half without keys to read does only them.
template <int DP, int NC>
__device__ __forceinline__ void decode_pair(const AttnArgs &a, int block, char *smem) {
  using M = ItemShared<DP, NC>;
  const DecodeLocals l(a);
  const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kItemThreads);
  const int tid = (int)threadIdx.x % kItemThreads, item = 2 * block + half, items = a.total_items;
  if (2 * block >= items) return;
  DecodeItem it{};
  if (item < items) it = launch_item(a, l, item);
  if (it.cnt == 0) {
    if (item < items) zero_queries<DP>(l.p, it, tid);
#pragma unroll
    for (int i = 0; i < M::BARRIERS; ++i) __builtin_amdgcn_s_barrier();
    return;
  }
  DecodeParams p = l.p;
  p.arrive_ctr = nullptr;
  process_item<DP, NC>(p, it, read_page(l.blocks, l.blocks_stride, it.b), l.kv_rows, smem + half * M::BYTES, tid);
}

}  // namespace xattn
