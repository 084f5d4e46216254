// Split-KV attention for rows with few query vectors per KV head (at most
// kStreamMaxVectors = 32 of G * count): the q_len = 1 decode step, drafted
// tokens and short appended chunks.
//
// Replaces, for those rows, the ATen FlashAttention-2 call of
// compiler/common/kernels/attention.cpp:66-72 / :116-117.  Math: for every
// query vector j = i*G + g of KV head h in row r,
//   out_j = sum_t softmax_t(scale * q_j . k_t) v_t  over keys t <= L - count + i
// (lower-right causal), fp32 scores / softmax / accumulation, bf16 in and out.
//
// Work item = (row, kv head, chunk of keys).  A block is 4 waves; each wave
// takes every fourth tile of the item through its own LDS buffers
// (decode_common.h); two blocks share a CU.  The four waves are combined
// through LDS at the end of the item.  One chunk per (row, head): the block
// writes normalised bf16 output.  Several chunks: each writes an fp32 partial
// record per query vector, combined by merge.hip or in the launch
// (merge_in_launch).  The schedule depends only on the lengths, so results are
// deterministic and a row's output never depends on another row's data.
//
// Padded queries (t >= count) get zeros from the row's items, each its share;
// a row with count == 0 is scheduled only for that.
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
__device__ __forceinline__ void zero_queries(const DecodeParams &a, const DecodeItem &it) {
  constexpr int CHUNKS = DP / 8, ROWS = kItemThreads / CHUNKS;
  const int n = a.T - it.cnt, D = a.D;
  const int t_begin = it.cnt + (int)((int64_t)n * it.split / it.nsplit);
  const int t_end = it.cnt + (int)((int64_t)n * (it.split + 1) / it.nsplit);
  const int c = (int)threadIdx.x % CHUNKS;
  if (c * 8 >= D) return;
  for (int g = 0; g < a.G; ++g) {
    uint16_t *const dst = a.out + it.b * a.o_sb + (int64_t)(it.h * a.G + g) * a.o_sh + c * 8;
    for (int t = t_begin + (int)threadIdx.x / CHUNKS; t < t_end; t += ROWS)
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

// One work item; every wave of the block calls it.  raw_page: the row's page
// table entry (read_page), awaited once the first loads are under way.
template <int DP, int NC>
__device__ __forceinline__ void process_item(const DecodeParams &a, DecodeItem &it, int raw_page, int kv_rows,
                                             char *smem) {
  using S = DecodeShape<DP, NC>;
  using M = ItemShared<DP, NC>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.G, D = a.D;
  if (it.cnt == 0) {
    zero_queries<DP>(a, it);
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
  if (it.cnt < a.T) zero_queries<DP>(a, it);

  // Combine the four waves, then write the output or a partial record.
  __syncthreads();  // every wave has read the query tile
  combine_waves<DP, NC, kItemWaves, 2 * S::STAGE>(
      w, smem, reinterpret_cast<float2 *>(smem + M::RING), qrows, D, wave,
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

template <int DP, int NC>
__global__ void __launch_bounds__(kItemThreads, 2) decode_kernel(const AttnArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[ItemShared<DP, NC>::BYTES];
  // Every argument of the block, loaded in one round trip (see XATTN_PIN_VIEW).
  RowLookup<RowSched> rows;
  rows.load(a.rows);
  int nrows = a.nrows;
  DecodeParams p{a.q,          a.k, a.v, a.out, a.o_sb,       a.o_sh, a.o_st, a.part_o, a.part_ml,
                 a.scale_log2, a.D, a.G, a.T,   a.arrive_ctr, a.tag};
  const int32_t *blocks = a.blocks;
  int64_t blocks_stride = a.blocks_stride;
  int kv_rows = a.kv_rows;
  asm volatile(""
               : XATTN_PIN_BEGINS(rows), XATTN_PIN_ROWSCHED(rows.first), "+s"(nrows), XATTN_PIN_VIEW(p.q),
                 XATTN_PIN_VIEW(p.k), XATTN_PIN_VIEW(p.v), "+s"(p.out), "+s"(p.o_sb), "+s"(p.o_sh), "+s"(p.o_st),
                 "+s"(p.part_o), "+s"(p.part_ml), "+s"(p.scale_log2), "+s"(p.D), "+s"(p.G), "+s"(p.T),
                 "+s"(blocks), "+s"(blocks_stride), "+s"(kv_rows));
  DecodeItem it;
  if (p.arrive_ctr == nullptr) {
    const int item = blockIdx.x;
    const RowSched rs = rows.find(a.rows, nrows, item);
    const int local = item - rs.item_begin, h = local / rs.nsplit;
    it = make_item(rs.batch, rs.count, rs.length, rs.nsplit, rs.ntiles, h, local - h * rs.nsplit, 0,
                   rs.rec_begin + (int64_t)local * (rs.count * p.G));
  } else {
    // In-launch merge (Hkv a multiple of 8): block b runs on XCD x = b % 8 and
    // takes, row after row, the items of the kv heads h = x (mod 8), so every
    // split of a (row, kv head) runs on one XCD and each XCD gets the same
    // work.  XCD x's list holds Hkv / 8 heads of each row: row r's part of it
    // starts at item_begin / 8.
    const int x = (int)(blockIdx.x % 8), slot = (int)(blockIdx.x / 8);
    const RowSched rs = rows.find(a.rows, nrows, 8 * slot);
    const int local = slot - rs.item_begin / 8, hh = local / rs.nsplit;
    const int h = 8 * hh + x;
    const int split = local - hh * rs.nsplit;
    it = make_item(rs.batch, rs.count, rs.length, rs.nsplit, rs.ntiles, h, split, rs.item_begin + h * rs.nsplit,
                   rs.rec_begin + (int64_t)(h * rs.nsplit + split) * (rs.count * p.G));
  }
  // The page is read while the loads issued for row it.b are in flight.
  const int raw_page = read_page(blocks, blocks_stride, it.b);
  process_item<DP, NC>(p, it, raw_page, kv_rows, smem);
}

// Graph-capture decode: the launch shape depends only on the tensor shapes.
// Lane r of every wave holds row r (B <= 64), takes its count and length from
// the device offsets and its splits from capture_splits; block b then runs the
// item, or exits past the last one.
template <int DP, int NC>
__global__ void __launch_bounds__(kItemThreads, 2) decode_capture_kernel(const CaptureArgs c) {
  constexpr int KT = DecodeShape<DP, NC>::KT;
  __shared__ __attribute__((aligned(16))) char smem[ItemShared<DP, NC>::BYTES];
  const int lane = threadIdx.x & 63;
  int count = 0, length = 1;
  if (lane < c.B) capture_row(c, lane, count, length);
  const int nsplit = capture_splits(c, lane, count, length);
  const int per = ((length + nsplit - 1) / nsplit + KT - 1) / KT * KT;  // equal splits, whole wave tiles
  const int item = blockIdx.x, mine = lane < c.B ? c.Hkv * nsplit : 0;
  const int end = wave_scan(mine), begin = end - mine;
  const unsigned long long before = __ballot(lane < c.B && begin <= item);
  const int r = __popcll(before) - 1;  // row 0 begins at 0
  if (item >= __builtin_amdgcn_readlane(end, r)) return;
  const int row_splits = __builtin_amdgcn_readlane(nsplit, r), local = item - __builtin_amdgcn_readlane(begin, r);
  const int h = local / row_splits, split = local - h * row_splits;
  DecodeItem it = make_item(r, __builtin_amdgcn_readlane(count, r), __builtin_amdgcn_readlane(length, r), row_splits,
                            __builtin_amdgcn_readlane(per, r), h, split, 0,
                            r * c.row_records + (int64_t)(h * c.splits_max + split) * (c.T * c.G));
  const DecodeParams p{c.q, c.k, c.v, c.out, c.o_sb, c.o_sh, c.o_st, c.part_o, c.part_ml, c.scale_log2, c.D, c.G, c.T};
  process_item<DP, NC>(p, it, read_page(c.blocks, c.blocks_stride, r), c.B, smem);
}

template <int DP>
static hipError_t launch_decode_capture_d(const CaptureArgs &c, int columns, int blocks, hipStream_t stream) {
  constexpr dim3 block(kItemThreads);
  if (columns == 1) hipLaunchKernelGGL((decode_capture_kernel<DP, 1>), dim3(blocks), block, 0, stream, c);
  else hipLaunchKernelGGL((decode_capture_kernel<DP, 2>), dim3(blocks), block, 0, stream, c);
  return hipGetLastError();
}

hipError_t launch_decode_capture(const CaptureArgs &c, int dp, int columns, int blocks, hipStream_t stream) {
  switch (dp) {
    case 64: return launch_decode_capture_d<64>(c, columns, blocks, stream);
    case 128: return launch_decode_capture_d<128>(c, columns, blocks, stream);
    default: return launch_decode_capture_d<256>(c, columns, blocks, stream);
  }
}

template <int DP>
static hipError_t launch_decode_d(const AttnArgs &a, int columns, int blocks, hipStream_t stream) {
  constexpr dim3 block(kItemThreads);
  if (columns == 1) hipLaunchKernelGGL((decode_kernel<DP, 1>), dim3(blocks), block, 0, stream, a);
  else hipLaunchKernelGGL((decode_kernel<DP, 2>), dim3(blocks), block, 0, stream, a);
  return hipGetLastError();
}

int decode_tokens_per_item(int dp) {
  switch (dp) {
    case 64: return 4 * DecodeShape<64, 1>::KT;
    case 128: return 4 * DecodeShape<128, 1>::KT;
    default: return 4 * DecodeShape<256, 1>::KT;
  }
}

// The XCC of each block of a small launch, for probe_xcd_dispatch.
constexpr int kXccProbeBlocks = 64;
__device__ uint32_t xcc_probe_ids[kXccProbeBlocks];

__global__ void __launch_bounds__(64) xcc_probe_kernel() {
  uint32_t xcc;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
  if (threadIdx.x == 0) xcc_probe_ids[blockIdx.x] = xcc & 15u;
}

hipError_t probe_xcd_dispatch(bool *round_robin, hipStream_t stream) {
  hipLaunchKernelGGL(xcc_probe_kernel, dim3(kXccProbeBlocks), dim3(64), 0, stream);
  hipError_t err = hipGetLastError();
  uint32_t ids[kXccProbeBlocks] = {};
  if (err == hipSuccess)
    err = hipMemcpyFromSymbolAsync(ids, HIP_SYMBOL(xcc_probe_ids), sizeof(ids), 0, hipMemcpyDeviceToHost, stream);
  if (err == hipSuccess) err = hipStreamSynchronize(stream);
  if (err != hipSuccess) return err;
  bool ok = true, distinct = false;
  for (int b = 8; b < kXccProbeBlocks; ++b) ok = ok && ids[b] == ids[b % 8];
  for (int b = 1; b < 8; ++b) distinct = distinct || ids[b] != ids[0];
  *round_robin = ok && distinct;
  return hipSuccess;
}

hipError_t launch_decode(const AttnArgs &a, int dp, int columns, int blocks, hipStream_t stream) {
  switch (dp) {
    case 64: return launch_decode_d<64>(a, columns, blocks, stream);
    case 128: return launch_decode_d<128>(a, columns, blocks, stream);
    default: return launch_decode_d<256>(a, columns, blocks, stream);
  }
}

}  // namespace xattn
