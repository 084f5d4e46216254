// Merge of split-KV partial records into the bf16 output.
//
// When the keys of a group of query vectors are split over several work
// items, each item writes, per query vector, an fp32 record: unnormalised
// output o[D] and the pair (m, l) -- running max in log2 units and sum.  This
// kernel combines the records of one query vector:
//   M = max_s m_s,  w_s = exp2(m_s - M),  out = sum_s w_s o_s / sum_s w_s l_s
// Each thread folds its share of the splits with an online rescale (running
// max, sum and accumulator), in increasing split order; thread states are then
// folded in a fixed order, so the result is deterministic.  Splits that saw no
// visible key carry m = -inf and weight 0.  Running as its own launch, it reads
// the records after the producing kernel has completed, which orders them
// without any device-scope fence inside the attention kernels.
//
// With few splits per vector (prefill, short decode rows) a 256-thread block
// (512 for D = 256) holds VPB query vectors x FC feature lanes (4 features
// each), one thread owning a vector's 4 features across all splits.  With
// many splits (long
// decode rows) a block holds FS feature lanes of one vector and SG = THREADS /
// FS split lanes: all FC feature lanes up to kMergeSliceSplits splits, past
// that a slice of them, the FC / FS slices of a vector being separate blocks,
// so a very long row's records are read by many CUs at once; THREADS (256 or
// 512) is then chosen so that a lane loads at most one batch of 16 records.
//
// Blocks are dealt to the 8 XCDs in contiguous runs of work groups (block b
// runs group (b % 8) * (grid / 8) + b / 8), the order the prefill kernel
// gives its items, so the records a head's tiles wrote through one XCD's L2
// are mostly read back on that XCD, and a vector's slices share the (m, l)
// reads in one L2.
#include "kernel_args.h"
#include "launch.h"
#include "merge_common.h"

namespace xattn {

// Query vectors per prefill record block (the prefill kernel's query tile).
constexpr int kMergeTile = 128;

// LDS states of a block with SG > 1 split lanes over FS feature lanes.
template <int FS, int SG>
using MergeRed = MergeState[SG > 1 ? SG : 1][SG > 1 ? FS : 1];

// Feature lanes per block past kMergeSliceSplits splits: 64 features, 256
// contiguous bytes of each record.  Measured on MI355X: slicing takes a
// 16384-key D = 256 row's merge from 10.3 to 7.2 us at 256 splits and from
// 6.5 to 5.9 us at 128, and makes merges of 17 to 52 splits 0.2-0.8 us
// slower than one block per vector.
constexpr int kMergeSliceLanes = 16;
constexpr int kMergeSliceSplits = 64;

// Records a lane loads before it folds any (IN): few with one thread for all splits
// (registers for more waves), all of its splits up to kMergeSliceSplits
// (merge_inflight), else 16.  Sixteen for head dim 64 as well, whose block past
// kMergeSliceSplits differs from the one below in nothing else (one KV head's row of
// 60000 keys, 235 splits, decode and merge: 13.3 us with 4, 12.9 with 16; 40000 keys and
// 2 heads 13.2 / 12.95; 79 splits 15.9 both).
constexpr int merge_inflight(int split_lanes) {
  return split_lanes == 1 ? 4 : kMergeSliceSplits / split_lanes;
}
constexpr int kMergeSliceInflight = 16;

constexpr MergeState kMergeStart{-INFINITY, 0.0f, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};

// Folds records first, first + SG, ... below nsplit of one query vector into st over
// this thread's 4 features and writes them as bf16 at dst.  Record s: o at
// part_o + o_base + s * o_step, (m, l) at part_ml + 2 * (ml_base + s * ml_step).
// With SG > 1 split lanes per feature group every thread of the block must call it
// (it synchronises the block); `active` is false for threads past the vectors or
// features, and f is the thread's feature lane within the block's FS.  Every record
// of a batch is loaded before any is folded: a lane's splits take
// ceil(nsplit / (SG * INFLIGHT)) memory round trips.
template <int FS, int SG, int INFLIGHT>
__device__ __forceinline__ void fold_and_write(MergeRed<FS, SG> &red, const float *part_o, const float *part_ml,
                                               int64_t o_base, int64_t o_step, int64_t ml_base, int64_t ml_step,
                                               int nsplit, bool active, int sg, int f, uint16_t *dst, MergeState st,
                                               int first) {
  if (active) {
    for (int s0 = first; s0 < nsplit; s0 += INFLIGHT * SG) {
      u32x2 ml[INFLIGHT];
      f32x4 o[INFLIGHT];
#pragma unroll
      for (int u = 0; u < INFLIGHT; ++u)
        if (s0 + u * SG < nsplit) {  // a lane loads only its own splits' records
          const int64_t sp = s0 + u * SG;
          ml[u] = *as_global(reinterpret_cast<const u32x2 *>(part_ml + 2 * (ml_base + sp * ml_step)));
          o[u] = *as_global(reinterpret_cast<const f32x4 *>(part_o + o_base + sp * o_step));
        }
#pragma unroll
      for (int u = 0; u < INFLIGHT; ++u)
        if (s0 + u * SG < nsplit) fold(st, __uint_as_float(ml[u].x), __uint_as_float(ml[u].y), o[u]);
    }
  }
  if constexpr (SG > 1) {
    red[sg][f] = st;
    __syncthreads();
    if (sg != 0) return;
    // The states are read eight at a time before they are folded (in split
    // lane order), so the fold waits for one LDS round trip per eight lanes.
    for (int k0 = 1; k0 < SG; k0 += 8) {
      MergeState other[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + u < SG) other[u] = red[k0 + u][f];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + u < SG) fold(st, other[u].m, other[u].l, other[u].o);
    }
  }
  if (!active) return;
  const float inv = 1.0f / st.l;
  *as_global(reinterpret_cast<u32x2 *>(dst)) =
      u32x2{pack_bf16x2(st.o.x * inv, st.o.y * inv), pack_bf16x2(st.o.z * inv, st.o.w * inv)};
}

// Every argument of a block, loaded in one round trip (see XATTN_PIN_VIEW).
struct MergeLocals {
  RowLookup<MergeRow> rows;
  int total_items, nrows, D, G;
  uint16_t *out;
  int64_t o_sb, o_sh, o_st;
  const float *part_o, *part_ml;
  __device__ __forceinline__ explicit MergeLocals(const MergeArgs &a)
      : total_items(a.total_items), nrows(a.nrows), D(a.D), G(a.G), out(a.out), o_sb(a.o_sb), o_sh(a.o_sh),
        o_st(a.o_st), part_o(a.part_o), part_ml(a.part_ml) {
    rows.load(a.rows);
    asm volatile(""
                 : XATTN_PIN_BEGINS(rows), XATTN_PIN_MERGEROW(rows.first), "+s"(total_items), "+s"(nrows), "+s"(D),
                   "+s"(G), "+s"(out), "+s"(o_sb), "+s"(o_sh), "+s"(o_st), "+s"(part_o), "+s"(part_ml));
  }
};

// Block `block` of those that merge vectors first .. end - 1: shared by the launches
// with host-planned arguments (merge_kernel, merge_both_kernel) and the
// graph-capture launch that reads them from device memory (merge_dev_kernel).
template <int DP, int SG, int THREADS, int FS, int IN, bool DEV>
__device__ __forceinline__ void merge_body(const MergeArgs &a, const MergeLocals &l, unsigned block, int first, int end) {
  constexpr int FC = DP / 4;                         // feature lanes of a vector
  static_assert(SG == 1 ? FS == FC : FS * SG == THREADS, "block shape");
  constexpr int NS = FC / FS;                        // feature slices per vector (SG > 1)
  constexpr int VPB = SG > 1 ? 1 : THREADS / FC;     // query vectors per block
  __shared__ MergeRed<FS, SG> red;

  // Few splits: vectors vary fastest across a block's threads (the prefill
  // record layout keeps a tile's vectors contiguous per feature group).
  // Many splits: the slice's feature lanes vary fastest.
  const int tid = threadIdx.x;
  const int fl = SG > 1 ? tid % FS : tid / VPB, sg = SG > 1 ? tid / FS : 0;
  const int vl = VPB == 1 ? 0 : tid % VPB;
  // Work groups: VPB vectors (few splits) or one slice of one vector.  The
  // blocks are the groups rounded up to a multiple of 8 (launch_merge_d).
  const int groups = SG > 1 ? (end - first) * NS : (end - first + VPB - 1) / VPB;
  // A grid sized for more groups (device-planned launches) leaves surplus blocks.
  if constexpr (DEV) {
    if ((int)(block / 8) >= (groups + 7) / 8) return;
  }
  const int group = (int)(block % 8) * ((groups + 7) / 8) + (int)(block / 8);
  const int vec = first + (SG > 1 ? group / NS : group * VPB + vl);
  const int f = SG > 1 ? (group - (vec - first) * NS) * FS + fl : fl;  // feature lane of the vector
  const bool vvalid = vec < end;
  const MergeRow mr = l.rows.template find<(SG > 1)>(a.rows, l.nrows, vvalid ? vec : first);
  const int local = vec - mr.item_begin;
  const int D = l.D, G = l.G, qrows = mr.count * G;
  const int h = local / qrows, j = local - h * qrows;
  const int d = f * 4;
  // Record s of this vector: o at part_o + o_base + s * o_step, (m, l) at
  // part_ml + 2 * (ml_base + s * ml_step).
  int64_t o_base, o_step, ml_base, ml_step;
  if (mr.tiles == 0) {
    ml_base = mr.rec_begin + (int64_t)h * mr.nsplit * qrows + j;
    ml_step = qrows;
    o_base = ml_base * D + d;
    o_step = ml_step * D;
  } else {
    const int tile = j / kMergeTile, jr = j - tile * kMergeTile;
    const int64_t blk = mr.rec_begin + ((int64_t)h * mr.nsplit * mr.tiles + tile) * kMergeTile;
    ml_base = blk + jr;
    ml_step = (int64_t)mr.tiles * kMergeTile;
    o_base = blk * D + (f * kMergeTile + jr) * 4;
    o_step = ml_step * D;
  }

  const int g = j % G, i = j / G;
  fold_and_write<FS, SG, IN>(red, l.part_o, l.part_ml, o_base, o_step, ml_base, ml_step, mr.nsplit, vvalid && d < D,
                             sg, fl,
                             l.out + mr.batch * l.o_sb + (int64_t)(h * G + g) * l.o_sh + (int64_t)i * l.o_st + d,
                             kMergeStart, sg);
}

// Threads of a block with one thread for all splits: 8 vectors per block for
// D = 256, so that a wave's load reads whole 128-byte lines of the prefill record
// layout (cfg5's merge 3 us faster than with 4 vectors and half lines; same
// outputs).
template <int DP>
constexpr int kMergeSerialThreads = DP == 256 ? 512 : 256;

template <int DP, int SG, int THREADS, int FS, int IN>
__global__ void __launch_bounds__(THREADS) merge_kernel(const MergeArgs a) {
  const MergeLocals l(a);
  merge_body<DP, SG, THREADS, FS, IN, false>(a, l, blockIdx.x, 0, l.total_items);
}

template <int DP, int SG, int THREADS, int FS, int IN>
__global__ void __launch_bounds__(THREADS) merge_dev_kernel(const MergeArgs *__restrict__ a) {
  const MergeLocals l(*a);
  merge_body<DP, SG, THREADS, FS, IN, true>(*a, l, blockIdx.x, 0, l.total_items);
}

// The merge's launch: host arguments `a`, or (DEV) the arguments at `dev`;
// the grid covers `vectors` query vectors.
template <int DP, int SG, int THREADS, int FS, int IN, bool DEV>
static void launch_merge_kernel(dim3 grid, const MergeArgs &a, const MergeArgs *dev, hipStream_t stream) {
  if constexpr (DEV)
    hipLaunchKernelGGL((merge_dev_kernel<DP, SG, THREADS, FS, IN>), grid, dim3(THREADS), 0, stream, dev);
  else
    hipLaunchKernelGGL((merge_kernel<DP, SG, THREADS, FS, IN>), grid, dim3(THREADS), 0, stream, a);
}

template <int DP, bool DEV>
static hipError_t launch_merge_d(const MergeArgs &a, const MergeArgs *dev, int max_splits, int64_t vectors,
                                 hipStream_t stream) {
  constexpr int FC = DP / 4;
  // Grids are rounded up to a multiple of the 8 XCDs; surplus groups exit.
  if (max_splits <= kMergeSerialSplits) {
    constexpr int THREADS = kMergeSerialThreads<DP>;
    constexpr int VPB = THREADS / FC;
    launch_merge_kernel<DP, 1, THREADS, FC, merge_inflight(1), DEV>(dim3(((vectors + VPB - 1) / VPB + 7) / 8 * 8), a, dev, stream);
  } else if (max_splits <= kMergeSliceSplits) {
    // One block per vector: a lane loads its splits in one batch.
    launch_merge_kernel<DP, 256 / FC, 256, FC, merge_inflight(256 / FC), DEV>(dim3((vectors + 7) / 8 * 8), a, dev, stream);
  } else {
    // One block per (vector, slice of FS feature lanes).
    constexpr int FS = FC < kMergeSliceLanes ? FC : kMergeSliceLanes;
    const dim3 grid((vectors * (FC / FS) + 7) / 8 * 8);
    if (max_splits <= kMergeSliceInflight * (256 / FS))
      launch_merge_kernel<DP, 256 / FS, 256, FS, kMergeSliceInflight, DEV>(grid, a, dev, stream);
    else
      launch_merge_kernel<DP, 512 / FS, 512, FS, kMergeSliceInflight, DEV>(grid, a, dev, stream);
  }
  return hipGetLastError();
}

// Graph-capture merge: one block per query vector of the capacity layout
// (row, kv head, vector j < T * G), with split lanes over the splits.  Vectors
// past the row's queries and rows of one split (written by the decode kernel
// directly) have nothing to merge.  A block waits for the device's lengths before
// it knows its splits; the records' places do not depend on them, so in small
// launches a lane's first records are loaded beside the lengths, whether its row
// has them or not (the workspace holds them all): eight layers' captured steps of
// 8 rows, 128 vectors, 156.4 -> 148.6 us.  Larger launches, whose records past the
// splits would be a load worth saving (2 KB a split lane; 512 vectors: 8 MB at
// most), wait.
constexpr int kMergeAheadVectors = 512;

// AHEAD: records of a lane loaded early, as many as a row of the most splits has
// (1 to 4; loads past them, all of one record, took a captured step of 16 rows at head
// dim 64 from 69.2 to 70.8 us).
template <int DP, int AHEAD>
__global__ void __launch_bounds__(256) merge_capture_kernel(const CaptureArgs c) {
  constexpr int FC = DP / 4, SG = 256 / FC;
  __shared__ MergeRed<FC, SG> red;
  const int tid = threadIdx.x, lane = tid & 63, f = tid % FC, sg = tid / FC, d = f * 4;
  const int r = (int)blockIdx.y, qv_max = c.T * c.G, h = (int)blockIdx.x / qv_max, j = (int)blockIdx.x - h * qv_max;
  int own_count, own_length;
  capture_row_uniform(c, r, own_count, own_length);
  // Nothing to merge past the row's queries, and in a row that one least item holds: such
  // blocks leave on scalar loads of their own row, before the splits of all rows are
  // worked out (one row of 30 keys: the launch 3.04 us without, 1.72 with).
  if (j >= own_count * c.G || own_length <= c.pass_min * c.pass_keys) return;  // block-uniform
  const int64_t ml_base = r * c.row_records + (int64_t)h * c.splits_max * qv_max + j, ml_step = qv_max;
  const int64_t o_base = ml_base * c.D + d, o_step = ml_step * c.D;
  u32x2 ml[AHEAD > 0 ? AHEAD : 1];
  f32x4 o[AHEAD > 0 ? AHEAD : 1];
  // Lanes past the features or the splits load others' records (a branch around a
  // load would wait for it).
  const int64_t o_first = ml_base * c.D + min(d, c.D - 4);
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) {
    const int64_t sp = min(sg + u * SG, c.splits_max - 1);
    ml[u] = *as_global(reinterpret_cast<const u32x2 *>(c.part_ml + 2 * (ml_base + sp * ml_step)));
    o[u] = *as_global(reinterpret_cast<const f32x4 *>(c.part_o + o_first + sp * o_step));
  }
  int count = 0, length = 1;
  if (lane < c.B) capture_row(c, lane, count, length);
  const int nsplit = __builtin_amdgcn_readlane(capture_splits(c, lane, count, length), r);
  if (nsplit <= 1) return;
  MergeState st = kMergeStart;
  if (d < c.D) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (sg + u * SG < nsplit) fold(st, __uint_as_float(ml[u].x), __uint_as_float(ml[u].y), o[u]);
  }
  const int g = j % c.G, i = j / c.G;
  fold_and_write<FC, SG, 16>(red, c.part_o, c.part_ml, o_base, o_step, ml_base, ml_step, nsplit, d < c.D, sg, f,
                             c.out + r * c.o_sb + (int64_t)(h * c.G + g) * c.o_sh + (int64_t)i * c.o_st + d, st,
                             sg + AHEAD * SG);
}

template <int DP>
static void launch_merge_capture_d(const CaptureArgs &c, hipStream_t stream) {
  const dim3 grid(c.Hkv * c.T * c.G, c.B), block(256);
  constexpr int SG = 256 / (DP / 4);
  if ((int64_t)grid.x * grid.y > kMergeAheadVectors)
    hipLaunchKernelGGL((merge_capture_kernel<DP, 0>), grid, block, 0, stream, c);
  else if (c.splits_max <= SG)
    hipLaunchKernelGGL((merge_capture_kernel<DP, 1>), grid, block, 0, stream, c);
  else if (c.splits_max <= 2 * SG)
    hipLaunchKernelGGL((merge_capture_kernel<DP, 2>), grid, block, 0, stream, c);
  else
    hipLaunchKernelGGL((merge_capture_kernel<DP, 4>), grid, block, 0, stream, c);
}

hipError_t launch_merge_capture(const CaptureArgs &c, int dp, hipStream_t stream) {
  switch (dp) {
    case 64: launch_merge_capture_d<64>(c, stream); break;
    case 128: launch_merge_capture_d<128>(c, stream); break;
    default: launch_merge_capture_d<256>(c, stream); break;
  }
  return hipGetLastError();
}

hipError_t launch_merge(const MergeArgs &a, int dp, int max_splits, hipStream_t stream) {
  switch (dp) {
    case 64: return launch_merge_d<64, false>(a, nullptr, max_splits, a.total_items, stream);
    case 128: return launch_merge_d<128, false>(a, nullptr, max_splits, a.total_items, stream);
    default: return launch_merge_d<256, false>(a, nullptr, max_splits, a.total_items, stream);
  }
}

// The rows of many splits (decode) and those of few (prefill) of a mixed batch in
// one launch: the first round8(lane_items) blocks take one vector each, the others
// several.  (A mixed step of 7 decode rows and a 384-token prefill row, D = 128: one launch
// of 5.7 us in place of two of 4.7 and 4.5, the step 45.6 -> 42.9 us.)
template <int DP>
__global__ void __launch_bounds__(kMergeSerialThreads<DP>) merge_both_kernel(const MergeArgs a) {
  constexpr int THREADS = kMergeSerialThreads<DP>, FC = DP / 4;
  int lane_items = a.lane_items;
  const MergeLocals l(a);
  asm volatile("" : "+s"(lane_items));
  const unsigned lane_blocks = (unsigned)(lane_items + 7) / 8 * 8, block = blockIdx.x;
  if (block < lane_blocks)
    merge_body<DP, THREADS / FC, THREADS, FC, merge_inflight(THREADS / FC), false>(a, l, block, 0, lane_items);
  else
    merge_body<DP, 1, THREADS, FC, merge_inflight(1), false>(a, l, block - lane_blocks, lane_items, l.total_items);
}

template <int DP>
static hipError_t launch_merge_both_d(const MergeArgs &a, hipStream_t stream) {
  constexpr int THREADS = kMergeSerialThreads<DP>, VPB = THREADS / (DP / 4);
  const int few = (a.total_items - a.lane_items + VPB - 1) / VPB;
  hipLaunchKernelGGL(merge_both_kernel<DP>, dim3((a.lane_items + 7) / 8 * 8 + (few + 7) / 8 * 8), dim3(THREADS), 0,
                     stream, a);
  return hipGetLastError();
}

hipError_t launch_merge_both(const MergeArgs &lanes, const MergeArgs &few, int dp, int lane_splits, int few_splits,
                             hipStream_t stream) {
  if (few_splits > kMergeSerialSplits || lane_splits > kMergeSliceSplits) {
    const hipError_t rc = launch_merge(lanes, dp, lane_splits, stream);
    return rc != hipSuccess ? rc : launch_merge(few, dp, few_splits, stream);
  }
  MergeArgs both = lanes;
  both.lane_items = lanes.total_items;
  both.total_items += few.total_items;
  for (int r = 0; r < few.nrows; ++r) {
    MergeRow &row = both.rows[both.nrows++];  // rows of one group: at most kMaxRows
    row = few.rows[r];
    row.item_begin += lanes.total_items;
  }
  if (lane_splits <= kMergeSerialSplits) return launch_merge(both, dp, kMergeSerialSplits, stream);
  switch (dp) {
    case 64: return launch_merge_both_d<64>(both, stream);
    case 128: return launch_merge_both_d<128>(both, stream);
    default: return launch_merge_both_d<256>(both, stream);
  }
}

hipError_t launch_merge_dev(const MergeArgs *a, int dp, int max_splits, int64_t max_vectors, hipStream_t stream) {
  const MergeArgs none{};
  switch (dp) {
    case 64: return launch_merge_d<64, true>(none, a, max_splits, max_vectors, stream);
    case 128: return launch_merge_d<128, true>(none, a, max_splits, max_vectors, stream);
    default: return launch_merge_d<256, true>(none, a, max_splits, max_vectors, stream);
  }
}

}  // namespace xattn
