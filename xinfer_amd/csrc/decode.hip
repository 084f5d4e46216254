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
#include "decode_item.h"
#include "launch.h"

namespace xattn {


template <int DP, int NC>
__global__ void __launch_bounds__(kItemThreads, 2) decode_kernel(const AttnArgs a) {
  __shared__ __attribute__((aligned(16))) char smem[ItemShared<DP, NC>::BYTES];
  const DecodeLocals l(a);
  const DecodeParams &p = l.p;
  DecodeItem it;
  if (p.arrive_ctr == nullptr) {
    const int item = blockIdx.x;
    it = launch_item(a, l, item);
  } else {
    // In-launch merge (Hkv a multiple of 8): block b runs on XCD x = b % 8 and
    // takes, row after row, the items of the kv heads h = x (mod 8), so every
    // split of a (row, kv head) runs on one XCD and each XCD gets the same
    // work.  XCD x's list holds Hkv / 8 heads of each row: row r's part of it
    // starts at item_begin / 8.
    const int x = (int)(blockIdx.x % 8), slot = (int)(blockIdx.x / 8);
    const RowSched rs = l.rows.find(a.rows, l.nrows, 8 * slot);
    const int local = slot - rs.item_begin / 8, hh = local / rs.nsplit;
    const int h = 8 * hh + x;
    const int split = local - hh * rs.nsplit;
    it = make_item(rs.batch, rs.count, rs.length, rs.nsplit, rs.ntiles, h, split, rs.item_begin + h * rs.nsplit,
                   rs.rec_begin + (int64_t)(h * rs.nsplit + split) * (rs.count * p.G));
  }
  // The page is read while the loads issued for row it.b are in flight.
  const int raw_page = read_page(l.blocks, l.blocks_stride, it.b);
  process_item<DP, NC>(p, it, raw_page, l.kv_rows, smem, threadIdx.x);
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
  process_item<DP, NC>(p, it, read_page(c.blocks, c.blocks_stride, r), c.B, smem, threadIdx.x);
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
