// C ABI of libxinfer_attention_ops.so: validation, work planning and launches.
//
// The planner turns host-side lengths into a static schedule carried in the
// kernel arguments (kernel_args.h): rows with at most 32 query vectors per KV
// head go to the decode kernel, the others to the MFMA prefill kernel; rows
// whose keys are split get fp32 partial records in the caller's workspace,
// combined by a merge launch after the attention kernels or, for decode rows
// whose launch allows it, by the last split of each (row, kv head) inside the
// decode launch (decode_item.h: merge_in_launch), which folds in the merge
// launch's order and arithmetic.  The schedule is a function of the shapes and
// lengths only, never of tensor data, so results are deterministic and each
// row is isolated from the others' contents.
#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <functional>
#include <mutex>
#include <numeric>
#include <vector>

#include "xinfer_attention.h"
#include "kernel_args.h"
#include "launch.h"

namespace xattn {
namespace {

constexpr int kCaptureDecodeMaxVectors = 8;  // graph capture: G * T at or below this takes the decode kernel
constexpr int kPrefillTileQ = 128;         // query vectors per prefill work item
constexpr int64_t kPrefillMinSplitKeys = 512;

int padded_dim(int64_t d) { return d <= 64 ? 64 : (d <= 128 ? 128 : 256); }
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct Geometry {
  int64_t B, Hq, Hkv, T, D, C;
};

bool attention_layout_ok(const xinfer_view4 &t) {
  if (t.data == nullptr || (reinterpret_cast<uintptr_t>(t.data) & 15u) != 0) return false;
  if (t.size[3] > 1 && t.stride[3] != 1) return false;
  for (int i = 0; i < 3; ++i)
    if (t.size[i] > 1 && (t.stride[i] % 8) != 0) return false;
  // One (row, head) slice is addressed with 32-bit byte offsets.
  if ((t.size[2] + 1) * t.stride[2] * 2 >= (int64_t(1) << 31)) return false;
  return true;
}

// The prefill kernel addresses one batch row of Q ([Hq, T, D]) with 32-bit
// byte offsets from the row's first head.
bool query_layout_ok(const xinfer_view4 &q) {
  return (q.size[1] * q.stride[1] + q.size[2] * q.stride[2]) * 2 < (int64_t(1) << 31);
}

View view_of(const xinfer_view4 &t) {
  return View{static_cast<const uint16_t *>(t.data), t.stride[0], t.stride[1], t.stride[2]};
}

int check_heads_and_dim(const Geometry &g) {
  if (g.Hq <= 0 || g.Hkv <= 0 || g.Hq % g.Hkv != 0) return XINFER_ERR_HEADS;
  if (g.D < 8 || g.D > 256 || g.D % 8 != 0) return XINFER_ERR_HEAD_DIM;
  return XINFER_OK;
}

struct Group {
  int row0 = 0, nrows = 0;
  AttnArgs dec{};
  int dec_items = 0, dec_columns = 1, dec_max_splits = 1;
  AttnArgs pre{};
  int pre_items = 0;
  // Merge launches of the decode rows and of the prefill rows: their layouts
  // differ (a thread folds a few splits, a row of lanes many).
  MergeArgs dec_merge{}, pre_merge{};
  int dec_merge_items = 0, pre_merge_items = 0, pre_max_splits = 1;
  // The decode launch may merge its split rows itself (merge_in_launch_pays).
  bool dec_fusable = false;
  bool both = false;  // decode and prefill rows in one launch (one_launch_pays)
};

struct Plan {
  std::vector<Group> groups;
  int64_t records = 0;
  int64_t D = 0;
  // Arrival counters of the decode in-launch merge: one per decode item of
  // the largest fusable group (the groups' launches run one after another and
  // leave every counter at zero).
  int64_t counters = 0;
  size_t part_ml_offset() const { return (size_t)((records * D * 4 + 255) / 256 * 256); }
  size_t counters_offset() const { return (part_ml_offset() + (size_t)records * 8 + 255) / 256 * 256; }
  size_t bytes() const { return records ? counters_offset() + (size_t)counters * 8 : 0; }
};

// Measured prefill costs on one MI355X CU, for the planner's choice of split
// size: one 64-key tile of a 128-vector item (D <= 128: 8 waves, two per
// SIMD; D = 256: 4 waves), and an item's fixed prologue, fold and epilogue.
double prefill_tile_us(int dp) { return dp <= 64 ? 0.9 : (dp <= 128 ? 1.15 : 1.9); }
constexpr double kPrefillItemUs = 4.5;
// Merge launch: fixed cost, and the record read at about 5 TB/s.
constexpr double kMergeLaunchUs = 5.0;
constexpr double kRecordBytesPerUs = 5.0e6;
constexpr int kCusPerXcd = 32;
// Prefill items that leave a quarter of the CUs free.
constexpr int kPrefillFreeItems = 8 * kCusPerXcd * 3 / 4;

// Decode merge choice.  The merge launch costs an empty kernel's time and the cold
// round trips of its records, four splits at a time up to kMergeSerialSplits, and of
// the records themselves, written and read.
constexpr double kDecodeRecordBytesPerUs = 3.0e6;
double merge_launch_us(int64_t splits, double record_bytes) {
  return (splits <= kMergeSerialSplits ? 2.0 + (double)ceil_div(splits, 4) : 4.5) + record_bytes / kDecodeRecordBytesPerUs;
}
// The in-launch merge makes every block wait, before it retires, for its record
// stores and one counter round trip, and leaves the last split of each (row, kv head)
// a fold at the tail, in rounds of the 256 quads of features its threads take at a
// time.  So it does not pay for many vectors of many splits.  Measured on MI355X, one
// row, 8 KV heads, D = 128, in the launch / by the merge launch: 8 splits of 8, 16, 32
// vectors 8.8 / 10.5, 9.2 / 9.8, 12.7 / 11.4 us, 3 splits of 32 10.2 / 9.5; D = 256: 5 splits of
// 16 10.8 / 10.4, 6 of 32 16.2 / 13.2; 16 rows, 2 splits of 32 vectors, D = 256: 22.5 / 25.3.
double merge_in_launch_us(int64_t splits, int64_t vectors, int dp) {
  return 1.5 + (double)ceil_div(vectors * (dp / 4), 64 * kDecodeWaves) * (0.05 + 0.12 * (double)splits);
}
// Resident decode blocks: 256 CUs x 2 (66 to 80 KB of each CU's 160 KB of LDS per
// block).  A launch of more would make its blocks wait more than once.
constexpr int64_t kDecodeResidentBlocks = 2 * kDecodeCus;

// Whether a decode launch merges its own split rows.  Only with Hkv a multiple of 8 (the
// kernel gives XCD x the kv heads h = x mod 8 of every row) and at most
// kMergeSerialSplits splits a row, the merge layout the in-launch fold reproduces.
bool merge_in_launch_pays(int64_t Hkv, int64_t items, int64_t splits, int64_t vectors, double record_bytes, int dp) {
  return Hkv % 8 == 0 && items <= kDecodeResidentBlocks && splits > 1 && splits <= kMergeSerialSplits &&
         merge_in_launch_us(splits, vectors, dp) < merge_launch_us(splits, record_bytes);
}

// Modelled time of a decode launch and its merge, without what no choice of items
// changes.  A CU alone with an item takes kDecodePassUs for a pass (64 KB at 45 GB/s),
// two items on it take as long as both in turn; HBM serves all CUs at
// kDecodeSharePassUs a pass each.  Past the resident blocks, CUs take items as they come
// free: most of a longest item is left at the end, and every item's start counts.
constexpr double kDecodePassUs = 1.5, kDecodeSharePassUs = 1.8;
struct DecodeRow {
  uint32_t passes, vectors;
};
struct DecodeLoad {
  std::array<DecodeRow, kMaxRows> rows;  // in launch order
  int n = 0;
  int64_t passes = 0;  // of all (row, kv head) pairs
  int64_t longest = 1, widest = 0;  // row's passes, row's vectors
};
// ceil(passes / m) by a multiplication: 2^40 / m rounded up is exact for passes and m
// below 2^19 (33 million keys), where it is used; a plan of 32 rows takes some 800 of them.
class SplitCount {
 public:
  SplitCount(int64_t m, int64_t longest)
      : m_((uint32_t)m), inverse_(longest < (1 << 19) && m < (1 << 19) ? ((uint64_t(1) << 40) - 1) / m_ + 1 : 0) {}
  uint32_t operator()(uint32_t passes) const {
    const uint32_t n = passes + m_ - 1;
    return inverse_ ? (uint32_t)((n * inverse_) >> 40) : n / m_;
  }

 private:
  uint32_t m_;
  uint64_t inverse_;
};

double decode_us(const Geometry &g, const DecodeLoad &load, int dp, int64_t m) {
  const SplitCount split_count(m, load.longest);
  int64_t items = 0, splits = 1, vectors = 0, records = 0, longest = 0, paired = 0;
  for (int r = 0; r < load.n; ++r) {
    const uint32_t passes = load.rows[r].passes, nsplit = split_count(passes);
    const int64_t size = nsplit == 1 ? passes : (passes + nsplit - 1) / nsplit;
    longest = std::max(longest, size);
    const int64_t next = items + g.Hkv * nsplit;
    if (items <= kDecodeCus && kDecodeCus < next) paired = size;  // shares the CU of the first item
    items = next;
    if (nsplit > 1) {
      splits = std::max<int64_t>(splits, nsplit);
      vectors = std::max<int64_t>(vectors, load.rows[r].vectors);
      records += g.Hkv * nsplit * load.rows[r].vectors;
    }
  }
  // One item a CU leaves HBM a little idle while it starts and ends (decode of 8 rows,
  // 126 MB: 27.1 us with 240 items, 26.8 with 512).
  const double share =
      (items <= kDecodeCus ? 1.02 : 1.0) * kDecodeSharePassUs * (double)load.passes / kDecodeCus;
  double us = items <= kDecodeResidentBlocks
                  ? std::max(kDecodePassUs * (double)(longest + paired), share)
                  : std::max(kDecodePassUs * (double)longest, share) + 0.75 * kDecodePassUs * (double)longest +
                        0.75 * (double)items / kDecodeResidentBlocks;
  if (splits > 1) {
    const double bytes = (double)(records * (4 * g.D + 8));
    us += merge_in_launch_pays(g.Hkv, items, splits, vectors, bytes, dp) ? merge_in_launch_us(splits, vectors, dp)
                                                                        : merge_launch_us(splits, bytes);
  }
  return us;
}

// Passes of a block's four waves (decode_tokens_per_item) per decode item.
//
// By decode_us, launches of at most one one-pass item per CU take items of one pass or of
// kDecodeItemRounds.  Others, and those with rows of more than kExactVectors query vectors
// (whose records are large), choose among the fewest passes that leave one item per
// CU, two, four or eight, those that bring every row within the merge in the
// launch, and no split.  Measured on MI355X against all numbers of passes, 287
// launches of 1-64 rows (uniform and log-uniform lengths up to 16384 keys; 16 / 8 and 32 / 8
// heads of 128, 8 / 8 of 64, 16 / 4 of 256): 2% above the best on average; 7.5% with
// one item per CU or two by evenness, four where neither was even, whose merge launch
// that rule did not count (32 rows of up to 1000 keys, D = 128: 20.6 us, now 15.5; 32
// of up to 700, 928 one-pass items, 19.5, now 14.1).
//
// Beside prefill rows, where the decode items are merged by a launch, the evenness
// rule (kernel_args.h: kDecodeCus) stays: 7 decode rows and 384 tokens, D = 128, in one
// launch 21.0 us with it, 24.1 with the few items that decode_us prefers.
int64_t choose_decode_passes(const Geometry &g, const DecodeLoad &load, int dp, bool prefill) {
  const int64_t longest = load.longest, pairs = g.Hkv * load.n;
  // The fewest passes per item, from `low`, that leave at most `limit` items.
  auto least = [&](int64_t limit, int64_t low) {
    auto fits = [&](int64_t m) {  // items only fall as m grows
      const SplitCount split_count(m, longest);
      int64_t count = 0;
      for (int r = 0; r < load.n; ++r) count += split_count(load.rows[r].passes);
      return g.Hkv * count <= std::max(limit, pairs);
    };
    low = std::max(low, ceil_div(load.passes, limit));
    int64_t high = low;
    for (int64_t step = 1; high < longest && !fits(high); step *= 2) {
      low = high + 1;
      high = std::min(longest, high + step);
    }
    while (low < high) {
      const int64_t mid = (low + high) / 2;
      if (fits(mid)) high = mid;
      else low = mid + 1;
    }
    return low;
  };
  if (prefill) {
    auto even = [&](int64_t m, int64_t limit) { return m * limit * kDecodeEvenDen <= load.passes * kDecodeEvenNum; };
    const int64_t m2 = least(2 * kDecodeCus, 1), m1 = least(kDecodeCus, m2);
    if (!even(m1, kDecodeCus) && !even(m2, 2 * kDecodeCus)) return least(4 * kDecodeCus, 1);
    return 2 * m2 < m1 ? m2 : m1;
  }
  int64_t best = 1;
  double best_us = INFINITY;
  auto consider = [&](int64_t m) {
    const double us = decode_us(g, load, dp, m);
    if (us < best_us) {
      best_us = us;
      best = m;
    }
  };
  if (load.passes <= kDecodeCus && load.widest <= kExactVectors) {
    consider(1);
    consider(kDecodeItemRounds);
    return best;
  }
  int64_t m = 0;
  for (int64_t limit = 8 * kDecodeCus; limit >= kDecodeCus; limit /= 2) {
    const int64_t next = std::min(least(limit, std::max<int64_t>(m, 1)), longest);
    if (next > m) consider(next);
    m = next;
  }
  if (g.Hkv % 8 == 0) consider(ceil_div(longest, kMergeSerialSplits));
  if (m < longest) consider(longest);
  return best;
}

// 64-key tiles of prefill item (split, query tile) of row rs: the key range
// of prefill.hip's split_range for that tile.
int64_t prefill_item_tiles(const RowSched &rs, int G, int split, int tile) {
  const int64_t qrows = (int64_t)rs.count * G, p0 = rs.length - rs.count;
  const int64_t j_last = std::min<int64_t>((int64_t)(tile + 1) * kPrefillTileQ, qrows) - 1;
  const int64_t kend = p0 + j_last / G + 1;
  const int64_t per = ceil_div(ceil_div(kend, rs.nsplit), 64) * 64;
  const int64_t ks0 = std::min(kend, split * per), ks1 = std::min(kend, ks0 + per);
  return ceil_div(ks1 - ks0, 64);
}

// Work of every prefill item of rows[0, nrows), in item order (row, kv head,
// split, query tile), in microseconds.
std::vector<double> prefill_item_work(const RowSched *rows, int nrows, int64_t Hkv, int G, int dp) {
  std::vector<double> work;
  for (int r = 0; r < nrows; ++r) {
    const RowSched &rs = rows[r];
    for (int64_t h = 0; h < Hkv; ++h)
      for (int split = 0; split < rs.nsplit; ++split)
        for (int tile = 0; tile < rs.ntiles; ++tile)
          work.push_back(prefill_item_tiles(rs, G, split, tile) * prefill_tile_us(dp) + kPrefillItemUs);
  }
  return work;
}

// Cut items (in order) into 8 contiguous runs of about equal work, one per
// XCD: on a ragged batch an equal number of items per XCD can leave the XCDs
// that hold the long rows with most of the work.  begin[0..8].
void xcd_runs(const std::vector<double> &work, int32_t *begin) {
  double total = 0;
  for (double w : work) total += w;
  begin[0] = 0;
  size_t i = 0;
  double done = 0;  // work of items [0, i)
  for (int x = 1; x < 8; ++x) {
    const double target = total * x / 8;
    // Take item i while that lands closer to the target than stopping before it.
    while (i < work.size() && (done + work[i]) - target < target - done) done += work[i++];
    begin[x] = (int32_t)i;
  }
  begin[8] = (int32_t)work.size();
}

// Time of the prefill launch when the items run as the hardware dispatches
// them: the blocks of each XCD, in order, to whichever of its CUs is free.
// The CUs' finishing times are kept in a min-heap (which of several tied CUs
// takes an item does not change the times that follow).
double simulated_prefill_us(const std::vector<double> &work) {
  int32_t begin[9];
  xcd_runs(work, begin);
  double span = 0;
  for (int x = 0; x < 8; ++x) {
    double free_at[kCusPerXcd] = {};  // all equal: already a heap
    for (int32_t i = begin[x]; i < begin[x + 1]; ++i) {
      std::pop_heap(free_at, free_at + kCusPerXcd, std::greater<double>());
      free_at[kCusPerXcd - 1] += work[(size_t)i];
      std::push_heap(free_at, free_at + kCusPerXcd, std::greater<double>());
    }
    span = std::max(span, *std::max_element(free_at, free_at + kCusPerXcd));
  }
  return span;
}

// Split count of a prefill row for keys-per-split `split_keys`.
int32_t prefill_splits(int64_t len, int64_t split_keys) {
  return (int32_t)std::max<int64_t>(1, ceil_div(len, split_keys));
}

// Keys per prefill split for the call: the split size, from about 256 to
// 2048 items' worth (at least kPrefillMinSplitKeys keys), whose launch,
// simulated as dispatched, plus its merge launch and the records' two trips
// through HBM, is fastest.  More, smaller items even out ragged rows; they
// cost per-item overhead, records and merge traffic.  The simulated span
// moves in jumps, when some row's split count changes, so the candidates are
// those change points: for each row and split count n, the smallest multiple
// of 64 keys that cuts the row into n splits (on the ragged D = 256 batch of
// 2235 tokens, cfg5, 3200-key splits measured 10 us faster than 2752-key
// ones, and 3264-key splits, one split fewer on one row, 4 us slower than
// 3200).  Candidates are simulated in increasing order of a lower bound on
// their time (total work over 256 CUs, or the longest item, plus the
// records), until that bound passes the best time found.
int64_t choose_split_keys(const Geometry &g, const std::vector<int32_t> &counts,
                          const std::vector<int32_t> &lengths, int G, int dp, int64_t decode_vectors) {
  int64_t prefill_keys = 0;
  std::vector<RowSched> rows;
  for (int64_t r = 0; r < g.B; ++r) {
    const int64_t qv = (int64_t)counts[r] * G;
    if (qv <= decode_vectors) continue;
    prefill_keys += g.Hkv * ceil_div(qv, kPrefillTileQ) * lengths[r];
    RowSched rs{};
    rs.count = counts[r];
    rs.length = lengths[r];
    rs.ntiles = (int32_t)ceil_div(qv, kPrefillTileQ);
    rows.push_back(rs);
  }
  if (rows.empty()) return kPrefillMinSplitKeys;
  auto keys_for = [&](int64_t target) {
    return std::max(kPrefillMinSplitKeys, ceil_div(ceil_div(prefill_keys, target), 64) * 64);
  };
  const int64_t lo = keys_for(2048), hi = keys_for(256);
  std::vector<int64_t> keys = {lo, hi};
  for (const RowSched &rs : rows)
    for (int64_t n = ceil_div(rs.length, hi); n <= ceil_div(rs.length, lo); ++n) {
      const int64_t k = std::max(kPrefillMinSplitKeys, ceil_div(ceil_div(rs.length, n), 64) * 64);
      if (k >= lo && k <= hi) keys.push_back(k);
    }
  std::sort(keys.begin(), keys.end());
  keys.erase(std::unique(keys.begin(), keys.end()), keys.end());
  // Per row and split count: the work of one kv head's items and its longest
  // item (every kv head has the same items).
  struct RowWork {
    int32_t nsplit;
    double total, longest;
    std::vector<double> items;  // one kv head's items, in order (split, tile)
  };
  std::vector<std::vector<RowWork>> row_work(rows.size());
  auto work_of = [&](size_t r, int32_t nsplit) -> const RowWork & {
    for (const RowWork &w : row_work[r])
      if (w.nsplit == nsplit) return w;
    RowSched rs = rows[r];
    rs.nsplit = nsplit;
    RowWork w{nsplit, 0.0, 0.0, {}};
    w.items.reserve((size_t)nsplit * rs.ntiles);
    for (int split = 0; split < nsplit; ++split)
      for (int tile = 0; tile < rs.ntiles; ++tile) {
        const double us = prefill_item_tiles(rs, G, split, tile) * prefill_tile_us(dp) + kPrefillItemUs;
        w.total += us;
        w.longest = std::max(w.longest, us);
        w.items.push_back(us);
      }
    row_work[r].push_back(w);
    return row_work[r].back();
  };
  struct Candidate {
    double bound, records_us;
    int64_t split_keys;
  };
  std::vector<Candidate> cands;
  cands.reserve(keys.size());
  for (const int64_t split_keys : keys) {
    int64_t records = 0;
    double total = 0, longest = 0;
    for (size_t r = 0; r < rows.size(); ++r) {
      const int32_t nsplit = prefill_splits(rows[r].length, split_keys);
      if (nsplit > 1) records += g.Hkv * nsplit * rows[r].ntiles * kPrefillTileQ;
      const RowWork &w = work_of(r, nsplit);
      total += g.Hkv * w.total;
      longest = std::max(longest, w.longest);
    }
    // Records cross HBM twice: written by the prefill kernel, read by the merge.
    const double records_us =
        records ? kMergeLaunchUs + 2.0 * (double)records * (dp * 4 + 8) / kRecordBytesPerUs : 0.0;
    cands.push_back({std::max(total / (8.0 * kCusPerXcd), longest) + records_us, records_us, split_keys});
  }
  // Ties go to the larger split (fewer items and records).
  std::sort(cands.begin(), cands.end(), [](const Candidate &a, const Candidate &b) {
    return a.bound != b.bound ? a.bound < b.bound : a.split_keys > b.split_keys;
  });
  int64_t best_keys = cands.front().split_keys;
  double best_us = -1;
  std::vector<double> work;
  for (const Candidate &c : cands) {
    if (best_us >= 0 && c.bound >= best_us) break;
    // Items in launch order (row, kv head, split, tile), as prefill_item_work lists them.
    work.clear();
    for (size_t r = 0; r < rows.size(); ++r) {
      const RowWork &w = work_of(r, prefill_splits(rows[r].length, c.split_keys));
      for (int64_t h = 0; h < g.Hkv; ++h) work.insert(work.end(), w.items.begin(), w.items.end());
    }
    const double us = simulated_prefill_us(work) + c.records_us;
    if (best_us < 0 || us < best_us || (us == best_us && c.split_keys > best_keys)) {
      best_us = us;
      best_keys = c.split_keys;
    }
  }
  return best_keys;
}

// Whether this device deals consecutive blocks to its 8 XCDs in turn, probed
// once per device.  The probe runs on a private non-blocking stream, with
// this thread in relaxed capture mode, so that neither the caller's stream
// nor a capture another stream holds sees its launch, copy or synchronise.
// A first call made while the caller's stream is being captured skips the
// probe; until the probe has run, and if it disagrees, the merge launch is
// used.
bool xcd_dispatch_round_robin(hipStream_t stream) {
  constexpr int kMaxDevices = 64;
  static std::mutex lock;
  static int8_t known[kMaxDevices] = {};  // 0 unknown, 1 round robin, -1 not
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return false;
  std::lock_guard<std::mutex> guard(lock);
  if (known[device] == 0) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess || status != hipStreamCaptureStatusNone) return false;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return false;
    hipStream_t probe_stream = nullptr;
    bool round_robin = false;
    hipError_t err = hipStreamCreateWithFlags(&probe_stream, hipStreamNonBlocking);
    if (err == hipSuccess) err = probe_xcd_dispatch(&round_robin, probe_stream);
    if (probe_stream != nullptr) (void)hipStreamDestroy(probe_stream);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (err != hipSuccess) return false;
    known[device] = round_robin ? 1 : -1;
  }
  return known[device] == 1;
}

// XINFER_DECODE_MERGE_LAUNCH=1 keeps every decode split on the merge launch
// (read once per process): the check that both paths give the same bits.
bool merge_launch_forced() {
  static const bool forced = [] {
    const char *value = std::getenv("XINFER_DECODE_MERGE_LAUNCH");
    return value != nullptr && value[0] == '1';
  }();
  return forced;
}

// A nonzero tag below 2^36 for every decode launch that counts arrivals; not a
// small number, which other data left in the workspace may look like.
uint64_t next_launch_tag() {
  static std::atomic<uint64_t> sequence{0};
  constexpr uint64_t kTags = (uint64_t(1) << 36) - 1;  // no common factor with the step below
  return sequence.fetch_add(1, std::memory_order_relaxed) % kTags * 0x5851f45ull % kTags + 1;
}

// Query vectors per KV head up to which a row of the call takes the decode
// kernel: kStreamMaxVectors, whose columns hold them and whose stream is bound by
// HBM; but kExactVectors, as far as the weights' precision needs it, in three cases where
// every decode row has more.  Without prefill rows: if a row fills two column groups, whose
// combination takes longer than a whole unsplit prefill item, and all keys are few, by
// shortest_keys.  Beside prefill rows, head dim 64, whose prefill items take little (0.9 us a tile): unless the prefill rows'
// items leave CUs free (one_launch_pays) and some row is longer than kShortRowKeys.  Head dims
// to 128 with at most two query heads per KV head: if no row is longer than
// kPrefillMinSplitKeys, where no prefill row is split and merged.  Measured on MI355X, short
// rows of 9-32 vectors on the decode / the prefill kernel:
// D = 64: beside 200 tokens, 1, 4, 12 rows of 32 keys 9.2 / 7.6, 9.3 / 7.7, 9.7 / 8.2 us, of 700 12.4 /
//  12.0, 13.1 / 12.5, 15.1 / 13.4, of 6000 14.3 / 14.5, 21.7 / 25.3, 40.1 / 46.8; beside 384 of 1400 keys
//  12 rows of 700 17.2 / 23.4; beside 812 tokens over 5000 keys (288 items) 4 rows of 32, 700,
//  6000 keys 24.7 / 24.1, 33.7 / 24.0, 41.1 / 32.9.
// D = 128, 2 heads: beside 200 tokens 1, 4, 12 rows of 200 keys 13.0 / 12.3, 14.1 / 12.7, 16.3 / 13.5,
//  of 700 14.5 / 16.8, 15.7 / 17.2, 21.2 / 29.0; beside 384 tokens 4 rows of 32 17.9 / 28.0;
//  beside 812 tokens 12 rows of 32 54.8 / 65.2, but 4 of 700 56.3 / 50.0.  4 heads: beside 200
//  tokens 4 rows of 200 keys 14.8 / 15.7.
// D = 256: beside 200 tokens 4 rows of 32 17.6 / 20.2, beside 384 12 of 32 32.2 / 62.9.
// Alone, 32 vectors: D = 256: 4 rows of 9, 68, 208 keys 9.8 / 7.5, 11.5 / 9.1, 13.4 / 13.5, one row of
//  208 12.6 / 12.9; D = 64: 33, 92, 232 keys 6.1 / 5.8, 6.3 / 6.25, 6.4 / 7.5; D = 128: 17 keys 7.0 / 7.2,
//  76 7.0 / 7.7.
// In each case only while the short rows' prefill items are few (pairs of row and KV head; items
// of kPrefillMinSplitKeys keys): alone, D = 256, 60 keys, 256 pairs 13.0 / 11.0, 512 18.1 / 21.9, D = 64,
//  48 keys, 128 pairs 6.6 / 6.1, 512 8.2 / 11.2; beside 200 tokens, 500 keys, 240 pairs D = 128 28.8 /
//  35.3, D = 64 16.1 / 18.0; D = 64 beside 812 tokens 1152 items 58.0 / 57.7, 2048 73.5 / 78.4, 2880 88 / 113.
constexpr int64_t kShortRowKeys = 1024;
constexpr int64_t shortest_keys(int64_t D) { return D <= 64 ? 48 : (D <= 128 ? 0 : 128); }
int64_t decode_vector_limit(const Geometry &g, const std::vector<int32_t> &counts, const std::vector<int32_t> &lengths,
                            int G) {
  bool narrow = false, wide = false;
  int64_t widest = 0, longest = 0, short_pairs = 0;
  int64_t prefill_items = 0, short_items = 0;  // of kPrefillMinSplitKeys keys
  for (int64_t r = 0; r < g.B; ++r) {
    const int64_t qv = (int64_t)counts[r] * G;
    if (qv > 0) longest = std::max<int64_t>(longest, lengths[r]);
    widest = std::max(widest, qv);
    if (qv > kStreamMaxVectors) {
      wide = true;
      prefill_items += g.Hkv * ceil_div(qv, kPrefillTileQ) * ceil_div(lengths[r], kPrefillMinSplitKeys);
    } else if (qv > kExactVectors) {
      short_pairs += g.Hkv;
      short_items += g.Hkv * ceil_div(lengths[r], kPrefillMinSplitKeys);
    } else if (qv > 0) {
      narrow = true;
    }
  }
  if (narrow) return kStreamMaxVectors;
  const bool free_cus = prefill_items <= kPrefillFreeItems;
  bool decode = true;
  if (!wide) decode = widest <= 16 || longest > shortest_keys(g.D) || short_pairs > kDecodeCus;
  else if (g.D <= 64) decode = free_cus ? longest > kShortRowKeys || short_items > kPrefillFreeItems : short_items > 1024;
  else if (g.D <= 128 && G <= 2) decode = longest > kPrefillMinSplitKeys || short_pairs > kPrefillFreeItems;
  return decode ? kStreamMaxVectors : kExactVectors;
}

// Whether the decode rows `dec` and the prefill rows whose items take `work`
// microseconds go in one launch, where decode items stream their keys on the CUs
// that the prefill items leave free or have left.  An item pair per CU streams less
// well than two independent blocks, and a CU holds one pair, so where the prefill items
// fill the chip it pays only for a few decode rows beside long prefill; where they leave CUs
// free (kPrefillFreeItems) the second launch and its merge cost more, while the decode
// rows' bytes (keys, and zeros of padded queries) take up to three times as long as
// the prefill items.  Measured, two launches -> one (us; ratio of the two times):
// few prefill items: D = 128: 7 decode rows and 384 tokens 33.8 -> 24.5 (0.9), 20 rows and 200
// tokens 27.7 -> 26.2 (1.5), 45.5 -> 41.5 (3.6), 7 long rows 43.3 -> 46.1 (3.6), 8 rows and 64
// tokens 92 -> 98 (17), 24 rows 126 -> 173 (25); D = 64: 20 rows and 200 tokens 27.4 -> 22.1
// (1.9), 8 long rows 51.9 -> 53.4 (5.9), 24 rows 69.6 -> 89.8 (8.8), but 60 rows 69.5 -> 61.6
// (8.2); D = 256: 7 rows and 200 tokens 37.0 -> 24.8 (1.0), 52.2 -> 45.2 (2.8), 20 rows 57.4 ->
// 48.1 (3.0), 106 -> 110 (7.9), 20 rows and 384 tokens 72.9 -> 76.9 (2.1), 122 -> 140 (5.1).
// Many: D = 128: 4 rows and 4 x 512 tokens 174 -> 162 (0.1), 1 row and 2000 tokens 198 -> 191
// (0.04), but 6 rows and 4 x 512 tokens 128 -> 131 (0.2), 5 rows and 512 tokens 36.9 -> 39.2
// (0.9), 7 long rows 45.2 -> 53.5 (1.8), 31 long rows and 4 x 512 tokens 187 -> 211 (0.7);
// D = 64 109 -> 126 (0.8).
constexpr double kDecodeBytesPerUs = 5.5e6;
bool one_launch_pays(const Geometry &g, const AttnArgs &dec, int G, const std::vector<double> &work) {
  double bytes = 0, total = 0, longest = 0;
  for (int r = 0; r < dec.nrows; ++r) {
    const RowSched &rs = dec.rows[r];
    if (rs.count > 0) bytes += 4.0 * (double)rs.length * (double)(g.Hkv * g.D);
    bytes += 2.0 * (double)(g.T - rs.count) * (double)(g.Hkv * G * g.D);
  }
  for (const double us : work) {
    total += us;
    longest = std::max(longest, us);
  }
  const double prefill_us = std::max(longest, total / (8.0 * kCusPerXcd));
  const bool free_cus = work.size() <= kPrefillFreeItems;
  return bytes / kDecodeBytesPerUs <= (free_cus ? 3.0 : 0.1) * prefill_us;
}

// The schedule of a call whose rows of up to decode_vectors query vectors per KV
// head take the decode kernel, its items `stretch` times as long as
// choose_decode_passes has them.
Plan plan_rows(const Geometry &g, const std::vector<int32_t> &counts, const std::vector<int32_t> &lengths,
               int64_t decode_vectors, int64_t stretch) {
  Plan plan;
  plan.D = g.D;
  const int G = (int)(g.Hq / g.Hkv);
  const int dp = padded_dim(g.D);

  // Keys per prefill split, chosen from the whole call's prefill work.
  const int64_t split_keys = choose_split_keys(g, counts, lengths, G, dp, decode_vectors);

  for (int64_t row0 = 0; row0 < g.B; row0 += kMaxRows) {
    Group grp;
    grp.row0 = (int)row0;
    grp.nrows = (int)std::min<int64_t>(kMaxRows, g.B - row0);
    int64_t records = 0;  // of this group: the groups' launches run one after another
    // Longer decode rows first: the launch's last items are then short ones.  Prefill
    // rows keep the batch's order, which choose_split_keys simulates (sorted as
    // well, a ragged D = 256 batch took 488 us in place of 457).
    std::array<int, kMaxRows> order;
    const auto order_end = order.begin() + grp.nrows;
    std::iota(order.begin(), order_end, 0);
    auto decode_length = [&](int r) {
      return (int64_t)counts[row0 + r] * G <= decode_vectors ? lengths[row0 + r] : 0;
    };
    std::sort(order.begin(), order_end, [&](int x, int y) {
      return decode_length(x) != decode_length(y) ? decode_length(x) > decode_length(y) : x < y;
    });
    DecodeLoad load;
    bool prefill = false;
    const int64_t pass = decode_tokens_per_item(dp);
    for (auto r = order.begin(); r != order_end; ++r) {
      const int64_t qv = (int64_t)counts[row0 + *r] * G;
      if (qv > decode_vectors) prefill = true;
      else if (qv > 0) {
        const int64_t passes = ceil_div(lengths[row0 + *r], pass);
        load.rows[load.n++] = {(uint32_t)passes, (uint32_t)qv};
        load.passes += g.Hkv * passes;
        load.longest = std::max(load.longest, passes);
        load.widest = std::max(load.widest, qv);
      }
    }
    const int64_t item_keys = choose_decode_passes(g, load, dp, prefill) * pass * stretch;
    int64_t split_vectors = 0, decode_records = 0;  // most vectors of a split decode row
    for (auto next = order.begin(); next != order_end; ++next) {
      const int r = *next;
      const int64_t b = row0 + r;
      const int cnt = counts[b], len = lengths[b];
      const int64_t qv = (int64_t)cnt * G;
      RowSched rs{};
      rs.batch = (int32_t)b;
      rs.count = cnt;
      rs.length = len;
      rs.ntiles = 1;
      rs.nsplit = 1;
      const bool decode = qv <= decode_vectors;  // includes rows with no query (zero fill only)
      if (decode) {
        grp.dec_columns = std::max(grp.dec_columns, decode_column_groups((int)qv));
        if (cnt > 0) rs.nsplit = (int32_t)ceil_div(len, item_keys);
        // Equal splits, in whole wave tiles: none is empty, since a split never
        // holds more than item_keys, a multiple of them.
        const int64_t tile = decode_tokens_per_item(dp) / kDecodeWaves;
        rs.ntiles = (int32_t)(ceil_div(ceil_div(len, rs.nsplit), tile) * tile);
        rs.item_begin = grp.dec_items;
        grp.dec_items += (int)(g.Hkv * rs.nsplit);
        grp.dec_max_splits = std::max(grp.dec_max_splits, (int)rs.nsplit);
        if (rs.nsplit > 1) {
          split_vectors = std::max(split_vectors, qv);
          decode_records += g.Hkv * rs.nsplit * qv;
        }
      } else {
        rs.ntiles = (int32_t)ceil_div(qv, kPrefillTileQ);
        rs.nsplit = prefill_splits(len, split_keys);
        rs.item_begin = grp.pre_items;
        grp.pre_items += (int)(g.Hkv * rs.ntiles * rs.nsplit);
        grp.pre_max_splits = std::max(grp.pre_max_splits, (int)rs.nsplit);
      }
      if (rs.nsplit > 1) {
        // Decode: [kv head][split][vector] records.  Prefill: per (kv head,
        // split, query tile) a block of kPrefillTileQ records.
        rs.rec_begin = records;
        records += g.Hkv * rs.nsplit * (decode ? qv : rs.ntiles * kPrefillTileQ);
        MergeArgs &merge = decode ? grp.dec_merge : grp.pre_merge;
        int &merge_items = decode ? grp.dec_merge_items : grp.pre_merge_items;
        MergeRow &mr = merge.rows[merge.nrows++];
        mr.batch = (int32_t)b;
        mr.count = cnt;
        mr.nsplit = rs.nsplit;
        mr.item_begin = merge_items;
        mr.tiles = decode ? 0 : rs.ntiles;
        mr.rec_begin = rs.rec_begin;
        merge_items += (int)(g.Hkv * qv);
      }
      AttnArgs &a = decode ? grp.dec : grp.pre;
      a.rows[a.nrows++] = rs;
    }
    plan.records = std::max(plan.records, records);
    grp.dec_fusable = merge_in_launch_pays(g.Hkv, grp.dec_items, grp.dec_max_splits, split_vectors,
                                           (double)(decode_records * (4 * g.D + 8)), dp);
    if (grp.dec_fusable) plan.counters = std::max<int64_t>(plan.counters, grp.dec_items);
    if (grp.pre_items > 0) {
      const std::vector<double> work = prefill_item_work(grp.pre.rows, grp.pre.nrows, g.Hkv, G, dp);
      xcd_runs(work, grp.pre.xcd_begin);
      if (grp.dec_items > 0) grp.both = one_launch_pays(g, grp.dec, G, work);
    }
    plan.groups.push_back(grp);
  }
  return plan;
}

// counts/lengths: per-row real queries and populated KV lengths (validated).
//
// max_bytes: what the entry point's own scratch holds (the allocation-free one),
// where the caller brings no workspace.  A plan that needs more gives way: longer
// decode items, then rows of more than kExactVectors vectors on the prefill
// kernel as well, whose records are those of their query tiles.  The last
// plan tried splits no decode row, so what is refused is refused for prefill
// records alone.
Plan make_plan(const Geometry &g, const std::vector<int32_t> &counts, const std::vector<int32_t> &lengths,
               size_t max_bytes) {
  const int64_t limit = decode_vector_limit(g, counts, lengths, (int)(g.Hq / g.Hkv));
  Plan plan = plan_rows(g, counts, lengths, limit, 1);
  if (plan.bytes() > max_bytes) plan = plan_rows(g, counts, lengths, limit, 2);
  const int64_t pass = decode_tokens_per_item(padded_dim(g.D));
  for (int64_t stretch = 1; plan.bytes() > max_bytes; stretch *= 2) {
    plan = plan_rows(g, counts, lengths, kExactVectors, stretch);
    if (stretch * pass >= g.C) break;  // every item at least a row's keys
  }
  return plan;
}

// The plan of this thread's last call.  A model step calls the operator once
// per layer with the same counts and lengths, and every call plans twice (its
// workspace size, then the launch), while planning a ragged prefill batch
// simulates its dispatch at several split sizes (about 0.36 ms for the
// batch-8 D = 256 prefill of 2235 tokens); a call whose geometry, counts,
// lengths and record limit equal the last one's reuses that plan.  A plan depends
// on nothing else: not on the device, the stream or the tensors' addresses.  The
// reference holds until the thread's next call.
const Plan &cached_plan(const Geometry &g, const std::vector<int32_t> &counts, const std::vector<int32_t> &lengths,
                 size_t max_bytes = SIZE_MAX) {
  struct Entry {
    bool valid = false;
    size_t max_bytes = 0;
    Geometry g{};
    std::vector<int32_t> counts, lengths;
    Plan plan;
  };
  thread_local Entry last;
  const bool same = last.valid && last.g.B == g.B && last.g.Hq == g.Hq && last.g.Hkv == g.Hkv &&
                    last.g.T == g.T && last.g.D == g.D && last.g.C == g.C && last.max_bytes == max_bytes &&
                    last.counts == counts && last.lengths == lengths;
  if (!same) {
    last.valid = false;
    last.plan = make_plan(g, counts, lengths, max_bytes);
    last.g = g;
    last.max_bytes = max_bytes;
    last.counts = counts;
    last.lengths = lengths;
    last.valid = true;
  }
  return last.plan;
}

// A page table (nullable) is a device int32 pointer with a non-negative row stride.
int check_blocks(const int32_t *blocks, int64_t blocks_stride) {
  if (blocks == nullptr) return XINFER_OK;
  if ((reinterpret_cast<uintptr_t>(blocks) & 3u) != 0 || blocks_stride < 0) return XINFER_ERR_ARGUMENT;
  return XINFER_OK;
}

int run_plan(const Plan &plan, const Geometry &g, const xinfer_view4 &q, const xinfer_view4 &k,
             const xinfer_view4 &v, const int32_t *blocks, int64_t blocks_stride, double scale,
             const xinfer_view4 &out, void *workspace, hipStream_t stream) {
  const int G = (int)(g.Hq / g.Hkv);
  const int dp = padded_dim(g.D);
  float *part_o = static_cast<float *>(workspace);
  float *part_ml =
      plan.records ? reinterpret_cast<float *>(static_cast<char *>(workspace) + plan.part_ml_offset())
                   : nullptr;
  // What is launched is a copy with the tensors' places filled in (a Group's
  // tables are 10 KB; of the empty ones nothing is copied).
  const auto attention_args = [&](const AttnArgs &planned, int items) {
    AttnArgs a = planned;
    a.q = view_of(q);
    a.k = view_of(k);
    a.v = view_of(v);
    a.out = static_cast<uint16_t *>(const_cast<void *>(out.data));
    a.o_sb = out.stride[0];
    a.o_sh = out.stride[1];
    a.o_st = out.stride[2];
    a.part_o = part_o;
    a.part_ml = part_ml;
    a.scale_log2 = (float)(scale * 1.4426950408889634);
    a.D = (int32_t)g.D;
    a.G = G;
    a.Hkv = (int32_t)g.Hkv;
    a.T = (int32_t)g.T;
    a.blocks = blocks;
    a.blocks_stride = blocks_stride;
    a.kv_rows = (int32_t)g.B;
    a.total_items = items;
    return a;
  };
  const auto merge_args = [&](const MergeArgs &planned, int items) {
    MergeArgs m = planned;
    m.out = static_cast<uint16_t *>(const_cast<void *>(out.data));
    m.o_sb = out.stride[0];
    m.o_sh = out.stride[1];
    m.o_st = out.stride[2];
    m.part_o = part_o;
    m.part_ml = part_ml;
    m.D = (int32_t)g.D;
    m.G = G;
    m.total_items = items;
    return m;
  };
  for (const Group &grp : plan.groups) {
    int dec_merge_items = grp.dec_merge_items;
    hipError_t rc = hipSuccess;
    if (grp.both) {
      rc = launch_attention_both(attention_args(grp.dec, grp.dec_items), attention_args(grp.pre, grp.pre_items), dp,
                                 grp.dec_columns, stream);
    } else {
      if (grp.dec_items > 0) {
        AttnArgs a = attention_args(grp.dec, grp.dec_items);
        if (grp.dec_fusable && !merge_launch_forced() && xcd_dispatch_round_robin(stream)) {
          a.arrive_ctr = reinterpret_cast<uint64_t *>(static_cast<char *>(workspace) + plan.counters_offset());
          a.tag = next_launch_tag();
          dec_merge_items = 0;  // the decode rows are merged in the launch
        }
        rc = launch_decode(a, dp, grp.dec_columns, grp.dec_items, stream);
      }
      if (rc == hipSuccess && grp.pre_items > 0)
        rc = launch_prefill(attention_args(grp.pre, grp.pre_items), dp, stream);
    }
    if (rc != hipSuccess) return XINFER_ERR_LAUNCH;
    if (dec_merge_items > 0 && grp.pre_merge_items > 0)
      rc = launch_merge_both(merge_args(grp.dec_merge, dec_merge_items), merge_args(grp.pre_merge, grp.pre_merge_items),
                             dp, grp.dec_max_splits, grp.pre_max_splits, stream);
    else if (dec_merge_items > 0)
      rc = launch_merge(merge_args(grp.dec_merge, dec_merge_items), dp, grp.dec_max_splits, stream);
    else if (grp.pre_merge_items > 0)
      rc = launch_merge(merge_args(grp.pre_merge, grp.pre_merge_items), dp, grp.pre_max_splits, stream);
    if (rc != hipSuccess) return XINFER_ERR_LAUNCH;
  }
  return XINFER_OK;
}

// The contiguous [B, Hq, T, D] output the operators allocate.
xinfer_view4 contiguous_output(const Geometry &g, void *out) {
  xinfer_view4 o{};
  o.data = out;
  const int64_t sizes[4] = {g.B, g.Hq, g.T, g.D};
  const int64_t strides[4] = {g.Hq * g.T * g.D, g.T * g.D, g.D, 1};
  for (int i = 0; i < 4; ++i) {
    o.size[i] = sizes[i];
    o.stride[i] = strides[i];
  }
  return o;
}

// An output view the kernels can write: q's sizes, unit feature stride, the
// other strides multiples of 8 elements, 16-byte aligned data.
int check_output(const Geometry &g, const xinfer_view4 *out) {
  if (out == nullptr || out->data == nullptr) return XINFER_ERR_ARGUMENT;
  const int64_t sizes[4] = {g.B, g.Hq, g.T, g.D};
  for (int i = 0; i < 4; ++i)
    if (out->size[i] != sizes[i]) return XINFER_ERR_QKV_SHAPES;
  if ((reinterpret_cast<uintptr_t>(out->data) & 15u) != 0 || out->stride[3] != 1) return XINFER_ERR_LAYOUT;
  for (int i = 0; i < 3; ++i)
    if (out->stride[i] % 8 != 0 || out->stride[i] < 0) return XINFER_ERR_LAYOUT;
  return XINFER_OK;
}

// Validation of xinfer::flash_attention (attention.cpp:84-104), in its order.
int check_flash(const xinfer_view4 *q, const xinfer_view4 *k, const xinfer_view4 *v,
                int64_t valid_length, Geometry &g) {
  if (!q || !k || !v) return XINFER_ERR_ARGUMENT;
  g = Geometry{q->size[0], q->size[1], k->size[1], q->size[2], q->size[3], k->size[2]};
  if (!(g.B > 0 && g.T >= 1 && g.T <= 512)) return XINFER_ERR_Q_SHAPE;
  bool same = true;
  for (int i = 0; i < 4; ++i) same = same && v->size[i] == k->size[i];
  if (!(k->size[0] == g.B && g.C > 0 && k->size[3] == g.D && same)) return XINFER_ERR_KV_SHAPE;
  if (int rc = check_heads_and_dim(g)) return rc;
  if (!(valid_length >= g.T && valid_length <= g.C)) return XINFER_ERR_PREFIX;
  return XINFER_OK;
}

// Validation of xinfer::batched_flash_attention (attention.cpp:17-45).
int check_batched(const xinfer_view4 *q, const xinfer_view4 *k, const xinfer_view4 *v,
                  const int32_t *offsets, Geometry &g, std::vector<int32_t> &counts,
                  std::vector<int32_t> &lengths) {
  if (!q || !k || !v || !offsets) return XINFER_ERR_ARGUMENT;
  g = Geometry{q->size[0], q->size[1], k->size[1], q->size[2], q->size[3], k->size[2]};
  bool same = true;
  for (int i = 0; i < 4; ++i) same = same && v->size[i] == k->size[i];
  if (!(same && k->size[0] == g.B && k->size[3] == g.D) || g.B < 0 || g.T < 0)
    return XINFER_ERR_QKV_SHAPES;
  if (int rc = check_heads_and_dim(g)) return rc;
  const int32_t *cuq = offsets, *cuk = offsets + g.B + 1;
  if (cuq[0] != 0 || cuk[0] != 0) return XINFER_ERR_OFFSETS_START;
  counts.resize(g.B);
  lengths.resize(g.B);
  for (int64_t r = 0; r < g.B; ++r) {
    const int64_t count = (int64_t)cuq[r + 1] - cuq[r], length = (int64_t)cuk[r + 1] - cuk[r];
    if (!(count >= 0 && count <= g.T && length >= count && length >= 1 && length <= g.C))
      return XINFER_ERR_LENGTHS;
    counts[r] = (int32_t)count;
    lengths[r] = (int32_t)length;
  }
  return XINFER_OK;
}

// Graph-capture mode (xinfer_batched_flash_attention_graph): a plan that
// depends only on the shapes.  Rows must take the decode kernel (at most
// kCaptureDecodeMaxVectors query vectors per KV head, i.e. T * G <= 8) and fit
// one row table (B <= kMaxRows, which the kernels' per-block tables assume).
// Records are laid out for every row at capacity.
struct CapturePlan {
  int dp = 0, columns = 1, splits_max = 0, decode_blocks = 0, pass_min = 1;
  int64_t row_records = 0, records = 0;
  int64_t dp_d = 0;  // the head dim D (records hold D floats)
  // Prefill shapes (T * Hq/Hkv > 8): every row takes the prefill kernel,
  // planned on the device; the workspace also holds the prefill and merge
  // arguments the plan kernel writes.
  bool prefill = false;
  int64_t items_max = 0, vectors_max = 0;
  size_t part_ml_offset() const { return (size_t)((records * dp_d * 4 + 255) / 256 * 256); }
  size_t records_bytes() const { return records ? part_ml_offset() + (size_t)records * 8 : 0; }
  size_t attn_offset() const { return (records_bytes() + 255) / 256 * 256; }
  size_t merge_offset() const { return attn_offset() + (sizeof(AttnArgs) + 255) / 256 * 256; }
  size_t bytes() const { return prefill ? merge_offset() + sizeof(MergeArgs) : records_bytes(); }
};
// A decode launch's records are sized for items of kDecodeItemRounds passes
// where the capacity layout has at least kCaptureManyItems items of one pass and
// at most kCaptureItems of the longer ones; else for items of one pass.
constexpr int64_t kCaptureManyItems = 1536, kCaptureItems = 2048;

int check_capture(const xinfer_view4 *q, const xinfer_view4 *k, const xinfer_view4 *v, Geometry &g,
                  CapturePlan &cp) {
  if (!q || !k || !v) return XINFER_ERR_ARGUMENT;
  g = Geometry{q->size[0], q->size[1], k->size[1], q->size[2], q->size[3], k->size[2]};
  bool same = true;
  for (int i = 0; i < 4; ++i) same = same && v->size[i] == k->size[i];
  if (!(same && k->size[0] == g.B && k->size[3] == g.D) || g.B < 0 || g.T < 0 || g.C <= 0)
    return XINFER_ERR_QKV_SHAPES;
  if (int rc = check_heads_and_dim(g)) return rc;
  const int64_t G = g.Hq / g.Hkv;
  if (g.B > kMaxRows) return XINFER_ERR_CAPTURE_ROWS;
  cp.dp = padded_dim(g.D);
  cp.dp_d = g.D;
  if (g.T * G > kCaptureDecodeMaxVectors) {
    // Prefill shapes: the device plan (prefill.hip:
    // prefill_capture_plan_kernel) picks the split size from the lengths, in
    // the range choose_split_keys searches, so that the items stay below
    // 2048 + one per (row, kv head, query tile); no row takes more than
    // kMergeSerialSplits splits (or splits below kPrefillMinSplitKeys keys).
    // The prefill grid, the records and the merge grid are sized for that.
    cp.prefill = true;
    const int64_t unsplit = g.B * g.Hkv * ceil_div(g.T * G, kPrefillTileQ);
    cp.splits_max = (int)std::min<int64_t>(kMergeSerialSplits, ceil_div(g.C, kPrefillMinSplitKeys));
    cp.items_max = std::min(2048 + unsplit, unsplit * cp.splits_max);
    cp.vectors_max = g.B * g.Hkv * g.T * G;
    cp.records = cp.splits_max > 1 ? cp.items_max * kPrefillTileQ : 0;
    // Item, record and vector indices are 32-bit on the device (a q tensor
    // that large would not fit in memory).
    if (cp.items_max * kPrefillTileQ >= (int64_t(1) << 31) || cp.vectors_max >= (int64_t(1) << 31))
      return XINFER_ERR_QKV_SHAPES;
    return XINFER_OK;
  }
  cp.columns = decode_column_groups((int)(g.T * G));
  const int tok_round = decode_tokens_per_item(cp.dp);
  const int64_t one_round_items = g.B * g.Hkv * ceil_div(g.C, tok_round);
  const int64_t multi_round_items = g.B * g.Hkv * ceil_div(g.C, (int64_t)kDecodeItemRounds * tok_round);
  const int rounds = one_round_items >= kCaptureManyItems && multi_round_items <= kCaptureItems ? kDecodeItemRounds : 1;
  cp.pass_min = rounds;
  cp.splits_max = (int)ceil_div(g.C, rounds * tok_round);
  const int64_t pairs = g.B * g.Hkv, vectors = g.T * G;
  cp.records = cp.splits_max > 1 ? pairs * cp.splits_max * vectors : 0;
  // Every item the kernel may lay out (device_common.h: capture_splits).
  cp.decode_blocks = (int)(ceil_div(std::min<int64_t>(pairs * cp.splits_max, 4 * kDecodeCus + pairs), 8) * 8);
  return XINFER_OK;
}

// The caller's workspace: at least `need` bytes, 16-byte aligned (the records
// take 16-byte stores; the argument blocks planned on the device are read
// with scalar loads).  A workspace of zero bytes may be null.
int check_workspace(const void *workspace, size_t bytes, size_t need) {
  if (bytes < need || (need && workspace == nullptr) || (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0)
    return XINFER_ERR_WORKSPACE;
  return XINFER_OK;
}

int check_common(const xinfer_view4 &q, const xinfer_view4 &k, const xinfer_view4 &v, double scale) {
  if (!(std::isfinite(scale) && scale > 0)) return XINFER_ERR_SCALE;
  if (!attention_layout_ok(q) || !query_layout_ok(q) || !attention_layout_ok(k) ||
      !attention_layout_ok(v))
    return XINFER_ERR_LAYOUT;
  return XINFER_OK;
}

}  // namespace
}  // namespace xattn

using namespace xattn;

extern "C" {

const char *xinfer_status_string(int status) {
  switch (status) {
    case XINFER_OK: return "Success";
    case XINFER_ERR_QKV_SHAPES: return "Invalid Q/K/V shapes";
    case XINFER_ERR_Q_SHAPE: return "Unsupported Q shape";
    case XINFER_ERR_KV_SHAPE:
      return "Expected matching full-capacity K/V inputs [batch,kv_heads,capacity,head_dim]";
    case XINFER_ERR_HEADS: return "Query heads must be a positive multiple of KV heads";
    case XINFER_ERR_HEAD_DIM: return "Flash head dimension must be a multiple of 8 in 8..256";
    case XINFER_ERR_PREFIX: return "Invalid valid-prefix length";
    case XINFER_ERR_SCALE: return "Attention scale must be finite and positive";
    case XINFER_ERR_OFFSETS_START: return "Cumulative lengths must start at zero";
    case XINFER_ERR_LENGTHS: return "Invalid query/KV lengths";
    case XINFER_ERR_WORKSPACE: return "Attention workspace is smaller than its size query or not 16-byte aligned";
    case XINFER_ERR_LAYOUT:
      return "Attention tensors need a unit feature stride, strides divisible by 8 and 16-byte "
             "aligned data";
    case XINFER_ERR_CACHE:
      return "Expected contiguous KV caches [batch,kv_heads,capacity,head_dim] matching key/value";
    case XINFER_ERR_LAUNCH: return "HIP kernel launch failed";
    case XINFER_ERR_ARGUMENT: return "Invalid argument";
    case XINFER_ERR_ROPE_SHAPE:
      return "Expected q [B,Hq,T,D], key/value [B,Hkv,T,D] and cos/sin [B,1,T,D] with D in {64,128,256}";
    case XINFER_ERR_EPS: return "RMSNorm epsilon must be finite and non-negative";
    case XINFER_ERR_CAPTURE_ROWS:
      return "Graph-capture attention takes at most 64 rows";
    case XINFER_ERR_SCRATCH:
      return "Attention needs more split-record scratch than the allocation-free entry point holds (32 MiB)";
    default: return "Unknown xinfer status";
  }
}

size_t xinfer_batched_flash_attention_workspace_size(const xinfer_view4 *q, const xinfer_view4 *k,
                                                     const int32_t *host_offsets) {
  Geometry g;
  std::vector<int32_t> counts, lengths;
  if (check_batched(q, k, k, host_offsets, g, counts, lengths) != XINFER_OK) return 0;
  return cached_plan(g, counts, lengths).bytes();
}

int xinfer_batched_flash_attention(const xinfer_view4 *q, const xinfer_view4 *k,
                                   const xinfer_view4 *v, const int32_t *host_offsets,
                                   const int32_t *blocks, int64_t blocks_stride, double scale,
                                   void *out, void *workspace, size_t workspace_bytes,
                                   void *stream) {
  Geometry g;
  std::vector<int32_t> counts, lengths;
  if (int rc = check_batched(q, k, v, host_offsets, g, counts, lengths)) return rc;
  if (int rc = check_common(*q, *k, *v, scale)) return rc;
  if (int rc = check_blocks(blocks, blocks_stride)) return rc;
  if (g.B == 0 || g.T == 0) return XINFER_OK;
  if (out == nullptr) return XINFER_ERR_ARGUMENT;
  const Plan &plan = cached_plan(g, counts, lengths);
  if (int rc = check_workspace(workspace, workspace_bytes, plan.bytes())) return rc;
  return run_plan(plan, g, *q, *k, *v, blocks, blocks_stride, scale, contiguous_output(g, out), workspace,
                  static_cast<hipStream_t>(stream));
}

size_t xinfer_batched_flash_attention_graph_workspace_size(const xinfer_view4 *q, const xinfer_view4 *k) {
  Geometry g;
  CapturePlan cp;
  if (check_capture(q, k, k, g, cp) != XINFER_OK) return 0;
  return cp.bytes();
}

int xinfer_batched_flash_attention_graph(const xinfer_view4 *q, const xinfer_view4 *k, const xinfer_view4 *v,
                                         const int32_t *device_offsets, const int32_t *blocks,
                                         int64_t blocks_stride, double scale, void *out, void *workspace,
                                         size_t workspace_bytes, void *stream) {
  Geometry g;
  CapturePlan cp;
  if (int rc = check_capture(q, k, v, g, cp)) return rc;
  if (int rc = check_common(*q, *k, *v, scale)) return rc;
  if (int rc = check_blocks(blocks, blocks_stride)) return rc;
  if (g.B == 0 || g.T == 0) return XINFER_OK;
  if (out == nullptr || device_offsets == nullptr) return XINFER_ERR_ARGUMENT;
  if (int rc = check_workspace(workspace, workspace_bytes, cp.bytes())) return rc;
  CaptureArgs c{};
  c.q = view_of(*q);
  c.k = view_of(*k);
  c.v = view_of(*v);
  c.out = static_cast<uint16_t *>(out);
  c.o_sb = g.Hq * g.T * g.D;
  c.o_sh = g.T * g.D;
  c.o_st = g.D;
  c.part_o = static_cast<float *>(workspace);
  c.part_ml = cp.records ? reinterpret_cast<float *>(static_cast<char *>(workspace) + cp.part_ml_offset()) : nullptr;
  c.offsets = device_offsets;
  c.scale_log2 = (float)(scale * 1.4426950408889634);
  c.D = (int32_t)g.D;
  c.G = (int32_t)(g.Hq / g.Hkv);
  c.Hkv = (int32_t)g.Hkv;
  c.T = (int32_t)g.T;
  c.B = (int32_t)g.B;
  c.C = (int32_t)g.C;
  c.blocks = blocks;
  c.blocks_stride = blocks_stride;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (cp.prefill) {
    char *ws = static_cast<char *>(workspace);
    PrefillPlanArgs pp{};
    pp.c = c;
    pp.attn = reinterpret_cast<AttnArgs *>(ws + cp.attn_offset());
    pp.merge = reinterpret_cast<MergeArgs *>(ws + cp.merge_offset());
    pp.items_max = (int32_t)cp.items_max;
    // 8 XCD runs of at most ceil(items_max / 8) items (the plan clamps its cuts).
    pp.run_max = (int32_t)ceil_div(cp.items_max, 8);
    pp.splits_max = cp.splits_max;
    pp.min_split_keys = (int32_t)kPrefillMinSplitKeys;
    pp.tile_us = (float)prefill_tile_us(cp.dp);
    pp.item_us = (float)kPrefillItemUs;
    pp.merge_us = (float)kMergeLaunchUs;
    pp.record_us = (float)(2.0 * (cp.dp * 4 + 8) / kRecordBytesPerUs);
    if (launch_prefill_capture(pp, cp.dp, (unsigned)(8 * pp.run_max), s) != hipSuccess) return XINFER_ERR_LAUNCH;
    if (cp.splits_max > 1 && launch_merge_dev(pp.merge, cp.dp, cp.splits_max, cp.vectors_max, s) != hipSuccess)
      return XINFER_ERR_LAUNCH;
    return XINFER_OK;
  }
  c.pass_keys = decode_tokens_per_item(cp.dp);
  c.pass_min = cp.pass_min;
  c.splits_max = cp.splits_max;
  c.row_records = g.Hkv * cp.splits_max * g.T * c.G;
  if (launch_decode_capture(c, cp.dp, cp.columns, cp.decode_blocks, s) != hipSuccess) return XINFER_ERR_LAUNCH;
  if (cp.splits_max > 1 && launch_merge_capture(c, cp.dp, s) != hipSuccess)
    return XINFER_ERR_LAUNCH;
  return XINFER_OK;
}

int xinfer_batched_flash_attention_noalloc(const xinfer_view4 *q, const xinfer_view4 *k,
                                           const xinfer_view4 *v, const int32_t *host_offsets,
                                           const int32_t *blocks, int64_t blocks_stride, double scale,
                                           void *out, void *stream) {
  static_assert(kScratchBytes == XINFER_NOALLOC_SCRATCH_BYTES, "scratch size of the C header");
  Geometry g;
  std::vector<int32_t> counts, lengths;
  if (int rc = check_batched(q, k, v, host_offsets, g, counts, lengths)) return rc;
  if (int rc = check_common(*q, *k, *v, scale)) return rc;
  if (int rc = check_blocks(blocks, blocks_stride)) return rc;
  if (g.B == 0 || g.T == 0) return XINFER_OK;
  if (out == nullptr) return XINFER_ERR_ARGUMENT;
  const Plan &plan = cached_plan(g, counts, lengths, kScratchBytes);
  if (plan.bytes() > kScratchBytes) return XINFER_ERR_SCRATCH;
  // The device address of the static scratch on the current device (never
  // the host-side name of the array).
  void *records = nullptr;
  if (plan.bytes() > 0 && scratch_pointer(&records) != hipSuccess) return XINFER_ERR_LAUNCH;
  return run_plan(plan, g, *q, *k, *v, blocks, blocks_stride, scale, contiguous_output(g, out), records,
                  static_cast<hipStream_t>(stream));
}

int xinfer_batched_flash_attention_out(const xinfer_view4 *q, const xinfer_view4 *k, const xinfer_view4 *v,
                                       const int32_t *host_offsets, const int32_t *blocks,
                                       int64_t blocks_stride, double scale, const xinfer_view4 *out,
                                       void *workspace, size_t workspace_bytes, void *stream) {
  Geometry g;
  std::vector<int32_t> counts, lengths;
  if (int rc = check_batched(q, k, v, host_offsets, g, counts, lengths)) return rc;
  if (int rc = check_common(*q, *k, *v, scale)) return rc;
  if (int rc = check_blocks(blocks, blocks_stride)) return rc;
  if (g.B == 0 || g.T == 0) return XINFER_OK;
  if (int rc = check_output(g, out)) return rc;
  const Plan &plan = cached_plan(g, counts, lengths);
  if (int rc = check_workspace(workspace, workspace_bytes, plan.bytes())) return rc;
  return run_plan(plan, g, *q, *k, *v, blocks, blocks_stride, scale, *out, workspace,
                  static_cast<hipStream_t>(stream));
}

size_t xinfer_flash_attention_workspace_size(const xinfer_view4 *q, const xinfer_view4 *k,
                                             int64_t valid_length) {
  Geometry g;
  if (check_flash(q, k, k, valid_length, g) != XINFER_OK) return 0;
  std::vector<int32_t> counts(g.B, (int32_t)g.T), lengths(g.B, (int32_t)valid_length);
  return cached_plan(g, counts, lengths).bytes();
}

int xinfer_flash_attention(const xinfer_view4 *q, const xinfer_view4 *k, const xinfer_view4 *v,
                           int64_t valid_length, double scale, void *out, void *workspace,
                           size_t workspace_bytes, void *stream) {
  Geometry g;
  if (int rc = check_flash(q, k, v, valid_length, g)) return rc;
  if (int rc = check_common(*q, *k, *v, scale)) return rc;
  if (out == nullptr) return XINFER_ERR_ARGUMENT;
  std::vector<int32_t> counts(g.B, (int32_t)g.T), lengths(g.B, (int32_t)valid_length);
  const Plan &plan = cached_plan(g, counts, lengths);
  if (int rc = check_workspace(workspace, workspace_bytes, plan.bytes())) return rc;
  return run_plan(plan, g, *q, *k, *v, nullptr, 0, scale, contiguous_output(g, out), workspace,
                  static_cast<hipStream_t>(stream));
}

int xinfer_append_kv_batched(const xinfer_view4 *key, const xinfer_view4 *value,
                             const int64_t *positions, int64_t pos_stride_b, int64_t pos_stride_t,
                             const int32_t *cu_query, const xinfer_view4 *cache_key,
                             const xinfer_view4 *cache_value, void *stream) {
  if (!key || !value || !cache_key || !cache_value) return XINFER_ERR_ARGUMENT;
  const int64_t B = key->size[0], H = key->size[1], T = key->size[2], D = key->size[3];
  for (int i = 0; i < 4; ++i)
    if (value->size[i] != key->size[i] || key->size[i] < 0) return XINFER_ERR_ARGUMENT;
  if (B == 0 || H == 0 || T == 0 || D == 0) return XINFER_OK;
  if (!positions || !cu_query || !key->data || !value->data) return XINFER_ERR_ARGUMENT;
  for (const xinfer_view4 *c : {cache_key, cache_value}) {
    if (!c->data || c->size[0] < B || c->size[1] != H || c->size[3] != D || c->size[2] <= 0)
      return XINFER_ERR_CACHE;
    if (c->stride[3] != 1 || c->stride[2] != D || c->stride[1] != c->size[2] * D ||
        c->stride[0] != H * c->size[2] * D)
      return XINFER_ERR_CACHE;
    for (int i = 0; i < 4; ++i)
      if (c->size[i] != cache_key->size[i]) return XINFER_ERR_CACHE;
  }
  AppendArgs a{};
  a.key = view_of(*key);
  a.value = view_of(*value);
  a.key_sd = key->stride[3];
  a.value_sd = value->stride[3];
  a.positions = positions;
  a.pos_sb = pos_stride_b;
  a.pos_st = pos_stride_t;
  a.cu_query = cu_query;
  a.cache_key = static_cast<uint16_t *>(const_cast<void *>(cache_key->data));
  a.cache_value = static_cast<uint16_t *>(const_cast<void *>(cache_value->data));
  a.B = (int32_t)B;
  a.H = (int32_t)H;
  a.T = (int32_t)T;
  a.D = (int32_t)D;
  a.C = (int32_t)cache_key->size[2];
  auto vec_ok = [&](const xinfer_view4 &t) {
    if ((reinterpret_cast<uintptr_t>(t.data) & 15u) != 0 || t.stride[3] != 1 || D % 8 != 0) return false;
    for (int i = 0; i < 3; ++i)
      if (t.size[i] > 1 && t.stride[i] % 8 != 0) return false;
    return true;
  };
  const bool vector = vec_ok(*key) && vec_ok(*value) &&
                      (reinterpret_cast<uintptr_t>(cache_key->data) & 15u) == 0 &&
                      (reinterpret_cast<uintptr_t>(cache_value->data) & 15u) == 0;
  return launch_append(a, vector, static_cast<hipStream_t>(stream)) == hipSuccess ? XINFER_OK
                                                                                  : XINFER_ERR_LAUNCH;
}

int xinfer_qk_norm_rope_append(const xinfer_view4 *q, const xinfer_view4 *key, const xinfer_view4 *value,
                               const void *q_weight, const void *k_weight, double eps,
                               const xinfer_view4 *cos, const xinfer_view4 *sin, const int64_t *positions,
                               int64_t pos_stride_b, int64_t pos_stride_t, const int32_t *cu_query,
                               void *q_out, const xinfer_view4 *cache_key, const xinfer_view4 *cache_value,
                               void *stream) {
  if (!q || !key || !value || !cos || !sin || !cache_key || !cache_value) return XINFER_ERR_ARGUMENT;
  const int64_t B = q->size[0], Hq = q->size[1], T = q->size[2], D = q->size[3], Hkv = key->size[1];
  for (int i = 0; i < 4; ++i)
    if (q->size[i] < 0 || key->size[i] < 0 || value->size[i] != key->size[i]) return XINFER_ERR_ROPE_SHAPE;
  if (key->size[0] != B || key->size[2] != T || key->size[3] != D || Hq <= 0 || Hkv <= 0 ||
      (D != 64 && D != 128 && D != 256))
    return XINFER_ERR_ROPE_SHAPE;
  for (const xinfer_view4 *r : {cos, sin})
    if (r->size[0] != B || r->size[1] != 1 || r->size[2] != T || r->size[3] != D) return XINFER_ERR_ROPE_SHAPE;
  if (!(std::isfinite(eps) && eps >= 0)) return XINFER_ERR_EPS;
  if (B == 0 || T == 0) return XINFER_OK;
  if (!q_weight || !k_weight || !positions || !cu_query || !q_out) return XINFER_ERR_ARGUMENT;
  // 16-byte rows: unit feature stride, other strides divisible by 8, aligned data.
  auto rows_ok = [](const xinfer_view4 &t) {
    if (t.data == nullptr || (reinterpret_cast<uintptr_t>(t.data) & 15u) != 0 || t.stride[3] != 1) return false;
    for (int i = 0; i < 3; ++i)
      if (t.size[i] > 1 && t.stride[i] % 8 != 0) return false;
    return true;
  };
  for (const xinfer_view4 *t : {q, key, value, cos, sin})
    if (!rows_ok(*t)) return XINFER_ERR_LAYOUT;
  for (const void *p : {q_weight, k_weight, static_cast<const void *>(q_out)})
    if ((reinterpret_cast<uintptr_t>(p) & 15u) != 0) return XINFER_ERR_LAYOUT;
  for (const xinfer_view4 *c : {cache_key, cache_value}) {
    if (!c->data || (reinterpret_cast<uintptr_t>(c->data) & 15u) != 0 || c->size[0] < B || c->size[1] != Hkv ||
        c->size[3] != D || c->size[2] <= 0)
      return XINFER_ERR_CACHE;
    if (c->stride[3] != 1 || c->stride[2] != D || c->stride[1] != c->size[2] * D ||
        c->stride[0] != Hkv * c->size[2] * D)
      return XINFER_ERR_CACHE;
    for (int i = 0; i < 4; ++i)
      if (c->size[i] != cache_key->size[i]) return XINFER_ERR_CACHE;
  }
  NormRopeArgs a{};
  a.q = view_of(*q);
  a.k = view_of(*key);
  a.v = view_of(*value);
  a.q_weight = static_cast<const uint16_t *>(q_weight);
  a.k_weight = static_cast<const uint16_t *>(k_weight);
  a.cos = view_of(*cos);
  a.sin = view_of(*sin);
  a.positions = positions;
  a.pos_sb = pos_stride_b;
  a.pos_st = pos_stride_t;
  a.cu_query = cu_query;
  a.q_out = static_cast<uint16_t *>(q_out);
  a.cache_key = static_cast<uint16_t *>(const_cast<void *>(cache_key->data));
  a.cache_value = static_cast<uint16_t *>(const_cast<void *>(cache_value->data));
  a.eps = (float)eps;
  a.B = (int32_t)B;
  a.T = (int32_t)T;
  a.Hq = (int32_t)Hq;
  a.Hkv = (int32_t)Hkv;
  a.D = (int32_t)D;
  a.C = (int32_t)cache_key->size[2];
  return launch_norm_rope(a, static_cast<hipStream_t>(stream)) == hipSuccess ? XINFER_OK : XINFER_ERR_LAUNCH;
}

int xinfer_projection_gemv(const void *x, const void *weight, void *out, int64_t n, int64_t k, int dtype,
                           void *stream) {
  if (!x || !weight || !out || n <= 0 || k <= 0 || k >= (int64_t(1) << 31) || n >= (int64_t(1) << 31) ||
      (dtype != XINFER_BF16 && dtype != XINFER_FP32))
    return XINFER_ERR_ARGUMENT;
  const int64_t size = dtype == XINFER_FP32 ? 4 : 2;
  const bool vec = (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(weight) & 15u) == 0 &&
                   (k * size) % 16 == 0;
  GemvArgs a{x, weight, out, n, k};
  return launch_gemv(a, dtype == XINFER_FP32, vec, static_cast<hipStream_t>(stream)) == hipSuccess
             ? XINFER_OK
             : XINFER_ERR_LAUNCH;
}

}  // extern "C"
