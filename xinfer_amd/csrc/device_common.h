// Device-side helpers for the gfx950 (CDNA4) attention kernels: bf16 bit
// conversions, 16-byte vector types, DPP row reductions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernel_args.h"

namespace xattn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Round-to-nearest-even float -> bf16 bits (hardware conversion on gfx950).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  return f32_to_bf16_bits(lo) | (f32_to_bf16_bits(hi) << 16);
}

__device__ __forceinline__ bf16x2 as_bf16x2(uint32_t w) { return __builtin_bit_cast(bf16x2, w); }
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 w) { return __builtin_bit_cast(bf16x8, w); }

// Global-memory pointer of p.  Kernels pin their arguments in SGPRs with an
// empty asm statement (XATTN_PIN_VIEW below); a pointer that went through it
// has lost the address space the compiler inferred for kernel arguments, and
// accesses through it would become flat instructions (which also count
// against the LDS counter).  as_global() restores the global address space.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T *as_global(T *p) {
  return (__attribute__((address_space(1))) T *)p;
}

// 16-byte global-memory load and store.
__device__ __forceinline__ u32x4 load16(const uint16_t *p) {
  return *as_global(reinterpret_cast<const u32x4 *>(p));
}
__device__ __forceinline__ void store16(uint16_t *p, u32x4 v) { *as_global(reinterpret_cast<u32x4 *>(p)) = v; }

// DPP lane move within a 16-lane row (gfx9 encodings).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}
constexpr int kDppXor1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // lane i <-> 7-i within each 8-lane half row
constexpr int kDppMirror = 0x140;     // lane i <-> 15-i within each 16-lane row

// All-reduce over lanes {l, l ^ 16} / {l, l ^ 32} with the gfx950 permlane
// swaps.  A swap of x with itself returns x's even-row (lower-half) and
// odd-row (upper-half) copies in its two results; their sum / max is the
// reduction over the pair on every lane, in the same order on both lanes.
__device__ __forceinline__ float pair_sum16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pair_sum32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float pair_max16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pair_max32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
constexpr int kDppRowRor8 = 0x128;    // lane i <- lane (i + 8) mod 16 within each row

// All-reduce (sum) over aligned groups of N lanes, N in {8,16,32,64}.  Every lane
// of a group ends with the same value (each level adds a pair of equal partials).
template <int N>
__device__ __forceinline__ float group_sum(float x) {
  x += dpp_move<kDppXor1>(x);
  x += dpp_move<kDppXor2>(x);
  x += dpp_move<kDppHalfMirror>(x);
  if constexpr (N >= 16) x += dpp_move<kDppMirror>(x);
  if constexpr (N >= 32) x = pair_sum16(x);
  if constexpr (N >= 64) x += __shfl_xor(x, 32);
  return x;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Raw buffer resource over [base, base + bytes): the 64-bit base lives in
// scalar registers and loads take a 32-bit lane offset plus a scalar offset.
// Range checking makes a load at or past `bytes` return zero without a
// memory access.  0x00020000 is the descriptor's fourth dword on the gfx9
// family (32-bit data format, no swizzle).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
// Loads with cache policy sc0 (scope beyond the CU): they miss in the CU's L1
// and read the XCD's L2, i.e. data other CUs of the same XCD stored during
// this launch.
__device__ __forceinline__ u32x4 buffer_load16_l2(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voffset, 0, 1));
}
__device__ __forceinline__ u32x2 buffer_load8_l2(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voffset, 0, 1));
}

// Kernel arguments reach a wave through scalar loads from the kernarg
// segment.  The compiler issues each load next to its first use and may load a
// value again at a later use, so a prologue that reads its arguments in stages
// waits one memory round trip per stage.  A kernel therefore copies the
// arguments it needs into locals and ties them all to SGPRs in ONE empty asm
// statement (separate statements are scheduling boundaries, and the loads
// would again come in stages): one round trip, and later uses read the
// registers.  These macros spell the operand lists.
#define XATTN_PIN_VIEW(v) "+s"((v).p), "+s"((v).sb), "+s"((v).sh), "+s"((v).st)
#define XATTN_PIN_ROWSCHED(r)                                                                 \
  "+s"((r).batch), "+s"((r).count), "+s"((r).length), "+s"((r).item_begin), "+s"((r).nsplit), \
      "+s"((r).ntiles), "+s"((r).rec_begin)
#define XATTN_PIN_MERGEROW(r)                                                                 \
  "+s"((r).batch), "+s"((r).count), "+s"((r).nsplit), "+s"((r).item_begin), "+s"((r).tiles), \
      "+s"((r).rec_begin)
#define XATTN_PIN_BEGINS(l)                                                                   \
  "+s"((l).begin[0]), "+s"((l).begin[1]), "+s"((l).begin[2]), "+s"((l).begin[3]),             \
      "+s"((l).begin[4]), "+s"((l).begin[5]), "+s"((l).begin[6]), "+s"((l).begin[7])

// Row lookup over a kernarg row table sorted by item_begin.  load() reads the
// first eight item_begin values and row 0 (the tables always hold kMaxRows >= 8
// rows, so the reads stay inside the arguments), to be pinned with the caller's
// other arguments (XATTN_PIN_BEGINS and the row's list); find() then needs a
// second round trip only for an item of a row other than 0.  Past eight rows
// every lane loads one row's item_begin, one round trip more: a scan of the table
// waited for each cold line of two rows in turn (decode of 32 rows: 44.8 against
// 37.9 us for the kernel, 5.6 against 4.8 us for its merge).  Up to eight rows the
// values of the first round trip decide.
template <typename Row>
struct RowLookup {
  static_assert(kMaxRows >= 8, "row table");
  int begin[8];
  Row first;
  __device__ __forceinline__ void load(const Row *rows) {
#pragma unroll
    for (int k = 0; k < 8; ++k) begin[k] = rows[k].item_begin;
    first = rows[0];
  }
  // Every lane of the wave calls it.  UNIFORM: with the same item.
  template <bool UNIFORM = true>
  __device__ __forceinline__ Row find(const Row *rows, int nrows, int item) const {
    int r = 0;
#pragma unroll
    for (int k = 1; k < 8; ++k) r = (k < nrows && begin[k] <= item) ? k : r;
    if (nrows > 8) {
      const int lane = threadIdx.x & 63, mine = rows[lane].item_begin;
      if constexpr (UNIFORM) {
        r = __popcll(__ballot(lane < nrows && mine <= item)) - 1;
      } else {
        for (int k = 8; k < nrows; ++k) r = __builtin_amdgcn_readlane(mine, k) <= item ? k : r;
      }
    }
    return r == 0 ? first : rows[r];
  }
};

// Cache row that holds row b's K/V under a page table (the reference's paged
// FlashAttention call, compiler/common/kernels/attention.cpp:39-40, 68-70):
// blocks[b * stride] clamped into [0, rows), so that no table can address
// outside k/v; b itself without a table.  Kernels issue the read before their
// first K/V loads (for row b) and clamp and compare it where those loads are
// awaited anyway, reissuing them only when the page differs.  The read is a
// scalar load (constant address space, block-uniform address), so waiting
// for it never waits for vector loads.
__device__ __forceinline__ int read_page(const int32_t *blocks, int64_t stride, int b) {
  if (blocks == nullptr) return b;
  typedef const __attribute__((address_space(4))) int32_t *table_ptr;
  return ((table_ptr)blocks)[(int64_t)b * stride];
}
__device__ __forceinline__ int page_in_range(int page, int rows) { return min(max(page, 0), rows - 1); }

// Inclusive prefix sum over the 64 lanes (DPP row shifts, then row broadcasts).
__device__ __forceinline__ int wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);  // row_bcast:31 into rows 2 and 3
  return x;
}
__device__ __forceinline__ int wave_total(int x) { return __builtin_amdgcn_readlane(wave_scan(x), 63); }

// Row r's query count and KV length from the device offsets, clamped to the
// ranges the host validates in the default mode (see CaptureArgs in kernel_args.h).
__device__ __forceinline__ void capture_row(const CaptureArgs &c, int r, int &count, int &length) {
  const int32_t *cuq = c.offsets, *cuk = c.offsets + c.B + 1;
  count = min(max(cuq[r + 1] - cuq[r], 0), min(c.T, c.C));
  length = min(max(cuk[r + 1] - cuk[r], max(count, 1)), c.C);
}
// The same of a block-uniform row, in scalar loads of one round trip.
__device__ __forceinline__ void capture_row_uniform(const CaptureArgs &c, int r, int &count, int &length) {
  typedef const __attribute__((address_space(4))) int32_t *offsets_ptr;
  const offsets_ptr cuq = (offsets_ptr)c.offsets, cuk = cuq + c.B + 1;
  int q0 = cuq[r], q1 = cuq[r + 1], k0 = cuk[r], k1 = cuk[r + 1];
  asm volatile("" : "+s"(q0), "+s"(q1), "+s"(k0), "+s"(k1));
  count = min(max(q1 - q0, 0), min(c.T, c.C));
  length = min(max(k1 - k0, max(count, 1)), c.C);
}


// Splits of row `lane` of a graph-capture decode launch (every lane of the wave
// calls it), from the device lengths: the evenness rule (kernel_args.h: kDecodeCus)
// with a coarse search; every captured launch is merged by a launch, so what a merge in the
// launch would save does not enter.  Items take whole passes of a block, at
// least c.pass_min; there are never more than 4 * kDecodeCus + the (row, kv head)
// pairs, and no row takes more than c.splits_max splits (the records hold those).
__device__ __forceinline__ int capture_splits(const CaptureArgs &c, int lane, int count, int length) {
  const bool active = lane < c.B && count > 0;
  const int passes = active ? (length + c.pass_keys - 1) / c.pass_keys : 0;
  const int total = c.Hkv * wave_total(passes);
  // The fewest passes per item that leave at most `limit` items, up to one past
  // the most that keep `limit` items about even.
  auto most = [&](int limit) { return (int)((int64_t)total * kDecodeEvenNum / (limit * kDecodeEvenDen)) + 1; };
  auto least = [&](int limit, int up_to) {
    int m = max(c.pass_min, (total + limit - 1) / limit);
    while (m < up_to && c.Hkv * wave_total((passes + m - 1) / m) > limit) m += 1 + m / 8;
    return m;
  };
  const int m1 = least(kDecodeCus, most(kDecodeCus)), m2 = least(2 * kDecodeCus, most(2 * kDecodeCus));
  int m = 2 * m2 < m1 ? m2 : m1;
  if (m1 >= most(kDecodeCus) && m2 >= most(2 * kDecodeCus)) m = least(4 * kDecodeCus, most(kDecodeCus));
  return active ? min((passes + m - 1) / m, c.splits_max) : 1;
}

}  // namespace xattn
