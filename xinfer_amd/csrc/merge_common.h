// The fold of split records, shared by the merge launch (merge.hip) and the decode
// launch's own merge (decode_item.h), so that both give the same bits.
#pragma once

#include "device_common.h"

namespace xattn {

// A running max (log2 units), sum and unnormalised quad of output features.
struct MergeState {
  float m, l;
  f32x4 o;
};

// The products that are fused are written out, so that no compiler chooses
// others in one of the kernels.
__device__ __forceinline__ void fold(MergeState &st, float ms, float ls, f32x4 os) {
  if (ms == -INFINITY) return;
  const float mn = fmaxf(st.m, ms);
  const float a = fast_exp2(st.m - mn), w = fast_exp2(ms - mn);  // st.m = -inf -> a = 0
  st.l = __builtin_fmaf(st.l, a, ls * w);
  st.o = f32x4{__builtin_fmaf(os.x, w, st.o.x * a), __builtin_fmaf(os.y, w, st.o.y * a),
               __builtin_fmaf(os.z, w, st.o.z * a), __builtin_fmaf(os.w, w, st.o.w * a)};
  st.m = mn;
}

}  // namespace xattn
