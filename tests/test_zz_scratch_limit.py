"""Calls whose fastest plan needs more records than the allocation-free entry point's scratch.

The plan then gives way (capi.cpp, make_plan): longer decode items, or rows of 9 to
32 query vectors per KV head on the prefill kernel, whose records fit.  A call is
refused only if the prefill rows alone need more.  Each call here asks for a
workspace beyond the scratch, so it takes such a plan, and must run and hold the
float64 oracle's gates.
"""

import ctypes

import pytest
import torch

from attn_helpers import log
from test_zz_no_alloc import SCRATCH_BYTES, case, check_oracle, host_offsets, view

# (Hq, Hkv, D, counts, lengths)
CALLS = (
    (32, 4, 128, [6, 0, 1, 4, 5, 8, 4, 431, 0, 4, 2, 1, 7, 5],
     [237, 1814, 1814, 1817, 1602, 1499, 1817, 2244, 1814, 1817, 237, 21, 350, 146]),
    (32, 8, 128, [189, 4], [5211, 5026]),
    (32, 4, 128, [0, 4, 1, 0, 2, 1, 395, 4, 4, 2], [715, 1821, 10707, 150, 1434, 3296, 9910, 2794, 178, 351]),
)


def cpu_view(sizes):
    strides = (sizes[1] * sizes[2] * sizes[3], sizes[2] * sizes[3], sizes[3], 1)
    return type(view(torch.empty(1, 1, 1, 1)))(1 << 20, (ctypes.c_int64 * 4)(*sizes), (ctypes.c_int64 * 4)(*strides))


@pytest.mark.skipif(torch.cuda.is_available(), reason="without a device the call ends before any launch")
@pytest.mark.parametrize("heads,kv_heads,dim,counts,lengths", CALLS)
def test_not_refused(library_path, heads, kv_heads, dim, counts, lengths):
    torch.ops.load_library(str(library_path))
    lib = ctypes.CDLL(str(library_path))
    lib.xinfer_batched_flash_attention_workspace_size.restype = ctypes.c_size_t
    q = cpu_view([len(counts), heads, max(counts), dim])
    k = cpu_view([len(counts), kv_heads, max(lengths), dim])
    host = host_offsets(counts, lengths)
    assert lib.xinfer_batched_flash_attention_workspace_size(ctypes.byref(q), ctypes.byref(k), host) > SCRATCH_BYTES
    status = lib.xinfer_batched_flash_attention_noalloc(ctypes.byref(q), ctypes.byref(k), ctypes.byref(k), host, None,
                                                        ctypes.c_int64(0), ctypes.c_double(dim ** -0.5),
                                                        ctypes.c_void_p(1 << 20), None)
    assert status == 13  # no device to launch on; not 17, the refusal


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv_heads,dim,counts,lengths", CALLS)
@torch.inference_mode()
def test_runs_within_the_gates(library_path, heads, kv_heads, dim, counts, lengths):
    lib = ctypes.CDLL(str(library_path))
    log(f"scratch limit: Hq={heads} Hkv={kv_heads} D={dim} counts={counts} lengths={lengths}")
    q, k, v = case(9, len(counts), heads, kv_heads, dim, max(lengths), counts, lengths)
    qv, kv, vv = view(q), view(k), view(v)
    out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    status = lib.xinfer_batched_flash_attention_noalloc(ctypes.byref(qv), ctypes.byref(kv), ctypes.byref(vv),
                                                        host_offsets(counts, lengths), None, ctypes.c_int64(0),
                                                        ctypes.c_double(dim ** -0.5), ctypes.c_void_p(out.data_ptr()),
                                                        stream)
    assert status == 0
    torch.cuda.synchronize()
    check_oracle(out, q, k, v, counts, lengths, dim ** -0.5)
