"""Which kernels serve a mixed batch, and that its rows hold the oracle's gates on each route.

Rows of 9 to 32 query vectors per KV head beside prefill rows take the decode kernel
or, with small heads or short keys, the prefill kernel (capi.cpp, decode_vector_limit);
decode and prefill rows take one launch or two (one_launch_pays).
"""

import pytest
import torch

from attn_helpers import log
from test_many_rows_gpu import check
from xinfer_amd.attention import batched_attention_metadata

pytestmark = pytest.mark.gpu

ONE, TWO, PREFILL = {"attention_both"}, {"decode", "prefill"}, {"prefill"}
# (Hq, Hkv, D, counts, lengths, kernels)
CASES = [
    # Short rows: head dim 64, all short; a longer row; prefill rows that fill the chip.
    (8, 8, 64, [77, 201, 13], [77, 201, 13], PREFILL),
    (8, 8, 64, [200, 24, 24], [200, 1024, 500], PREFILL),
    (8, 8, 64, [200, 24, 24], [200, 1025, 500], ONE),
    (8, 8, 64, [512, 300] + [24] * 4, [3000, 2000] + [2000] * 4, PREFILL),
    # Two query heads per KV head, no key split; one split; four heads.
    (16, 8, 128, [200, 12, 12], [200, 512, 40], PREFILL),
    (16, 8, 128, [200, 12, 12], [200, 513, 40], ONE),
    (32, 8, 128, [200, 6, 6], [200, 512, 40], ONE),
    (16, 4, 256, [200, 6, 6], [200, 512, 40], ONE),
    # Rows of 17-32 vectors alone: few keys, and one row of more; up to 16 vectors; head dim 128.
    (16, 4, 256, [8, 5], [8, 128], PREFILL),
    (16, 4, 256, [8, 5], [8, 129], {"decode"}),
    (16, 4, 256, [4, 3], [8, 128], {"decode"}),
    (8, 8, 64, [32, 20], [48, 20], PREFILL),
    (8, 8, 64, [32, 20], [49, 20], {"decode"}),
    (16, 8, 128, [16, 9], [16, 9], {"decode"}),
    # More short rows than the prefill kernel's blocks take at once.
    (16, 4, 256, [8] * 64, [60] * 64, PREFILL),
    (16, 4, 256, [8] * 64 + [7], [60] * 65, {"decode"}),
    (16, 8, 128, [200] + [12] * 24, [200] + [300] * 24, PREFILL),
    (16, 8, 128, [200] + [12] * 25, [200] + [300] * 25, ONE),
    (8, 8, 64, [200] + [24] * 25, [200] + [300] * 25, ONE),
    (8, 8, 64, [512, 300] + [24] * 11, [3000, 2000] + [6000] * 11, {"decode", "prefill"}),
    # Decode rows beside few prefill items, many of them; beside prefill items that fill the chip.
    (8, 8, 64, [200] + [1] * 4, [200, 3000, 40, 700, 2000], ONE),
    (16, 8, 128, [200] + [1] * 7, [200] + [2000] * 7, ONE),
    (16, 4, 256, [200] + [1] * 20, [200] + [6000] * 20, TWO),
    (16, 8, 128, [64] + [1] * 8, [64] + [8000] * 8, TWO),
    (8, 8, 64, [64] + [1] * 8, [64] + [8000] * 8, TWO),
    (16, 8, 128, [512, 300] + [1] * 6, [3000, 2000] + [3000] * 6, TWO),
]


@pytest.mark.parametrize("heads,kv_heads,dim,counts,lengths,kernels", CASES)
@torch.inference_mode()
def test_kernels_of_a_mixed_batch(gpu_ops, heads, kv_heads, dim, counts, lengths, kernels):
    log(f"mixed route Hq={heads} Hkv={kv_heads} D={dim} counts={counts} lengths={lengths}")
    check(gpu_ops, heads, kv_heads, dim, counts, lengths, max(lengths) + 3)
    q = torch.randn(len(counts), heads, max(counts), dim, device="cuda").to(torch.bfloat16)
    k = torch.randn(len(counts), kv_heads, max(lengths), dim, device="cuda").to(torch.bfloat16)
    host, cu, blocks = batched_attention_metadata(
        torch.tensor(lengths, dtype=torch.int32), torch.tensor(counts, dtype=torch.int32), "cuda")
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as profile:
        gpu_ops.batched_flash_attention(q, k, k, host, cu, blocks, dim ** -0.5)
        torch.cuda.synchronize()
    names = [e.name.split("xattn::")[1].split("_kernel")[0] for e in profile.events() if "xattn::" in e.name]
    assert {name.removesuffix("_d256") for name in names if "merge" not in name} == kernels, names
