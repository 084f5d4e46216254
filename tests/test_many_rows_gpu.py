"""Launches of more than eight rows: the row of a work item found from one load per lane.

Nine and 64 rows fill one launch, 67 take two; items of every row occur, first and
last, of decode rows, split prefill rows and merges (one vector per block and
several).  Every row is held to the float64 oracle by the gates of the other parity
tests.
"""

import pytest
import torch

from attn_helpers import MAX_ABS, MEAN_ABS, log, row_errors
from oracle import attention as oracle
from test_short_rows_gpu import f64
from xinfer_amd.attention import batched_attention_metadata

pytestmark = pytest.mark.gpu


def check(gpu_ops, heads, kv_heads, dim, counts, lengths, capacity):
    generator = torch.Generator().manual_seed(len(counts))
    q = torch.randn(len(counts), heads, max(counts), dim, generator=generator).to(torch.bfloat16)
    k, v = (torch.randn(len(counts), kv_heads, capacity, dim, generator=generator).to(torch.bfloat16)
            for _ in range(2))
    host, cu, blocks = batched_attention_metadata(
        torch.tensor(lengths, dtype=torch.int32), torch.tensor(counts, dtype=torch.int32), "cuda")
    out = gpu_ops.batched_flash_attention(q.cuda(), k.cuda(), v.cuda(), host, cu, blocks, dim ** -0.5).cpu()
    expected = oracle.attention(f64(q), f64(k), f64(v), counts, lengths, dim ** -0.5)
    for r, count in enumerate(counts):
        assert torch.count_nonzero(out[r, :, count:]).item() == 0
        if count == 0:
            continue
        errors = row_errors(out[r:r + 1, :, :count].float().flatten(1),
                            torch.from_numpy(expected[r:r + 1, :, :count]).float().flatten(1))
        assert errors["max_abs"] <= MAX_ABS and errors["mean_abs"] <= MEAN_ABS, (r, errors)
        assert errors["relative_l2"] < 0.01 and errors["peak_relative"] <= 0.05, (r, errors)


@pytest.mark.parametrize("rows", (9, 64, 67))
@pytest.mark.parametrize("what", ("decode", "mixed", "prefill"))
@pytest.mark.parametrize("dim", (64, 256))
@torch.inference_mode()
def test_every_row_of_a_launch(gpu_ops, rows, what, dim):
    heads, kv_heads, capacity = (8, 8, 1501) if what == "decode" else (4, 1, 1501)
    counts = [{"decode": 1, "mixed": (1, 40, 2)[r % 3], "prefill": 33 + r % 5}[what] for r in range(rows)]
    lengths = [n + (r * 389 + (0 if r % 2 else 1100)) % (capacity - 40) for r, n in enumerate(counts)]
    log(f"rows of a launch {what} rows={rows} D={dim} Hq={heads} Hkv={kv_heads}")
    check(gpu_ops, heads, kv_heads, dim, counts, lengths, capacity)


@pytest.mark.parametrize("dim", (64, 72, 128, 256))
@torch.inference_mode()
def test_decode_and_prefill_rows_merge_together(gpu_ops, dim):
    """Decode rows of more than eight splits (and of fewer) beside split prefill rows."""
    counts, lengths = [1, 40, 2, 33, 1, 65], [3000, 2900, 2400, 1500, 700, 513]
    log(f"merge of both kinds D={dim} counts={counts} lengths={lengths}")
    check(gpu_ops, 12, 3, dim, counts, lengths, 3001)


@pytest.mark.parametrize("dim", (64, 72, 128, 256))
@pytest.mark.parametrize("counts,lengths", [
    ([0, 96, 1, 1, 5, 130], [9, 900, 1, 700, 200, 1301]),  # one launch; an odd number of decode items, a row without queries
    ([1, 1, 70], [40, 33, 70]),                            # one item a head, no splits
    ([1] * 40 + [40] * 3, [1100] * 40 + [50, 60, 70]),     # two launches: the decode rows take longer
])
@torch.inference_mode()
def test_decode_and_prefill_rows_launch_together(gpu_ops, dim, counts, lengths):
    log(f"launch of both kinds D={dim} counts={counts} lengths={lengths}")
    check(gpu_ops, 6, 3, dim, counts, lengths, 1303)
