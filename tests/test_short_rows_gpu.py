"""Rows of few query vectors: the decode kernel's columns, tiles and splits.

A row of up to 32 query vectors per KV head takes the decode kernel, whose
16-column groups hold up to 5 vectors with fp32 weights (three columns each) or
16 with bf16 weights in one group, 8 or 32 in two.  The rows here have the
vector counts on both sides of each of those limits (33 takes the prefill kernel
beside them), and lengths around a wave's tile (64, 32, 16 keys for padded head
dims 64, 128, 256), a block's pass (four tiles) and several splits.  Keys past a
row's length and queries past its count are NaN, K, V and Q are views of wider
rows.  Each result is held to the float64 oracle by the gates of the other
parity tests, and a repeat must give the same bits.
"""

import numpy as np
import pytest
import torch

from attn_helpers import MAX_ABS, MEAN_ABS, log, row_errors
from oracle import attention as oracle
from xinfer_amd.attention import batched_attention_metadata

pytestmark = pytest.mark.gpu

# (name, Hq, Hkv, counts, lengths as (passes, tiles, keys) beyond the count, capacity)
CASES = (
    ("one_vector_groups", 3, 3, [5, 6, 8, 9, 16, 17, 32, 33],
     [(0, 1, -5), (1, 0, -6), (1, 0, 0), (2, 1, 1), (0, 0, 0), (3, 0, 3), (4, 2, -1), (1, 0, 0)]),
    ("exact_weights", 8, 4, [1, 2, 3, 4, 0, 1], [(0, 0, 0), (0, 1, -1), (1, 0, 1), (9, 1, 2), (0, 1, 0), (5, 3, -1)]),
    ("wide_rows_only", 16, 4, [3, 4, 5, 8, 7], [(0, 1, 0), (6, 0, -1), (2, 0, 1), (3, 2, 5), (12, 0, 0)]),
)


def view(shape, dim, generator):
    wide = torch.full((*shape, dim + 8), float("nan"), dtype=torch.bfloat16)
    wide[..., :dim] = torch.randn(*shape, dim, generator=generator).to(torch.bfloat16)
    return wide.cuda()[..., :dim]


def f64(x):
    return torch.nan_to_num(x.detach().float(), nan=0.0).cpu().numpy().astype(np.float64)


@pytest.mark.parametrize("dim", (64, 72, 128, 256))
@pytest.mark.parametrize("name,heads,kv_heads,counts,places", CASES, ids=[c[0] for c in CASES])
@torch.inference_mode()
def test_vector_counts_and_tiles(gpu_ops, dim, name, heads, kv_heads, counts, places):
    tile = 64 if dim <= 64 else (32 if dim <= 128 else 16)
    lengths = [n + max(0, p * 4 * tile + t * tile + k) + (n == 0) for n, (p, t, k) in zip(counts, places)]
    capacity = max(lengths) + 5  # not a multiple of 256: no page table
    log(f"short rows {name} D={dim}: Hq={heads} Hkv={kv_heads} counts={counts} lengths={lengths}")
    generator = torch.Generator().manual_seed(dim + len(name))
    batch, tokens = len(counts), max(counts)
    q = view((batch, heads, tokens), dim, generator)
    k, v = (view((batch, kv_heads, capacity), dim, generator) for _ in range(2))
    for r, (count, length) in enumerate(zip(counts, lengths)):
        k[r, :, length:], v[r, :, length:], q[r, :, count:] = float("nan"), float("nan"), float("nan")
    host, cu, blocks = batched_attention_metadata(
        torch.tensor(lengths, dtype=torch.int32), torch.tensor(counts, dtype=torch.int32), "cuda")
    out = gpu_ops.batched_flash_attention(q, k, v, host, cu, blocks, dim ** -0.5).cpu()
    expected = oracle.attention(f64(q), f64(k), f64(v), counts, lengths, dim ** -0.5)
    for r, count in enumerate(counts):
        assert torch.count_nonzero(out[r, :, count:]).item() == 0
        if count:
            errors = row_errors(out[r:r + 1, :, :count].float().flatten(1),
                                torch.from_numpy(expected[r:r + 1, :, :count]).float().flatten(1))
            assert errors["max_abs"] <= MAX_ABS and errors["mean_abs"] <= MEAN_ABS, (r, errors)
            assert errors["relative_l2"] < 0.01 and errors["peak_relative"] <= 0.05, (r, errors)
    again = gpu_ops.batched_flash_attention(q, k, v, host, cu, blocks, dim ** -0.5).cpu()
    assert torch.equal(again.view(torch.int16), out.view(torch.int16))


@pytest.mark.parametrize("dim", (64, 128, 256))
@torch.inference_mode()
def test_infinite_values_stay_infinite(gpu_ops, dim):
    """An infinite value times the zero remainder of an exact weight is no NaN."""
    lengths = [1, 40, 700]
    log(f"infinite values D={dim} lengths={lengths}")
    generator = torch.Generator().manual_seed(dim)
    q = torch.randn(3, 4, 1, dim, generator=generator).to(torch.bfloat16).cuda()
    k, v = (torch.randn(3, 2, 704, dim, generator=generator).to(torch.bfloat16).cuda() for _ in range(2))
    v[:, :, 0, 3], v[:, :, 0, dim - 1] = float("inf"), float("-inf")
    host, cu, blocks = batched_attention_metadata(
        torch.tensor(lengths, dtype=torch.int32), torch.ones(3, dtype=torch.int32), "cuda")
    out = gpu_ops.batched_flash_attention(q, k, v, host, cu, blocks, dim ** -0.5).cpu().float()
    assert (out[..., 3] == float("inf")).all() and (out[..., dim - 1] == float("-inf")).all()
    rest = [d for d in range(dim) if d not in (3, dim - 1)]
    assert torch.isfinite(out[..., rest]).all()
