"""The fused norm + RoPE + append over token counts: both launch shapes of the kernel.

From 2048 tokens the kernel takes other blocks and does not read the keys and
values of padded tokens.  The head counts here leave tasks with unused lanes
(a wave takes 512 / dim heads of one kind).  Values and untouched slots are
compared bit for bit with the oracle.  For the rotated elements the sum of
squares may differ in its last bit, which flips few roundings (under 1% of the
elements): one of y (2^-7 of it), hence one more of w * y, so xn differs by at most
2 * 2^-7 |xn|; its products p = xn cos and q = rot sin by that and one rounding
of each, their sum by one more: 4 * 2^-7 (|p| + |q|) in all, to first order, which
in units of a result that p and q nearly cancel in can be many.
"""

import numpy as np
import pytest
import torch

from oracle import norm_rope as ref
from test_norm_rope import bits, draw


@pytest.mark.gpu
@torch.inference_mode()
@pytest.mark.parametrize("dim,heads,kv_heads", [(64, 9, 3), (128, 5, 5), (256, 3, 1)])
@pytest.mark.parametrize("batch,tokens", [(1, 1), (1, 2047), (4, 512), (2048, 1)])
def test_token_counts_against_the_oracle(gpu_ops, batch, tokens, dim, heads, kv_heads):
    from attn_helpers import log
    from xinfer_amd.norm_rope import qk_norm_rope_append

    log(f"norm/rope/append tokens {batch}x{tokens} heads={heads}/{kv_heads} dim={dim}")
    capacity = max(tokens, 8)
    inputs = draw(5, batch, tokens, heads, kv_heads, dim)
    counts = [(tokens * (r % 4 + 1) + 3) // 4 if r % 5 else 0 for r in range(1, batch + 1)]
    positions = torch.arange(tokens).repeat(batch, 1)
    positions[:, -1] = torch.tensor([capacity, -1] * batch)[:batch]  # outside the cache
    cu = torch.tensor([0] + list(np.cumsum(counts)), dtype=torch.int32)
    g = torch.Generator().manual_seed(6)
    caches = [torch.randn(batch, kv_heads, capacity, dim, generator=g).to(torch.bfloat16) for _ in range(2)]
    got_k, got_v = (c.cuda() for c in caches)
    q, k, v, qw, kw, cos, sin = (t.cuda() for t in inputs)
    q_out = qk_norm_rope_append(q, k, v, qw, kw, 1e-6, cos, sin, positions.cuda(), cu.cuda(), got_k, got_v)

    want_k, want_v = (bits(c).copy() for c in caches)
    q, k, v, qw, kw, cos, sin = (bits(t) for t in inputs)
    want_q = ref.norm_rope_append(q, k, v, qw, kw, 1e-6, cos, sin, positions.numpy(), cu.numpy(), want_k, want_v)

    def terms(x, w):
        xn = np.abs(ref.bf16_to_f32(ref.rms_norm(x, w, 1e-6))).transpose(0, 2, 1, 3)
        c, s = (np.abs(ref.bf16_to_f32(t))[:, None] for t in (cos, sin))
        return xn * c + np.roll(xn, dim // 2, axis=-1) * s

    def check(actual, expected, size):
        a, e = ref.bf16_to_f32(actual), ref.bf16_to_f32(expected)
        assert (np.abs(a - e) <= 4.1 * 2.0**-7 * size).all() and (a != e).mean() < 0.01

    check(bits(q_out.cpu()), want_q, terms(q, qw))
    key_terms, sizes = terms(k, kw), np.zeros(want_k.shape, np.float32)
    for r in range(batch):
        for t in range(counts[r]):
            if 0 <= positions[r, t] < capacity:
                sizes[r, :, positions[r, t]] = np.maximum(sizes[r, :, positions[r, t]], key_terms[r, :, t])
    check(bits(got_k.cpu()), want_k, sizes)
    assert np.array_equal(bits(got_v.cpu()), want_v)


@pytest.mark.gpu
@torch.inference_mode()
@pytest.mark.parametrize("dim,heads,kv_heads", [(64, 70, 9), (128, 32, 8), (256, 16, 4)])
@pytest.mark.parametrize("batch,tokens", [(1, 3), (383, 1), (3, 128), (1, 385)])
def test_tasks_spread_over_blocks(gpu_ops, batch, tokens, dim, heads, kv_heads):
    """More than eight tasks a token: below 384 tokens over several blocks, above in one block's turns."""
    test_token_counts_against_the_oracle(gpu_ops, batch, tokens, dim, heads, kv_heads)
