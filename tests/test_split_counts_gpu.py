"""Rows of very many key splits: every layout of the merge launch against the oracle.

Past 64 splits a block folds a slice of a vector's features (all of them at head dim
64), past 256 with twice the threads; the lanes' batches hold 16 records.
"""

import pytest
import torch

from attn_helpers import log
from test_many_rows_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,dim,length", [(8, 8, 64, 20000), (8, 1, 64, 20001), (2, 1, 64, 66000),
                                                       (4, 1, 128, 20000), (4, 1, 256, 20001)])
@torch.inference_mode()
def test_one_long_row(gpu_ops, heads, kv_heads, dim, length):
    log(f"one long row Hq={heads} Hkv={kv_heads} D={dim} length={length}")
    check(gpu_ops, heads, kv_heads, dim, [1], [length], length + 3)
