"""The planner's decode items and merges, read from the workspace a call asks for.

The workspace holds D floats and two for (m, l) per record, each part rounded up to
256 bytes, and 8 bytes per item where the decode launch merges its own split rows.
Passes of an item: 256, 128, 64 keys for padded head dims 64, 128, 256.
"""

import ctypes

import pytest

from test_library_cpu import decode_workspace, expected_workspace, lib  # noqa: F401

CASES = [
    # (name, counts, lengths, Hq, Hkv, D, passes per item, merged in the launch)
    # One one-pass item per CU, and one row's more: two passes each.
    ("256_items", [1] * 8, [1024] * 3 + [1] * 3 + [300, 130], 16, 8, 128, 1, True),
    ("264_items", [1] * 8, [1024] * 3 + [1] * 3 + [300, 300], 16, 8, 128, 2, True),
    # 32 short rows, 864 items of one pass: long items, merged in the launch, not four per CU and a launch.
    ("short_rows", [1] * 32, [23 * r + 11 for r in range(32)], 16, 8, 128, 2, True),
    ("short_rows_d64", [1] * 16, [187 * r + 100 for r in range(16)], 8, 8, 64, 4, True),
    # A merge launch for each: KV heads that are no multiple of 8; one long row.
    ("four_kv_heads", [1] * 4, [1024, 4096, 8192, 16384], 16, 4, 256, 8, False),
    # Rows of many vectors: by the length of the fold.
    ("short_fold", [8] * 16, [420] * 16, 32, 8, 256, 4, True),
    ("long_fold", [8], [380], 32, 8, 256, 1, False),
]


@pytest.mark.parametrize("name,counts,lengths,heads,kv_heads,dim,passes,in_launch", CASES, ids=[c[0] for c in CASES])
def test_items_and_merge(lib, name, counts, lengths, heads, kv_heads, dim, passes, in_launch):  # noqa: F811
    keys = passes * {64: 256, 128: 128, 256: 64}[dim]
    splits = [-(-length // keys) for length in lengths]
    group = heads // kv_heads
    records = kv_heads * sum(s * n * group for s, n in zip(splits, counts) if s > 1)
    counters = kv_heads * sum(splits) if in_launch else 0
    assert decode_workspace(lib, counts, lengths, heads, kv_heads, dim, 16384) == expected_workspace(records, dim,
                                                                                                      counters)


def test_rows_on_both_sides_of_the_multiplied_division(lib):  # noqa: F811
    """34 million keys: 2^19 passes at head dim 256, where the planner goes on to divide."""
    for passes in ((1 << 19) - 5, (1 << 19) + 5):
        length = 64 * passes
        assert decode_workspace(lib, [1], [length], 1, 1, 256, length) == expected_workspace(512, 256, 0)
