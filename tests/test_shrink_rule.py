"""Which segment shrinks split K over workgroups, by the workspace they ask
for (split sums), on the 256 CUs the library assumes without a GPU."""

import pytest

from multi_lora_amd import _ffi

F32, F16, BF16 = 0, 1, 2


def split_bytes(in_dim, r_max, n, rows, bs, max_len, dtype):
    return _ffi.lib().mlora_shrink_workspace_bytes(in_dim, r_max, n, rows, bs, max_len, dtype)


def test_codes():
    import torch
    assert [_ffi.dtype_code(t) for t in (torch.float32, torch.float16, torch.bfloat16)] == [F32, F16, BF16]


@pytest.mark.parametrize("name,in_dim,r_max,n,rows,bs,max_len,dtype,split", [
    # Two prompts and 64 decode rows: half of the tiles hold one row, and the
    # expand adds the split sums itself.
    ("mixed o", 4096, 16, 1, 1088, 66, 512, BF16, True),
    ("mixed gate|up", 4096, 16, 2, 1088, 66, 512, BF16, True),
    ("mixed q|k|v", 4096, 16, 3, 1088, 66, 512, BF16, True),
    ("mixed, short K", 1024, 16, 1, 1088, 66, 512, BF16, False),
    # Long segments.
    ("one prompt, rank 16", 4096, 16, 1, 203, 1, 203, BF16, False),
    ("one prompt, rank 64", 4096, 64, 1, 203, 1, 203, BF16, True),
    ("prompts on every CU", 4096, 8, 1, 3900, 13, 300, BF16, True),
    ("prompts on every CU, short K", 2048, 32, 1, 3900, 13, 300, BF16, False),
    # fp32: few large tiles split, small ones and many do not.
    ("fp32, few rows, long K", 8192, 8, 1, 17, 1, 17, F32, True),
    ("fp32, few rows", 2048, 8, 1, 17, 1, 17, F32, False),
    ("fp32 prompts", 8192, 64, 1, 3900, 13, 300, F32, False),
    # K not made of 16-byte chunks.
    ("odd K, few rows", 14001, 8, 1, 17, 1, 17, BF16, True),
    ("odd K, prompts", 4101, 64, 1, 4075, 8, 1024, F16, True),  # the aligned plan of this size splits
])
def test_split_or_whole(name, in_dim, r_max, n, rows, bs, max_len, dtype, split):
    assert (split_bytes(in_dim, r_max, n, rows, bs, max_len, dtype) > 0) is split, name


def test_the_query_covers_rows_that_turn_out_unaligned():
    # Aligned, this decode-shaped call runs whole (200 tiles); from rows off a
    # 16-byte boundary it splits.
    assert split_bytes(4096, 20, 1, 200, 200, 1, BF16) > 0
