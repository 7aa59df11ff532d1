"""Which segment shrinks split K over workgroups (CPU only).

A call that splits needs a workspace for its split sums and is turned down
without one; any other goes on to its launch, which fails here for want of a
device before it touches the placeholder addresses.  The library assumes 256
CUs without a GPU.
"""

import ctypes

import pytest
import torch

from multi_lora_amd import _ffi
from tests import test_gpu_segments

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="launches on placeholder addresses")

F32, F16, BF16 = (_ffi.dtype_code(t) for t in (torch.float32, torch.float16, torch.bfloat16))
WORKSPACE = -3


def query(in_dim, r_max, n, rows, bs, max_len, dtype):
    return _ffi.lib().mlora_shrink_workspace_bytes(in_dim, r_max, n, rows, bs, max_len, dtype)


def splits(in_dim, r_max, n, rows, bs, max_len, dtype, offset=0):
    """offset: bytes the rows of x are off a 16-byte boundary."""
    meta = _ffi.SegMeta(256, 512, 768, 1024, bs, max_len, 4, BF16)
    sl = _ffi.SliceArray()
    for i in range(n):
        sl[i].a, sl[i].a_slot_stride, sl[i].a_row_stride = (i + 1) << 40, r_max * in_dim, in_dim
    rc = _ffi.lib().mlora_shrink((1 << 45) + offset, in_dim, rows, in_dim, sl, n, r_max, 1, 1 << 46, n * r_max,
                                 ctypes.byref(meta), dtype, None, 0, None)
    assert rc == WORKSPACE or rc > 0, _ffi.lib().mlora_last_error()
    return rc == WORKSPACE


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
    ("fp32 decode", 4096, 32, 3, 256, 256, 1, F32, False),
    ("fp32 decode, few rows", 4096, 32, 1, 8, 8, 1, F32, True),
    # K not made of 16-byte chunks.
    ("odd K, few rows", 14001, 8, 1, 17, 1, 17, BF16, True),
    ("odd K, one prompt", 4101, 8, 1, 203, 1, 203, BF16, False),
    ("odd K, prompts", 4101, 64, 1, 4075, 8, 1024, F16, False),
    ("odd K, mixed, several blocks", 14001, 64, 1, 1088, 66, 512, BF16, False),
    ("odd K, mixed, one block", 14001, 8, 1, 1088, 66, 512, BF16, True),
])
def test_split_or_whole(name, in_dim, r_max, n, rows, bs, max_len, dtype, split):
    assert splits(in_dim, r_max, n, rows, bs, max_len, dtype) is split, name
    if split:
        assert query(in_dim, r_max, n, rows, bs, max_len, dtype) > 0


@pytest.mark.parametrize("shape", [
    (4096, 20, 1, 200, 200, 1),    # decode-shaped on 200 CUs
    (14336, 16, 1, 300, 1, 300),   # planned in 128-row tiles when aligned
    (4096, 16, 1, 17, 1, 17),
])
def test_the_query_covers_rows_that_turn_out_unaligned(shape):
    for offset in (0, 2):
        if splits(*shape, BF16, offset):
            assert query(*shape, BF16) > 0
    assert splits(*shape, BF16, 2)


# Cases of the GPU tests that stand for split sums, added by the expand or
# reduced into a private mid.
SPLIT_CASES = {"mixed", "mixed_r64", "decode_split", "long", "rmax4_split", "rmax4_split_f16", "rmax12_split",
               "rmax12_mixed_bf16", "qkv_r64_mixed", "qkv_r64_decode", "qkv_r64_long", "long_k8192",
               "long_k14336_f16", "wide_mixed", "long_ranks", "narrow_split", "r64_f16", "r64_streamed"}


def gpu_cases():
    out = list(test_gpu_segments.MIXED_CASES)
    for f in (test_gpu_segments.test_one_call_equals_two_calls, test_gpu_segments.test_apply_ignores_what_the_workspace_held):
        out += [c for m in f.pytestmark if m.name == "parametrize" and "in_dim" in m.args[0] for c in m.args[1]]
    return out


def test_gpu_cases_of_split_sums_are_split():
    seen = set()
    for name, lens, _, _, in_dim, outs, r_max, dtype in gpu_cases():
        if name in SPLIT_CASES:
            seen.add(name)
            assert splits(in_dim, r_max, len(outs), sum(lens), len(lens), max(lens), _ffi.dtype_code(dtype)), name
    assert seen == SPLIT_CASES
