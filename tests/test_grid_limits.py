"""Calls near the launch limits (CPU only: without a device every launch fails
before it touches the placeholder addresses, and says why)."""

import ctypes

import pytest
import torch

from multi_lora_amd import _ffi

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="launches on placeholder addresses")

INVALID_CONFIGURATION = 9


def test_fused_norm_of_many_short_rows_is_not_too_tall_a_grid():
    """700,000 rows of 256 elements over 2,000 entries: one shrink item an
    entry, so with the items next to each other the norm row blocks alone
    would fill more than 65,535 rows of the grid."""
    rows, k, r = 700_000, 256, 16
    meta = _ffi.SegMeta(256, 512, 768, 1024, 2000, 350, 2000, _ffi.MLORA_BF16)
    meta.plan, meta.plan_cap, meta.plan_entries = 1 << 40, 50_000, 2000
    sl = _ffi.SliceArray()
    sl[0].a, sl[0].a_slot_stride, sl[0].a_row_stride = 1 << 41, r * k, k
    sl[0].b, sl[0].b_slot_stride, sl[0].b_row_stride, sl[0].out_dim = 1 << 42, 256 * r, r, 256
    lib = _ffi.lib()
    need = lib.mlora_grouped_workspace_bytes(k, r, 1, rows, 2000, _ffi.MLORA_BF16, 2)
    assert need > 0
    rc = lib.mlora_rmsnorm_apply_grouped(1 << 43, k, rows, k, 1 << 44, 1e-5, 1 << 45, k, sl, 1, r, 1 << 46, 256,
                                         ctypes.byref(meta), _ffi.MLORA_BF16, 1 << 47, need, 1, None)
    assert rc > 0 and rc != INVALID_CONFIGURATION, lib.mlora_last_error()


def test_decode_attention_counts_its_512_threads():
    """More workgroups than fit a launch's 2^32 work-items are turned down
    before anything else is looked at (null pointers here)."""
    lib = _ffi.lib()

    def call(batch):
        return lib.mlora_decode_attention(None, 64, None, 64, None, 64, None, None, 0, None, None, None, 0, None, None,
                                          64, batch, 1, 1, 64, 8, 0.125, _ffi.MLORA_BF16, None)

    most = (2 ** 32 - 1) // 512
    assert call(most) == -1 and b"null" in lib.mlora_last_error()
    assert call(most + 1) == -2
