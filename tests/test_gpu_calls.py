"""The native form of the ordinary calls (multi_lora_amd/_calls.so, GPU)
against the general Python path it stands in for: the same bits where it
takes a call, and calls that are not plain are left to the Python path."""

import pytest
import torch

from multi_lora_amd import HipLoRABackend, _ffi, synthetic
from multi_lora_amd.kernels import fused_add_rmsnorm, rmsnorm_fwd, sgemm_lora_a_fwd, sgemm_lora_b_fwd
from multi_lora_amd.kernels.lora_ops import (LinkedWorkspace, Workspace, apply_grouped, apply_segments, expand,
                                             rmsnorm_apply_grouped, shrink)

pytestmark = pytest.mark.gpu


def decode(dev, dtype=torch.bfloat16):
    return synthetic.decode_qkv(device=dev, dtype=dtype, tokens=37, hidden=1024, outs=[512, 256, 256], n_slots=12,
                                n_adapters=9, rank=16)


def prompts(dev, dtype=torch.bfloat16):
    return synthetic.prefill_mlp(device=dev, dtype=dtype, part="gate_up", n_seg=3, min_len=20, max_len=90, hidden=512,
                                 inter=768, r_max=32)


def taken(wl, out, x=None, a=None, b=None, cols=None, linked=None, seg=None):
    return _ffi.calls().apply_multi(wl.x if x is None else x, a or wl.a_stacks, b or wl.b_stacks, wl.meta, out, cols,
                                    linked or LinkedWorkspace(), seg or Workspace())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("make,general", [(decode, "grouped"), (prompts, "segments")])
def test_native_apply_gives_the_general_paths_bits(dev, make, general, dtype):
    wl = make(dev, dtype)
    got, want = wl.clone_base(), wl.clone_base()
    for cols in (None, wl.col_offsets, tuple(wl.col_offsets)):
        got.copy_(wl.base)
        assert taken(wl, got, a=tuple(wl.a_stacks), cols=cols) is True
        want.copy_(wl.base)
        if general == "segments" or not apply_grouped(wl.x, wl.a_stacks, wl.b_stacks, wl.meta, want, wl.col_offsets,
                                                      workspace=LinkedWorkspace()):
            apply_segments(wl.x, wl.a_stacks, wl.b_stacks, wl.meta, want, wl.col_offsets, workspace=Workspace())
        assert torch.equal(got, want)


def test_calls_that_are_not_plain_are_left_to_python(dev):
    wl = decode(dev)
    out = wl.clone_base()
    wide = torch.empty(wl.tokens, 2048, dtype=wl.x.dtype, device=dev)
    wide[:, :1024] = wl.x
    bare = synthetic.make_meta(wl.seg_lens, wl.seg_slots, wl.slot_ranks, wl.scalings, dev, torch.bfloat16,
                               with_plan=False)
    strided = [a.transpose(1, 2).contiguous().transpose(1, 2) for a in wl.a_stacks]
    assert taken(wl, out, x=wide[:, :1024]) is None
    assert taken(wl, out, a=strided) is None
    assert taken(wl, out, x=wl.x.cpu()) is None
    assert taken(wl, out, x=wl.x.half()) is None
    assert taken(wl, out, cols=[0, 512, -1]) is None
    assert taken(wl, out, cols=[0, 512, 900]) is None
    assert taken(wl, out[:-1]) is None
    assert torch.equal(out, wl.base)
    want = wl.clone_base()
    assert taken(wl, want) is True
    be = HipLoRABackend()
    for x, a, meta in ((wide[:, :1024], wl.a_stacks, wl.meta), (wl.x, strided, wl.meta), (wl.x, wl.a_stacks, bare)):
        be.set_kernel_input_metadata(meta)
        got = be.apply_lora_multi(x, a, wl.b_stacks, wl.clone_base(), wl.col_offsets)
        assert torch.equal(got, want)
    with pytest.raises(ValueError, match="output must cover"):
        be.apply_lora_multi(wl.x, wl.a_stacks, wl.b_stacks, out[:-1], wl.col_offsets)
    with pytest.raises(RuntimeError, match="GPU"):
        be.apply_lora_multi(wl.x.cpu(), wl.a_stacks, wl.b_stacks, out, wl.col_offsets)


def test_a_capture_without_a_workspace_raises_as_before(dev):
    wl = decode(dev)
    be = HipLoRABackend()
    be.set_kernel_input_metadata(wl.meta)
    out = wl.clone_base()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with pytest.raises(RuntimeError, match="workspace of the capturing stream"):
        with torch.cuda.graph(graph, stream=stream):
            be.apply_lora_multi(wl.x, wl.a_stacks, wl.b_stacks, out, wl.col_offsets)


def test_native_fused_norm_and_two_call_forms(dev):
    wl = decode(dev)
    w, eps = wl.extra["norm_weight"], wl.extra["eps"]
    y, out = torch.empty_like(wl.x), wl.clone_base()
    args = (wl.a_stacks, wl.b_stacks, wl.meta, out, wl.col_offsets)
    assert _ffi.calls().rmsnorm_apply(wl.x, w, eps, y, *args, LinkedWorkspace(), 3) is True
    y2, out2 = torch.empty_like(wl.x), wl.clone_base()
    assert rmsnorm_apply_grouped(wl.x, w, eps, y2, wl.a_stacks, wl.b_stacks, wl.meta, out2, wl.col_offsets,
                                 LinkedWorkspace())
    assert torch.equal(y, y2) and torch.equal(out, out2)
    assert torch.equal(y, rmsnorm_fwd(wl.x, w, eps))
    assert torch.equal(rmsnorm_fwd(wl.x.t().contiguous().t(), w, eps), y)  # not contiguous: the Python path
    res, res2 = wl.x.clone(), wl.x.clone()
    got = fused_add_rmsnorm(wl.x, res, w, eps)
    want = fused_add_rmsnorm(wl.x.t().contiguous().t(), res2, w, eps)
    assert torch.equal(got, want) and torch.equal(res, res2)
    assert got.shape == wl.x.shape and rmsnorm_fwd(wl.x[None], w, eps).shape == (1,) + wl.x.shape

    p = prompts(dev)
    buf = torch.full((p.tokens + 3, 40), 7.0, dtype=p.x.dtype, device=dev)
    mid = sgemm_lora_a_fwd(p.x, p.a_stacks[0], p.meta, buf)
    want_mid = shrink(p.x, [p.a_stacks[0]], p.meta, torch.empty_like(mid).contiguous(), workspace=Workspace())
    assert torch.equal(mid, want_mid) and mid.data_ptr() == buf.data_ptr() and bool((buf[:, 32:] == 7).all())
    mid = mid.contiguous()
    one, two = p.base[:, :768].contiguous(), p.base[:, :768].contiguous()
    assert sgemm_lora_b_fwd(mid, p.b_stacks[0], p.meta, one) is one
    expand(mid, [p.b_stacks[0]], p.meta, two, [0])
    assert torch.equal(one, two)


@pytest.mark.parametrize("make", [decode, prompts])
def test_stacks_live_for_the_length_of_the_call(dev, make):
    """A list that loses its stacks while the call makes its workspace: their
    memory may go to other tensors only after the call."""
    wl = make(dev)
    want, got = wl.clone_base(), wl.clone_base()
    assert taken(wl, want, cols=wl.col_offsets) is True
    a, b = [t.clone() for t in wl.a_stacks], [t.clone() for t in wl.b_stacks]
    sizes = [t.numel() for t in a + b]
    spoilt = []

    def spoil(get):
        def run(*args):
            a.clear()
            b.clear()
            spoilt.extend(torch.full((n,), float("nan"), dtype=wl.x.dtype, device=dev) for n in sizes)
            return get(*args)
        return run

    linked, seg = LinkedWorkspace(), Workspace()
    linked.get, seg.get = spoil(linked.get), spoil(seg.get)
    assert taken(wl, got, a=a, b=b, cols=wl.col_offsets, linked=linked, seg=seg) is True
    torch.cuda.synchronize()
    assert spoilt and torch.equal(got, want)
