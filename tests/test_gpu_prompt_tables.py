"""Batches with segments of more than 16 rows over a packed table (GPU).

Such a batch reads the table's columns, never its plan: the results match
the oracle at the edges of the 16-row tiles and follow every write to the
columns, also one that torch's version counters do not see, and a captured
call gives the bits of the eager one.
"""

import pytest
import torch

from multi_lora_amd import HipLoRABackend
from multi_lora_amd.batch_info import BatchLoRAInfo, empty_kernel_input_metadata, write_kernel_input_metadata
from multi_lora_amd.synthetic import make_meta
from oracle.lora_ref import apply_f64
from tests.gpu_helpers import assert_tol_f64

pytestmark = pytest.mark.gpu


def packed(lens, slots, ranks, scal, dtype, dev, meta=None):
    meta = empty_kernel_input_metadata(device=dev, dtype=dtype) if meta is None else meta
    return write_kernel_input_metadata(meta, BatchLoRAInfo(slots, ranks, scal), device=dev, dtype=dtype, seq_lens=lens)


def inputs(lens, ranks, in_dim, outs, r_max, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    n = len(ranks)
    x = torch.randn(sum(lens), in_dim, generator=g).to(dtype)
    a = [(torch.randn(n, r_max, in_dim, generator=g) * in_dim ** -0.5).to(dtype) for _ in outs]
    b = [(torch.randn(n, o, r_max, generator=g) * 0.05).to(dtype) for o in outs]
    base = torch.randn(sum(lens), sum(outs), generator=g).to(dtype)
    return x, a, b, base, [sum(outs[:i]) for i in range(len(outs))], [0.5 + 0.25 * i for i in range(n)]


@pytest.mark.parametrize("lens,slots,ranks,in_dim,outs,r_max,dtype", [
    ([17], [0], [8, 0], 256, [256], 8, torch.bfloat16),
    ([16, 33, 0, 1, 48], [1, 0, 1, 2, 1], [16, 9, 0], 1000, [264, 72], 16, torch.float16),
    ([203], [3], [0, 0, 0, 64], 4096, [1024], 64, torch.bfloat16),
    ([31, 1, 1, 5, 64, 100, 2], [0, 1, 0, 2, 3, 3, 0], [64, 33, 0, 7], 520, [512, 128, 128], 64, torch.bfloat16),
    ([40] * 20, [i % 3 for i in range(20)], [8, 16, 0], 14336, [128], 16, torch.float16),
])
def test_prompt_batches_match_the_oracle(dev, lens, slots, ranks, in_dim, outs, r_max, dtype):
    x, a, b, base, cols, scal = inputs(lens, ranks, in_dim, outs, r_max, dtype, sum(lens))
    meta = packed(lens, slots, ranks, scal, dtype, dev)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)
    out = base.to(dev)
    be.apply_lora_multi(xd, ad, bd, out, cols)
    want = apply_f64(x, a, b, make_meta(lens, slots, ranks, scal, "cpu", dtype), base, cols)
    assert_tol_f64(out.cpu(), want)
    live = torch.cat([torch.full((n,), ranks[s] > 0) for n, s in zip(lens, slots)])
    assert torch.equal(out.cpu()[~live], base[~live])


def test_eager_calls_follow_every_write_to_the_columns(dev):
    lens, slots, ranks, dtype = [60, 30], [0, 1], [16, 16, 16], torch.bfloat16
    x, a, b, base, cols, scal = inputs(lens, ranks, 512, [256], 16, dtype, 3)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    meta = packed(lens, slots, ranks, scal, dtype, dev)
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)

    def check(want_lens, want_slots, rows=len(x)):
        out = base.to(dev)[:rows]
        be.apply_lora_multi(xd[:rows], ad, bd, out, cols)
        want = apply_f64(x[:rows], a, b, make_meta(want_lens, want_slots, ranks, scal, "cpu", dtype), base[:rows], cols)
        assert_tol_f64(out.cpu(), want)

    def column(v):
        return torch.tensor(v, dtype=torch.int32, device=dev)

    check(lens, slots)
    check([60, 11], slots, rows=71)               # fewer rows than the table lists
    with torch.inference_mode():
        meta.weight_indices[:2] = column([2, 0])
    check(lens, [2, 0])                           # a column written directly
    with torch.inference_mode():
        assert packed([50, 40], [1, 2], ranks, scal, dtype, dev, meta) is meta
    check([50, 40], [1, 2])
    meta.weight_indices.data[:2] = column([0, 2])
    check([50, 40], [0, 2])                       # written with no version counted
    meta.seg_indptr.data[1:2] = column([35])
    check([35, 55], [0, 2])
    meta.weight_indices = column([2, 1])
    check([35, 55], [2, 1])                       # a column replaced


def test_eager_calls_follow_a_replayed_write_to_the_columns(dev):
    lens, ranks, dtype = [60, 30], [16, 16, 16], torch.bfloat16
    x, a, b, base, cols, scal = inputs(lens, ranks, 512, [256], 16, dtype, 4)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    meta = packed(lens, [0, 1], ranks, scal, dtype, dev)
    new = torch.tensor([2, 2], dtype=torch.int32, device=dev)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        meta.weight_indices[:2].copy_(new)
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)
    for slots in ([2, 0], [1, 1]):
        # Rewritten eagerly, then by the replay, which counts no version.
        assert packed(lens, [0, 1], ranks, scal, dtype, dev, meta) is meta
        new.copy_(torch.tensor(slots, dtype=torch.int32))
        graph.replay()
        out = base.to(dev)
        be.apply_lora_multi(xd, ad, bd, out, cols)
        want = apply_f64(x, a, b, make_meta(lens, slots, ranks, scal, "cpu", dtype), base, cols)
        assert_tol_f64(out.cpu(), want)


def test_captured_calls_give_the_eager_bits_and_follow_the_columns(dev):
    ranks, dtype = [16, 8, 16, 16], torch.bfloat16
    scal = [1.0] * 4
    lens, slots = [200, 190], [2, 0]
    x, a, b, base, cols, _ = inputs(lens, ranks, 4096, [256], 16, dtype, 5)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    meta = packed([20, 20], [0, 1], ranks, scal, dtype, dev)
    # More 16-row tiles than the table was made for.
    assert packed(lens, slots, ranks, scal, dtype, dev, meta) is meta and meta.plan_entries > meta.plan_cap
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)
    out = base.to(dev)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        be.apply_lora_multi(xd, ad, bd, out, cols)
    eager = out.clone()
    buf = be.workspace.buf
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        be.apply_lora_multi(xd, ad, bd, out, cols)
    assert be.workspace.buf is buf                # the warm-up left nothing to allocate
    for s in ([2, 0], [1, 3], [0, 0]):            # a replay follows the columns however they are written
        meta.weight_indices[:2] = torch.tensor(s, dtype=torch.int32, device=dev)
        out.copy_(base)
        graph.replay()
        torch.cuda.synchronize()
        assert_tol_f64(out.cpu(), apply_f64(x, a, b, make_meta(lens, s, ranks, scal, "cpu", dtype), base, cols))
        if s == slots:
            assert torch.equal(out, eager)
