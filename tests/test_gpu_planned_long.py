"""Batches with segments of more than 16 rows on the slot-planned path (GPU).

The backend sends such a batch through its packed table's plan while the
items' reads stay small; the results must match the oracle at the edges of
the 16-row entries, and the segment path must take over wherever the plan
does not describe the table any more.
"""

import pytest
import torch

from multi_lora_amd import HipLoRABackend
from multi_lora_amd.batch_info import BatchLoRAInfo, empty_kernel_input_metadata, write_kernel_input_metadata
from multi_lora_amd.kernels.lora_ops import planned_pays
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
def test_planned_long_batches_match_the_oracle(dev, lens, slots, ranks, in_dim, outs, r_max, dtype):
    x, a, b, base, cols, scal = inputs(lens, ranks, in_dim, outs, r_max, dtype, sum(lens))
    meta = packed(lens, slots, ranks, scal, dtype, dev)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    assert planned_pays(meta, xd, ad, bd)
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)
    out = base.to(dev)
    be.apply_lora_multi(xd, ad, bd, out, cols)
    torch.cuda.synchronize()
    assert be.linked_workspace.counters()[1] == 0
    want = apply_f64(x, a, b, make_meta(lens, slots, ranks, scal, "cpu", dtype), base, cols)
    assert_tol_f64(out.cpu(), want)
    live = torch.cat([torch.full((n,), ranks[s] > 0) for n, s in zip(lens, slots)])
    assert torch.equal(out.cpu()[~live], base[~live])


def test_a_plan_that_does_not_describe_the_table_is_not_used(dev):
    lens, slots, ranks, dtype = [60, 30], [0, 1], [16, 16, 16], torch.bfloat16
    x, a, b, base, cols, scal = inputs(lens, ranks, 512, [256], 16, dtype, 3)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    with torch.inference_mode():
        meta = packed(lens, slots, ranks, scal, dtype, dev)
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)

    def check(want_lens, want_slots, pays, rows=len(x)):
        assert planned_pays(meta, xd[:rows], ad, bd) == pays
        out = base.to(dev)[:rows]
        be.apply_lora_multi(xd[:rows], ad, bd, out, cols)
        want = apply_f64(x[:rows], a, b, make_meta(want_lens, want_slots, ranks, scal, "cpu", dtype), base[:rows], cols)
        assert_tol_f64(out.cpu(), want)

    check(lens, slots, True)
    check([60, 11], slots, False, rows=71)       # planned rows past the call's
    with torch.inference_mode():
        meta.weight_indices[:2] = torch.tensor([2, 0], dtype=torch.int32, device=dev)
    check(lens, [2, 0], False)                    # a column written directly
    with torch.inference_mode():                  # (a table made in inference mode is rewritten in it)
        assert packed([50, 40], [1, 2], ranks, scal, dtype, dev, meta) is meta
    check([50, 40], [1, 2], True)
    meta.weight_indices = torch.tensor([2, 1], dtype=torch.int32, device=dev)
    check([50, 40], [2, 1], False)                # a column replaced


def test_rewrites_beyond_the_plan_and_captured_calls_run_as_segments(dev):
    ranks, dtype = [16, 8, 16, 16], torch.bfloat16
    scal = [1.0] * 4
    meta = packed([20, 20], [0, 1], ranks, scal, dtype, dev)
    lens, slots = [200, 190], [2, 0]              # more entries than the plan was made for
    x, a, b, base, cols, _ = inputs(lens, ranks, 512, [256], 16, dtype, 5)
    xd, ad, bd = x.to(dev), [t.to(dev) for t in a], [t.to(dev) for t in b]
    assert packed(lens, slots, ranks, scal, dtype, dev, meta) is meta and meta.plan_entries > meta.plan_cap
    assert not planned_pays(meta, xd, ad, bd)
    meta = packed(lens, slots, ranks, scal, dtype, dev)
    assert planned_pays(meta, xd, ad, bd)
    be = HipLoRABackend()
    be.set_kernel_input_metadata(meta)
    out = base.to(dev)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        be.apply_lora_multi(xd, ad, bd, out, cols)
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
