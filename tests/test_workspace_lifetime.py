"""Workspace buffers outlive their replacement by a larger one: a graph
captured with a buffer reads and writes it on every replay."""

import weakref

import pytest
import torch

from multi_lora_amd import HipLoRABackend, synthetic
from multi_lora_amd.kernels import lora_ops
from multi_lora_amd.kernels.lora_ops import LinkedWorkspace, Workspace

CPU = torch.device("cpu")


def test_a_replaced_segment_buffer_is_kept():
    ws = Workspace()
    ptr, _ = ws.get(1, CPU)
    first, alive = ws.buf, weakref.ref(ws.buf)
    big, size = ws.get(first.numel() + 1, CPU)
    assert big != ptr and size >= first.numel() + 1
    del first
    assert alive() is not None
    assert ws.get(1, CPU) == (big, size)          # the newest one serves
    for n in (1 << 22, 1 << 23, (1 << 23) + 1, 1 << 25):
        ws.get(n, CPU)
    assert sum(b.numel() for b in ws.kept) < 2 * ws.buf.numel()
    ws.buf = torch.empty(0, dtype=torch.uint8, device="meta")  # another device's buffer had its turn
    newest = ws.kept[-1]
    ws.get(1, CPU)
    assert ws.buf is newest


def test_a_replaced_decode_buffer_is_kept(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    ws, dev = LinkedWorkspace(), torch.device("cpu", 0)
    ws.get(1, dev, 7)
    alive = weakref.ref(ws.bufs[(0, 7)])
    ws.get(ws.bufs[(0, 7)].numel() + 1, dev, 7)
    assert alive() is not None and ws.bufs[(0, 7)] is not alive()
    alive()[:4].view(torch.int32).fill_(3)          # a replay of the old graph still counts
    assert ws.counters()[0] == 3
    ws.get(1, dev, 8)
    assert len(ws.bufs) == 2 and len(ws.replaced) == 1


def test_growth():
    assert lora_ops._grown(5, []) == 1 << 20
    assert lora_ops._grown(3 << 20, [torch.empty(1 << 20, dtype=torch.uint8)]) == 3 << 20
    assert lora_ops._grown((1 << 20) + 1, [torch.empty(1 << 20, dtype=torch.uint8)]) == 2 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["decode", "segments"])
def test_a_captured_call_survives_a_larger_call_on_its_stream(dev, kind):
    if kind == "decode":
        small = synthetic.decode_qkv(device=dev, tokens=16, hidden=1024, outs=[512, 256, 256], n_slots=12,
                                     n_adapters=9, rank=16)
        large = synthetic.decode_qkv(device=dev, tokens=256, hidden=4096, outs=[512, 256, 256], n_slots=12,
                                     n_adapters=9, rank=64)
    else:
        small = synthetic.prefill_mlp(device=dev, dtype=torch.bfloat16, part="gate_up", n_seg=2, min_len=20,
                                      max_len=40, hidden=1024, inter=512, r_max=32)
        large = synthetic.prefill_mlp(device=dev, dtype=torch.bfloat16, part="gate_up", n_seg=4, min_len=400,
                                      max_len=800, hidden=4096, inter=512, r_max=64)
    be, stream = HipLoRABackend(), torch.cuda.Stream()

    def call(wl, out):
        be.set_kernel_input_metadata(wl.meta)
        return be.apply_lora_multi(wl.x, wl.a_stacks, wl.b_stacks, out, wl.col_offsets)

    def newest():
        return be.workspace.buf if kind == "segments" else next(iter(be.linked_workspace.bufs.values()))

    out, want = small.clone_base(), small.clone_base()
    big, big_want = large.clone_base(), large.clone_base()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call(small, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call(small, out)
    before = newest()
    with torch.cuda.stream(stream):
        call(large, big_want)
    assert newest() is not before and newest().numel() > before.numel()
    # Allocations of the old buffer's size: none of them may be the memory the graph uses.
    with torch.cuda.stream(stream):
        fills = [torch.full((before.numel(),), 0x5A, dtype=torch.uint8, device=dev) for _ in range(4)]
    for _ in range(3):
        with torch.cuda.stream(stream):
            out.copy_(small.base)
            graph.replay()
            big.copy_(large.base)
            call(large, big)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(big, big_want)
        assert all(bool((f == 0x5A).all()) for f in fills)
