"""When the decoder's one-launch kernels step aside for torch's operations."""

import pytest
import torch
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from multi_lora_amd.kernels import decode_attn


class Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("make,want", [
    (lambda: torch.no_grad(), False), (lambda: torch.inference_mode(), False), (lambda: torch.device("cpu"), False),
    (lambda: forward_ad.dual_level(), True), (lambda: Dispatch(), True), (lambda: Functions(), True),
])
def test_contexts(make, want):
    with make():
        assert decode_attn._followed() is want
    assert decode_attn._followed() is False


def test_transforms_tracing_and_compilation(monkeypatch):
    seen = []

    def f(x):
        seen.append(decode_attn._followed())
        return x * 2

    x = torch.ones(2, 3)
    torch.func.vmap(f)(x)
    torch.func.jvp(f, (x,), (x,))
    torch.func.grad(lambda v: f(v).sum())(x)
    torch.jit.trace(f, (x,), check_trace=False)
    assert seen == [True] * 4
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert decode_attn._followed()


@pytest.mark.parametrize("key_heads,rep,longest", [(1, 8, 600), (63, 8, 600), (64, 8, 1024), (1, 4, 1024), (63, 1, 1024),
                                                   (64, 4, 2048), (512, 2, 2048)])
def test_longest_cache_by_the_workgroups_it_makes(key_heads, rep, longest):
    assert decode_attn._max_len(key_heads, rep) == longest
