"""The decoder's one-launch decode attention and SiLU gate (GPU) against the
same arithmetic in float64, over cache lengths around the kernel's chunks,
every head grouping, strided inputs, and calls it leaves to torch."""

import pytest
import torch
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from multi_lora_amd.decoder import MLP, Attention, DecoderConfig, Rotary, StaticKV
from multi_lora_amd.kernels.decode_attn import decode_attention, silu_mul

pytestmark = pytest.mark.gpu

# One rounding of the stored output, plus the new key's rounding in one of the
# scores: within a unit of the output's largest magnitude.
TOL = {torch.bfloat16: 2e-2, torch.float16: 3e-3}


def inputs(dev, b, heads, kv_heads, d, length, dtype, pad, seed):
    g = torch.Generator().manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)  # noqa: E731
    qkv = rn(b, (heads + 2 * kv_heads) * d + pad)
    q, k, v = qkv[:, :heads * d], qkv[:, heads * d:(heads + kv_heads) * d], qkv[:, (heads + kv_heads) * d:(heads + 2 * kv_heads) * d]
    ang = torch.rand(b, 1, d // 2, generator=g) * 6
    cos = torch.cat((ang.cos(), ang.cos()), -1).to(dtype).to(dev)
    sin = torch.cat((-ang.sin(), ang.sin()), -1).to(dtype).to(dev)
    hide = (torch.rand(b, 1, 1, length, generator=g) < 0.3).to(dev)
    return q, k, v, cos, sin, rn(b, kv_heads, d, length), rn(b, kv_heads, length, d), hide


def reference(q, k, v, cos, sin, keys, values, hide, pos, scale):
    b, kv_heads, d, length = keys.shape
    rot = lambda t: t * cos.double() + t.roll(d // 2, -1) * sin.double()  # noqa: E731
    qr = rot(q.double().view(b, -1, d)).view(b, kv_heads, -1, d)
    kr = rot(k.double().view(b, -1, d)).to(q.dtype)
    keys, values = keys.clone(), values.clone()
    keys[..., pos], values[:, :, pos] = kr, v.view(b, kv_heads, d)
    scores = (qr @ keys.double()) * scale
    probs = torch.softmax(scores.masked_fill(hide, float("-inf")), -1)
    return (probs @ values.double()).reshape(b, -1), keys, values


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,heads,kv_heads,d,length,pad", [
    (1, 1, 1, 64, 1, 0), (3, 4, 2, 64, 17, 3), (2, 8, 2, 128, 208, 8), (5, 8, 1, 128, 255, 0), (2, 8, 8, 64, 256, 0),
    (1, 16, 2, 128, 257, 0), (64, 4, 1, 128, 2048, 8),
])
def test_decode_attention(dev, b, heads, kv_heads, d, length, pad, dtype):
    for pos in {0, length // 2, length - 1}:
        args = inputs(dev, b, heads, kv_heads, d, length, dtype, pad, length + pos)
        args[-1][..., pos] = False                       # a step attends its own token
        want, keys, values = reference(*args, pos, d ** -0.5)
        got = decode_attention(*args, torch.tensor([pos], device=dev), d ** -0.5)
        assert got is not None
        torch.cuda.synchronize()
        assert (got.double() - want).abs().max().item() <= TOL[dtype] * max(1.0, want.abs().max().item())
        # the cache holds the new token (rotary: one rounding) and is otherwise untouched
        assert torch.equal(args[6], values)
        diff = (args[5].double() - keys.double()).abs()
        assert diff[..., pos].max().item() <= TOL[dtype] * 4
        diff[..., pos] = 0
        assert not diff.any()


def test_decode_attention_positions_and_refusals(dev):
    args = inputs(dev, 2, 4, 2, 64, 40, torch.bfloat16, 0, 1)
    keys, values = args[5].clone(), args[6].clone()
    for pos in (-1, 40):                                  # outside the cache: nothing is written, no answer
        assert bool(decode_attention(*args, torch.tensor([pos], device=dev), 0.125).isnan().all())
    assert torch.equal(args[5], keys) and torch.equal(args[6], values)
    at = torch.tensor([3], device=dev)
    assert decode_attention(*[t.float() if t.dtype == torch.bfloat16 else t for t in args], at, 0.125) is None
    assert decode_attention(*args[:5], args[5].transpose(2, 3).contiguous().transpose(2, 3), *args[6:], at, 0.125) is None
    assert decode_attention(args[0].clone().requires_grad_(), *args[1:], at, 0.125) is None
    assert torch.equal(args[5], keys) and torch.equal(args[6], values)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 8), (33, 1, 264), (5, 3, 7168)])
def test_silu_mul(dev, shape, dtype):
    both = torch.randn(*shape[:-1], 2 * shape[-1], generator=torch.Generator().manual_seed(1)).mul(4).to(dtype).to(dev)
    gate, up = both[..., :shape[-1]], both[..., shape[-1]:]
    got = silu_mul(gate, up)
    want = torch.nn.functional.silu(gate.double()) * up.double()
    assert got.shape == gate.shape and got.is_contiguous()
    torch.testing.assert_close(got.double(), want, rtol=2.0 ** (-8 if dtype == torch.bfloat16 else -11), atol=1e-6)
    assert silu_mul(gate.float(), up.float()) is None and silu_mul(gate[..., :-1], up[..., :-1]) is None


CONFIG = DecoderConfig(hidden_size=256, intermediate_size=512, num_attention_heads=4, num_key_value_heads=2)
POS = 5


def layer(dev, kind):
    """One decode step through the decoder's module ``kind``, as a function of its input."""
    torch.manual_seed(3)
    if kind == "mlp":
        return MLP(CONFIG).to(dev, torch.bfloat16).requires_grad_(False)
    attn = Attention(CONFIG).to(dev, torch.bfloat16).requires_grad_(False)
    inv = 1.0 / (CONFIG.rope_theta ** (torch.arange(0, 64, 2, device=dev) / 64))
    rot = Rotary.make(torch.full((3,), POS, device=dev), inv, torch.bfloat16)
    hide = (torch.arange(8, device=dev) > POS).view(1, 1, 1, 8).expand(3, 1, 1, 8)
    filled = [torch.randn(3, 2, 64, 8, device=dev).bfloat16(), torch.randn(3, 2, 8, 64, device=dev).bfloat16()]
    at = torch.tensor([POS], device=dev)

    def run(x):
        kv = StaticKV(CONFIG, 3, 8, dev, torch.bfloat16)
        kv.keys[0].copy_(filled[0])
        kv.values[0].copy_(filled[1])
        return attn(x, rot, hide, kv, 0, at)

    return run


def rows(dev, seed):
    return torch.randn(3, 1, 256, generator=torch.Generator().manual_seed(seed)).bfloat16().to(dev)


def close(got, want):
    torch.testing.assert_close(got.float(), want.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("kind", ["mlp", "attention"])
def test_forward_mode_keeps_the_tangent(dev, kind, grad):
    f, x, t = layer(dev, kind), rows(dev, 1), rows(dev, 2)
    with torch.set_grad_enabled(grad):
        with forward_ad.dual_level():
            out = forward_ad.unpack_dual(f(forward_ad.make_dual(x, t)))
        assert out.tangent is not None
        step = 0.125  # a power of two: x +- step * t differ from x by few roundings
        want = (f(x + step * t).float() - f(x - step * t).float()) / (2 * step)
    close(out.primal, f(x))
    assert (out.tangent.float() - want).norm() <= 0.1 * want.norm()


def test_function_transforms_and_traces_see_torch_operations(dev):
    f, x, t = layer(dev, "mlp"), rows(dev, 1), rows(dev, 2)
    want = f(x)
    close(torch.func.vmap(f)(x), want)
    assert bool(torch.func.jvp(f, (x,), (t,))[1].any())
    traced = torch.jit.trace(f, (t,), check_trace=False)
    close(traced(x), want)
    attn = layer(dev, "attention")
    close(torch.jit.trace(attn, (t,), check_trace=False)(x), attn(x))


class Counting(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


class CountingFunctions(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.seen.append(getattr(func, "__name__", ""))
        return func(*args, **(kwargs or {}))


def test_modes_see_torch_operations_and_a_default_device_does_not_matter(dev):
    gate, up = rows(dev, 1), rows(dev, 2)
    f, x = layer(dev, "mlp"), rows(dev, 1)
    with Counting() as mode:
        f(x)
    assert any("silu" in s for s in mode.seen)
    with CountingFunctions() as mode:
        f(x)
    assert any("silu" in s for s in mode.seen)
    with torch.device(dev):
        assert silu_mul(gate, up) is not None


def test_calls_of_another_device_than_the_current_one_are_left_to_torch(dev, monkeypatch):
    gate, up = rows(dev, 1), rows(dev, 2)
    assert silu_mul(gate, up) is not None
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert silu_mul(gate, up) is None


def test_the_cache_write_is_counted_and_inference_caches_stay_refused(dev):
    args = inputs(dev, 2, 4, 2, 64, 40, torch.bfloat16, 0, 1)
    at = torch.tensor([3], device=dev)
    before = args[5]._version, args[6]._version
    assert decode_attention(*args, at, 0.125) is not None
    assert args[5]._version > before[0] and args[6]._version > before[1]
    with torch.inference_mode():
        made = inputs(dev, 2, 4, 2, 64, 40, torch.bfloat16, 0, 1)
        assert decode_attention(*made, at, 0.125) is not None
    assert decode_attention(*made, at, 0.125) is None


@pytest.mark.parametrize("heads,length", [(8, 600), (4, 1024)])
def test_caches_past_the_longest_one_are_left_to_torch(dev, heads, length):
    at = torch.tensor([1], device=dev)
    for n, taken in ((length, True), (length + 1, False)):
        args = inputs(dev, 1, heads, 1, 64, n, torch.bfloat16, 0, 1)
        assert (decode_attention(*args, at, 0.125) is not None) is taken
