"""The decoder's one-launch decode attention and SiLU gate (GPU) against the
same arithmetic in float64, over cache lengths around the kernel's chunks,
every head grouping, strided inputs, and calls it leaves to torch."""

import pytest
import torch

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
    for pos in (-1, 40):                                  # outside the cache: nothing is written
        assert decode_attention(*args, torch.tensor([pos], device=dev), 0.125) is not None
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
