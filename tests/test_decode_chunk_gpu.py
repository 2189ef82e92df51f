"""Decode attention over bf16 caches of heads of 64 and 128 numbers (csrc/hybrid/attn_chunk.h): 64 keys at a time, at the edges of a chunk and of
the splits, key and value widths mixed, with and without biases, against 64-bit sums."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV, BF16 = "cuda", torch.bfloat16


@pytest.mark.parametrize("dim,vdim", [(64, 64), (64, 128), (128, 64), (128, 128)])
@pytest.mark.parametrize("b,h,g", [(1, 2, 1), (9, 32, 4)])
@pytest.mark.parametrize("slot,window", [(0, 0), (62, 0), (63, 0), (64, 0), (129, 0), (700, 0), (700, 65), (1900, 0)])
def test_keys_by_chunk(dim, vdim, b, h, g, slot, window):
    gen = torch.Generator(device=DEV).manual_seed(slot + dim)
    rand = lambda *s: torch.randn(*s, generator=gen, device=DEV)  # noqa: E731
    t = slot + 3
    q, kc, vc = rand(b, 1, h, dim), rand(b, g, t, dim).to(BF16), rand(b, g, t, vdim).to(BF16)
    kc[:, :, slot + 1:], vc[:, :, slot + 1:] = float("nan"), float("nan")  # (nothing behind the token is read into a sum)
    bias, sink = rand(90, h), rand(h)
    got = hy.attn_bias(q, kc, vc, slot, dim ** -0.5, 20.0, bias, None, sink, window=window)
    lo = max(0, slot + 1 - window) if window else 0
    k, v = (x[:, :, lo:slot + 1].double().repeat_interleave(h // g, 1) for x in (kc, vc))
    s = 20 * torch.tanh((k @ q.double().transpose(1, 2).transpose(2, 3).reshape(b, h, dim, 1)).squeeze(-1) * dim ** -0.5 / 20)
    s = s + bias.double()[(slot - torch.arange(lo, slot + 1, device=DEV)).clamp(max=89)].t()[None]
    p = torch.softmax(torch.cat([s, sink.double().view(1, h, 1).expand(b, h, 1)], -1), -1)[..., :-1]
    want = (p[..., None] * v).sum(2).reshape(b, h * vdim)
    # a score of size up to 10 is a sum of dim products rounded at 2^-24 of their size: 10 sqrt(16) 2^-24 into the exponential, and as much for
    # tanh's and exp's own roundings; the sums of weights and values lose less
    assert float((got.double().reshape(b, -1) - want).norm() / want.norm()) < 5e-6
