"""Prompt attention over fp32 caches on the fp32 matrix instruction (csrc/hybrid/attn_f32.hip) against the CPU op, at the edges of
its tiles and with numbers that are none."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _both(q, kc, vc, s0, scale, **kw):
    want = hy.attn_bias(q, kc, vc, s0, scale, **kw)
    got = hy.attn_bias(q.to(DEV), kc.to(DEV), vc.to(DEV), torch.tensor([s0], dtype=torch.int32, device=DEV), scale,
                       **{k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()})
    return got.cpu(), want


@pytest.mark.parametrize("b,s,s0,h,g,dim,vdim", [(1, 2, 0, 2, 1, 64, 64), (2, 15, 1, 4, 2, 64, 128), (1, 16, 48, 2, 2, 128, 64),
                                                 (1, 17, 63, 2, 1, 128, 128), (3, 65, 0, 2, 1, 64, 64), (1, 200, 400, 2, 1, 128, 128)])
@pytest.mark.parametrize("how", ["plain", "bias", "chunk", "window", "sink", "gate"])
def test_as_the_cpu_op(b, s, s0, h, g, dim, vdim, how):
    t = s0 + s + 5
    q, kc, vc = torch.randn(b, s, h, dim), torch.randn(b, g, t, dim), torch.randn(b, g, t, vdim)
    kc[:, :, s0 + s:], vc[:, :, s0 + s:] = float("nan"), float("nan")  # (slots that hold nothing yet)
    kw = {"plain": {}, "bias": dict(softcap=20.0, bias=torch.randn(40, h)), "chunk": dict(chunk=24, head_scale=torch.rand(h) + 0.5),
          "window": dict(window=37, keep_first=5), "sink": dict(sink=torch.randn(h)),
          "gate": dict(gate=torch.randn(b * s, h * vdim), gate_cols=True)}[how]
    got, want = _both(q, kc, vc, s0, dim ** -0.5, **kw)
    assert float((got - want).abs().max() / want.abs().max()) < 2e-5


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("where", ["key", "value", "query"])
def test_a_number_that_is_none_reaches_no_query_before_it(where, bad):
    b, s, h, dim = 1, 70, 2, 64
    q, kc, vc = torch.randn(b, s, h, dim), torch.randn(b, 1, s, dim), torch.randn(b, 1, s, dim)
    (q if where == "query" else kc if where == "key" else vc).view(-1, dim)[2 * 37 if where == "query" else 37, 3] = bad
    if where == "value":  # (the CPU op multiplies hidden values by 0: what it gives without the number, and where it is seen)
        clean = vc.clone()
        clean.view(-1, dim)[37, 3] = 0.0
        got, _ = _both(q, kc, vc, 0, 0.125)
        want = hy.attn_bias(q, kc, clean, 0, 0.125)
        ok = torch.ones(s, h, dim, dtype=torch.bool)
        ok[37:, :, 3] = False
        ok = ok.reshape(s, -1)
    else:
        got, want = _both(q, kc, vc, 0, 0.125)
        ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), ok) and float((got - want)[ok].abs().max()) < 2e-5 * float(want[ok].abs().max())


@pytest.mark.parametrize("at", [5, 37, 69])
@pytest.mark.parametrize("bad", [(float("inf"), float("inf")), (float("-inf"), float("inf")), (float("nan"), float("inf"))])
@pytest.mark.parametrize("window", [0, 20])
@pytest.mark.parametrize("dim", [64, 128])
def test_a_value_without_end_is_the_same_in_every_tile(at, bad, window, dim):
    """What a query gets that sees one or both of two keys whose values are not finite in a column: the infinity, NaN where they
    are of both signs or one is NaN, wherever the keys lie in tiles of 16 with and without hidden keys. Queries that see neither,
    and the other columns, as without them."""
    s, h = 90, 2
    q, kc, vc = torch.randn(1, s, h, dim) * 0.1, torch.randn(1, 1, s, dim), torch.randn(1, 1, s, dim)
    held = vc.clone()
    for j, x in zip((at, at + 7), bad):
        held[0, 0, j, 3], vc[0, 0, j, 3] = x, 0.0
    kw = dict(window=window) if window else {}
    want = hy.attn_bias(q, kc, vc, 0, dim ** -0.5, **kw).view(s, h, dim)
    for i in range(s):
        seen = [x for j, x in zip((at, at + 7), bad) if j <= i and (not window or i - j < window)]
        if seen:
            want[i, :, 3] = sum(seen)
    got = _both(q, kc, held, 0, dim ** -0.5, **kw)[0].view(s, h, dim)
    ok = torch.isfinite(want)
    assert torch.equal(torch.nan_to_num(got, 7e30, 8e30, 9e30)[~ok], torch.nan_to_num(want, 7e30, 8e30, 9e30)[~ok])
    assert torch.equal(torch.isfinite(got), ok) and float((got - want)[ok].abs().max()) < 2e-5 * float(want[ok].abs().max())


@pytest.mark.parametrize("s,s0,bias,dim", [(2, 62, False, 128), (2, 63, False, 128), (2, 123, True, 64), (2, 124, True, 64), (4, 28, False, 64), (4, 29, True, 128)])
def test_a_few_queries_of_many_rows_in_either_form(s, s0, bias, dim):
    """Slots that the host knows choose the form for a few queries over few keys, slots on the device never do: the same from both,
    on either side of the rule's line, and as the CPU op."""
    b, h, g = 200, 4, 2
    q, kc, vc = torch.randn(b, s, h, dim), torch.randn(b, g, s0 + s + 3, dim), torch.randn(b, g, s0 + s + 3, dim)
    kw = dict(softcap=20.0, bias=torch.randn(40, h)) if bias else {}
    dev = {k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()}
    got = hy.attn_bias(q.to(DEV), kc.to(DEV), vc.to(DEV), s0, dim ** -0.5, **dev).cpu()
    tiles, want = _both(q, kc, vc, s0, dim ** -0.5, **kw)
    for y in (got, tiles):
        assert float((y - want).abs().max() / want.abs().max()) < 2e-5
