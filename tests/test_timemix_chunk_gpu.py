"""The time-mix memory of a prompt in chunks on the matrix cores (csrc/hybrid/timemix_chunk.hip): against the ops on the CPU at the
edges of its chunks and segments, against 64 bits, and with numbers that are none."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(b, s, h, shift=-2.0, seed=0):
    g = torch.Generator().manual_seed(seed)
    r, k, v, w = (torch.randn(b * s, h, 64, generator=g) for _ in range(4))
    return [r, k, v, w + shift, torch.randn(h, 64, generator=g), torch.randn(h, 64, generator=g)], torch.randn(b, h, 64, 64, generator=g)


def _rel(a, b):
    return float((a.float().cpu() - b.float()).abs().max() / b.abs().max())


@pytest.mark.parametrize("b,s,h", [(1, 2, 3), (1, 15, 2), (2, 16, 2), (1, 17, 5), (3, 31, 2), (1, 32, 1), (1, 33, 2), (2, 47, 3), (1, 300, 4),
                                   (40, 20, 16), (1, 130, 600)])
@pytest.mark.parametrize("shift", [-5.0, 0.0, 3.0])
def test_chunks_as_token_by_token(b, s, h, shift):
    """Output, carried state and the normed output (fp32 and a bf16 column slice) as the CPU ops; decays from nearly one to zero."""
    x, st = _inputs(b, s, h, shift)
    gate, w = torch.randn(b * s, h * 64), torch.rand(h * 64) + 0.5
    dev = [t.to(DEV) for t in x]
    ref_st, dev_st = st.clone(), st.to(DEV)
    ref, got = hy.timemix_scan(*x, ref_st, b, s), hy.timemix_scan(*dev, dev_st, b, s)
    assert _rel(got, ref) < 2e-5 and _rel(dev_st, ref_st) < 2e-5
    ref = hy.gated_rmsnorm(ref, gate, w, 1e-6, hy.GATE_SILU, gain=0.5)
    for dtype, tol in ((torch.float32, 2e-5), (torch.bfloat16, 2.0 ** -8)):
        dev_st = st.to(DEV)
        out = torch.zeros(b * s, h * 64 + 8, dtype=dtype, device=DEV)[:, 4:4 + h * 64]
        got = hy.timemix_memory(*dev, dev_st, b, s, gate.to(DEV), w.to(DEV), 1e-6, 0.5, out)
        assert got is out and _rel(got, ref) < tol and _rel(dev_st, ref_st) < 2e-5


def test_no_rows():
    """An empty batch of a prompt gives an empty result (there are no heads to deal segments to)."""
    x, st = _inputs(0, 5, 2)
    got = hy.timemix_scan(*[t.to(DEV) for t in x], st.to(DEV), 0, 5)
    assert got.shape == (0, 2, 64) and got.is_cuda


@pytest.mark.parametrize("b,s,shift", [(1, 777, -3.0), (2, 130, -3.0), (1, 17, 0.0), (3, 64, 1.0), (1, 400, -5.0), (1, 1000, -2.0)])
def test_no_less_exact_than_the_scan(b, s, shift):
    """Relative errors (2-norm) against 64 bits beside those of the token-by-token scan, which rows off 16 bytes still take. Both are
    sums of thousands of roundings, the same to a few parts in a hundred from one set of inputs to the next: 2 % of scatter."""
    h = 8
    x, st = _inputs(b, s, h, shift, 1)
    dev, S, S_scan = [t.to(DEV) for t in x], st.to(DEV), st.to(DEV)
    o = hy.timemix_scan(*dev, S, b, s)
    odd = torch.zeros(b * s, h * 64 + 1, device=DEV)
    odd[:, :h * 64] = dev[0].reshape(b * s, -1)
    o_scan = hy.timemix_scan(odd[:, :h * 64].unflatten(1, (h, 64)), *dev[1:], S_scan, b, s)
    r, k, v, w = (t.double().reshape(b, s, h, 64) for t in dev[:4])
    d, S64, ref = torch.exp(-torch.exp(w + dev[4].double())), st.to(DEV).double(), torch.empty_like(v)
    for t in range(s):
        kv = k[:, t, :, :, None] * v[:, t, :, None]
        ref[:, t] = ((S64 + dev[5].double()[None, :, :, None] * kv) * r[:, t, :, :, None]).sum(2)
        S64 = S64 * d[:, t, :, :, None] + kv
    err = lambda y, z: float((y.double().reshape(z.shape) - z).norm() / z.norm())  # noqa: E731
    assert err(o, ref) <= 1.02 * err(o_scan, ref)
    assert err(S, S64) <= 1.02 * err(S_scan, S64)


@pytest.mark.parametrize("operand", range(4))
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("b,s", [(1, 45), (2, 70)])
def test_a_number_that_is_none_reaches_no_token_before_it(b, s, operand, bad):
    h = 2
    x, st = _inputs(b, s, h, -1.0, 2)
    x[operand].reshape(b * s, -1)[(b - 1) * s + 37, 3] = bad
    S = st.clone().to(DEV)
    got = hy.timemix_scan(*[t.to(DEV) for t in x], S, b, s).cpu()
    want = hy.timemix_scan(*x, st, b, s)
    assert torch.isfinite(got.reshape(b, s, -1)[:, :37]).all()
    for w, y in ((want, got), (st, S.cpu())):
        ok = torch.isfinite(w)
        assert torch.equal(torch.isfinite(y), ok) and float((y - w)[ok].abs().max()) < 2e-5 * float(w[ok].abs().max())


@pytest.mark.parametrize("b,s", [(1, 1), (2, 63), (1, 64), (1, 65), (3, 130), (1, 1023), (2, 1024), (1, 1025), (1, 2113)])
def test_gates_of_the_exponential_memory(b, s):
    """The running maximum over blocks of 64 and 1024 tokens: every token's factors and the carried maximum as the CPU's chain."""
    h, cap = 3, 15.0
    proj, bias, m = torch.randn(b * s, 2 * h + 5) * 6.0, torch.randn(2 * h), torch.rand(b, h) * 8.0
    m_dev = m.to(DEV)
    got = hy.mlstm_prep(proj.to(DEV), 1, h + 2, bias.to(DEV), cap, m_dev, b, s, h)
    want = hy.mlstm_prep(proj, 1, h + 2, bias, cap, m, b, s, h)
    for x, y in zip(got, want):  # (tanh, exp and log of the two sides: a few units in the last place of exponents up to 15)
        assert float(((x.cpu() - y).abs() / y.abs().clamp_min(1e-12)).max()) < 2e-5
    assert float((m_dev.cpu() - m).abs().max()) < 15.0 * 2.0 ** -21
