"""A few rows that are bf16 already (csrc/hybrid/rows_gemv.hip, rows_mid.hip) and the kernels that write them: the products against
64-bit sums, and every writer's bf16 result as its fp32 result rounded."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV, BF16, F32 = "cuda", torch.bfloat16, torch.float32


def _tol(k):
    # exact products, summed in 64 bits but for runs of up to eight products, or in four fp32 chains of K / 128: 9e-8, or 3.0e-9 sqrt(k), of the
    # result measured; a quarter as much again
    return 1.2e-7 + 3e-9 * k ** 0.5


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("m", [3, 4, 5, 8, 9, 16, 17, 64])
@pytest.mark.parametrize("n,k", [(20, 64), (36, 72), (64, 4096), (260, 704), (2048, 5632), (4100, 256), (16400, 128)])
def test_products(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(n + k)
    x = torch.randn(m, k, generator=g, device=DEV).to(BF16)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    if not hy.few_bf16(m, w):  # (nine rows and more: whole 64-deep steps, as the tiles for them)
        assert m > 8 and (k % 64 or k < 128)
    want = x.double() @ w.double().t()
    assert _err(hy.linear(x, w), want) < _tol(k)
    low = hy.linear(x, w, out_dtype=BF16)
    assert torch.equal(low.to(BF16), hy.linear(x, w).to(BF16))
    res = torch.randn(m, n, generator=g, device=DEV)
    want2 = res.double() + want
    assert _err(hy.linear_add_(res, x, w), want2) < _tol(k)
    if n % 8 == 0 and hy.few_bf16(m, w, hy.ACT_SWIGLU):
        a, b = want.chunk(2, -1)
        got = hy.linear(x, w, swiglu=True, out_dtype=BF16)
        assert got.dtype == BF16 and _err(got, torch.nn.functional.silu(a) * b) < 2.0 ** -8
    # as fp32 rows of the same numbers: the same products
    assert _err(hy.linear(x.float(), w), want) < _tol(k)


@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("n,k", [(64, 8), (65, 64), (70, 128), (2048, 64), (2050, 120), (300, 32)])
def test_short_rows(m, n, k):
    """One or two fp32 rows of up to 128 numbers: exact products, eight at a time added in 24 bits, these sums in 64: 3.3e-8 (K 64) and 4.1e-8
    (K 128) of the result measured, with the result's own rounding; twice that."""
    g = torch.Generator(device=DEV).manual_seed(n + k)
    x = torch.randn(m, k + 4, generator=g, device=DEV)[:, :k]  # (rows apart)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    want = x.to(BF16).double() @ w.double().t()
    got = hy.linear(x, w)
    assert got.shape == (m, n) and _err(got, want) < 8e-8
    # a weight that is none stays in its column, also where the row ends inside the instruction's step
    w[n - 1, k - 1] = float("inf")
    bad = hy.linear(x, w)
    assert torch.equal(bad[:, :-1], got[:, :-1]) and not bool(torch.isfinite(bad[:, -1]).any())


@pytest.mark.parametrize("n,k", [(2048, 5632), (10304, 2048), (4096, 4096)])
def test_three_and_four_rows_are_no_less_exact_than_fp32_ones_were(n, k):
    """fp32 rows, rounded in the launch, were added in 64 bits every two products: 5.5e-8 to 5.6e-8 (every four: 6.4e-8 to 7.0e-8)."""
    g = torch.Generator(device=DEV).manual_seed(k)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    for m in (3, 4):
        x = torch.randn(m, k, generator=g, device=DEV).to(BF16)
        assert _err(hy.linear(x, w), x.double() @ w.double().t()) < 6e-8, m
        if n == k:
            each, ww = torch.randn(4, m, k, generator=g, device=DEV).to(BF16), w[:4096].view(4, 1024, k)
            assert _err(hy.stacked_linear(each, ww), torch.stack([each[i].double() @ ww[i].double().t() for i in range(4)])) < 6e-8, m


@pytest.mark.parametrize("m", [3, 5, 8, 9, 13, 16])
def test_several_products_in_one_launch(m):
    g = torch.Generator(device=DEV).manual_seed(m)
    x = torch.randn(4, m, 512, generator=g, device=DEV).to(BF16)
    w = (torch.randn(4, 260, 512, generator=g, device=DEV) * 512 ** -0.5).to(BF16)
    assert hy.few_bf16(m, w)
    assert _err(hy.stacked_linear(x, w), torch.einsum("emk,enk->emn", x.double(), w.double())) < _tol(512)


@pytest.mark.parametrize("m", [3, 8, 20, 64])
@pytest.mark.parametrize("d", [264, 1024])
def test_norms_gates_and_the_stream(m, d):
    g = torch.Generator(device=DEV).manual_seed(m)
    gain, y = torch.randn(d, generator=g, device=DEV), torch.randn(m, d, generator=g, device=DEV)
    h = hy.RmsInput(y, gain, 1e-5)
    assert torch.equal(h.rows(), hy.rms_rows(y, gain, 1e-5).to(BF16)) and torch.equal(h.value(), hy.rms_rows(y, gain, 1e-5))
    w = (torch.randn(72, d, generator=g, device=DEV) * d ** -0.5).to(BF16)
    table, ids = torch.randn(50, 100, generator=g, device=DEV), torch.arange(m, device=DEV).to(torch.int32) % 50
    r, plain = hy.Residual(y.clone()), hy.Residual(y.clone())
    for q in (r, plain):
        q.add(y, gain, 1e-5)
    x = plain.value()
    got = hy.linear_rows_gated(r, w, ids, table, 20)
    z = x.to(BF16).double() @ w.double().t()
    want = 0.5 * z * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (z + 0.044715 * z ** 3))) * table[ids.long(), 20:92].double()
    assert torch.equal(r.value(), x) and _err(got, want) < 16 * _tol(d)  # (the gate's slope over its size)


@pytest.mark.parametrize("m,d", [(3, 96), (13, 2048)])
@pytest.mark.parametrize("s", [1, 4])
def test_writers_of_blends_and_turned_heads(m, d, s):
    g = torch.Generator(device=DEV).manual_seed(d)
    h, mu, prev = (torch.randn(*z, generator=g, device=DEV) for z in ((m * s, d), (5, d), (m, d)))
    a, b = prev.clone(), prev.clone()
    assert torch.equal(hy.token_shift(h, a, mu, m, s, BF16), hy.token_shift(h, b, mu, m, s).to(BF16)) and torch.equal(a, b)
    if s == 1:
        x = lambda: hy.RmsInput(h, mu[0].contiguous(), 1e-5)
        a, b = prev.clone(), prev.clone()
        assert torch.equal(hy.token_shift(x(), a, mu, m, 1, BF16), hy.token_shift(x(), b, mu, m, 1).to(BF16))
    pos, freq = torch.arange(m * s, device=DEV).to(torch.int32), hy.rotary_freqs(1e4, 16, DEV)
    wide = torch.zeros(m * s, d + 16, dtype=BF16, device=DEV)[:, 8:8 + d]
    want = hy.rotate_heads(h, pos, freq, d // 32, -1.0, 0.7, offset=4)
    assert torch.equal(hy.rotate_heads(h, pos, freq, d // 32, -1.0, 0.7, out=wide, offset=4), want.to(BF16))


@pytest.mark.parametrize("b,t,slot", [(3, 40, 7), (5, 200, 199), (13, 1100, 1050)])
@pytest.mark.parametrize("rope", [False, True])
def test_one_token_of_an_attention(b, t, slot, rope):
    h, g, dim = 4, 2, 64
    gen = torch.Generator(device=DEV).manual_seed(b)
    proj = torch.randn(b, h * dim + 2 * g * dim, generator=gen, device=DEV)
    pos, at = torch.full((b,), slot, dtype=torch.int32, device=DEV), torch.tensor([slot], dtype=torch.int32, device=DEV)
    freq = hy.rotary_freqs(1e4, dim, DEV)
    how = dict(rope=(None, freq, freq, 0.7)) if rope else dict(norm=(1e-5, 0.1, 7))
    got = []
    for dt in (F32, BF16):
        gen.manual_seed(b + 1)
        kc, vc = (torch.randn(b, g, t, dim, generator=gen, device=DEV).to(BF16) for _ in range(2))
        tickets = torch.zeros(b * h * 32, dtype=torch.int32, device=DEV)
        out = torch.zeros(b, h * dim + 16, dtype=dt, device=DEV)[:, 8:8 + h * dim]
        got.append(hy.attn_step(proj, pos, at, tickets, h, True, kc, vc, dim ** -0.5, out=out, **how))
        q = torch.randn(b, 1, h, dim, generator=gen, device=DEV)
        out = torch.zeros(b, h * dim, dtype=dt, device=DEV)
        got.append(hy.attn_bias(q, kc, vc, at, dim ** -0.5, out=out, turn=(pos, freq, -1.0, 0.7) if rope else None))
    assert torch.equal(got[2], got[0].to(BF16)) and torch.equal(got[3], got[1].to(BF16))


@pytest.mark.parametrize("b", [3, 13])
@pytest.mark.parametrize("s", [1, 40])
def test_recurrences(b, s):
    h, dim = 2, 64
    for which in ("memory", "time mix", "delta"):
        got = []
        for dt in (F32, BF16):
            gen = torch.Generator(device=DEV).manual_seed(s)
            rnd = lambda *z: torch.randn(*z, generator=gen, device=DEV)
            out = torch.zeros(b * s, h * dim + 16, dtype=dt, device=DEV)[:, 8:8 + h * dim]
            if which == "memory":
                y = hy.mlstm_memory(rnd(b * s, 4 * h * dim + 2 * h), h, dim, dim, rnd(2 * h), 5.0, rnd(b, h), rnd(b, h, dim, dim + 1), b, s,
                                    rnd(h * dim), 1e-5, 0.5, out)
            elif which == "time mix":
                r, k, v, pre = (rnd(b * s, h, dim) for _ in range(4))
                y = hy.timemix_memory(r, k, v, pre, rnd(h, dim), rnd(h, dim), rnd(b, h, dim, dim), b, s, rnd(b * s, h * dim), rnd(h * dim), 1e-5, 0.5, out)
            else:
                q, k, v = (rnd(b * s, h, dim) for _ in range(3))
                y = hy.delta_memory(q, torch.nn.functional.normalize(k, dim=-1), v, torch.rand(b * s, h, generator=gen, device=DEV), torch.rand(b * s, h, generator=gen, device=DEV),
                                    rnd(b, h, dim, dim), b, s, rnd(b * s, h * dim), rnd(dim), 1e-5, out)
            got.append(y)
        assert got[1].dtype == BF16 and torch.equal(got[1], got[0].to(BF16)), which
