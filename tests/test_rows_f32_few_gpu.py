"""One and two rows on fp32 weights (csrc/hybrid/rows_gemv.hip, ``rows_walk_f32_kernel``): K at the edges of its forms, ragged columns, gated
and not, normed, with a pending residual add, several matrices at once and rows with an expert each, against 64-bit sums."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV, F32, F64 = "cuda", torch.float32, torch.float64
# up to 16 products one behind the other in each of two chains and their join, the 256 threads' parts added in 64 bits: roundings of random
# sign, sqrt(17) 2^-24 = 2.5e-7 of the sum's share; a norm or a gate adds a few more of one number
TOL = 6e-7


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


def _rand(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _rms(x, gain, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * gain


# (columns: groups of one, two and four weight rows, and remainders of them)
@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("k", [512, 1020, 1024, 1028, 2048, 2052, 4096, 4100, 5632, 6144, 6148, 8192, 8196])
@pytest.mark.parametrize("n", [17, 1027, 4101])
def test_rows(rows, k, n):
    g = torch.Generator(device=DEV).manual_seed(k + n + rows)
    x, w, gain = _rand(g, 2, k)[:rows], _rand(g, 2 * n, k) * k ** -0.5, _rand(g, k)
    for gated in (False, True):
        for normed in (False, True):
            ww = w if gated else w[:n].contiguous()
            out = torch.full((rows, n), float("nan"), device=DEV)
            hy.ext().linear_rows(x, None, ww, out, None, None, None, rows, hy.ACT_SWIGLU if gated else hy.ACT_NONE, 0.0, 1.0, None,
                                 gain if normed else None, 1e-5)
            y = (_rms(x.double(), gain.double(), 1e-5) if normed else x.double()) @ ww.double().t()
            if gated:
                y = torch.nn.functional.silu(y[:, :n]) * y[:, n:]
            assert _err(out, y) < TOL, (gated, normed)


def test_infinite_weights_stay_in_their_columns():
    w = torch.ones(40, 1028, device=DEV)
    w[3, 0], w[5, 1027] = float("inf"), float("-inf")
    out = hy.linear(torch.ones(1, 1028, device=DEV), w)
    want = torch.full((1, 40), 1028.0, device=DEV)
    want[0, 3], want[0, 5] = float("inf"), float("-inf")
    assert torch.equal(out, want)


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("k", [1024, 2048, 2816, 4096])
def test_pending_add_and_gate(rows, k):
    g = torch.Generator(device=DEV).manual_seed(k)
    x, y, rw, w, gain = _rand(g, rows, k), _rand(g, 2 * rows, k), _rand(g, k), _rand(g, 66, k) * k ** -0.5, _rand(g, k)
    table, ids = _rand(g, 9, 80), torch.tensor([8, 3][:rows], device=DEV)
    want_x = x.double() + _rms(y.double().view(rows, 2, k).sum(1) * 0.5, rw.double(), 1e-6)
    r = hy.Residual(x.clone())
    r.add(y, rw, 1e-6, 2, 0.5)
    got = hy.linear_rows_gated(r, w, ids, table, 7)
    assert r.pending is None  # (it was one launch)
    z = want_x @ w.double().t()
    want = torch.nn.functional.gelu(z, approximate="tanh") * table[ids][:, 7:73].double()
    assert _err(r.value(), want_x) < TOL and _err(got, want) < TOL
    r = hy.Residual(x.clone())
    r.add(y, rw, 1e-6, 2, 0.5)
    assert _err(hy.head_linear(r, gain, 1e-5, w, 30.0), 30 * torch.tanh(_rms(want_x, gain.double(), 1e-5) @ w.double().t() / 30)) < TOL


@pytest.mark.parametrize("rows", [1, 2])
@pytest.mark.parametrize("k", [256, 2048, 2056, 4096])
def test_several_matrices(rows, k):
    g = torch.Generator(device=DEV).manual_seed(k)
    x, gain, prev, mu = _rand(g, rows, k), _rand(g, k), _rand(g, rows, k), torch.rand(2, k, generator=g, device=DEV)
    ws = [_rand(g, n, k) * k ** -0.5 for n in (1030, 64, 515)]
    outs, row = hy.shifted_linears(hy.RmsInput(x, gain, 1e-5), prev, mu, [(ws[0], -1, 0.0), (ws[1], 1, 2.0), (ws[2], 0, 0.0)])
    v = _rms(x.double(), gain.double(), 1e-5)
    mixed = [v + (prev.double() - v) * m.double() for m in mu]
    assert _err(row, v) < TOL and _err(outs[0], v @ ws[0].double().t()) < TOL
    assert _err(outs[1], 2 * torch.tanh(mixed[1] @ ws[1].double().t() / 2)) < TOL
    assert _err(outs[2], mixed[0] @ ws[2].double().t()) < TOL


@pytest.mark.parametrize("tokens", [1, 2, 4])
def test_experts_by_table(tokens):
    g = torch.Generator(device=DEV).manual_seed(tokens)
    k, f, e, top = 1024, 515 * 4, 5, 2
    x, gu, down = _rand(g, tokens, k), _rand(g, e, 2 * f, k) * k ** -0.5, _rand(g, e, k, f) * f ** -0.5
    table = torch.rand(11, e, generator=g, device=DEV).argsort(1)[:, :top].to(torch.int32).contiguous()
    ids = torch.tensor([10, 0, 7, 3][:tokens], device=DEV)
    y = torch.empty(tokens * top, k, device=DEV)
    h = torch.empty(tokens * top, f, device=DEV)
    assert hy.ext().table_rows(x, ids.to(torch.int32), table, gu, down, h, y, None, 1, 1.0, None, 0.0, None)
    for t in range(tokens):
        for c in range(top):
            i = int(table[ids[t], c])
            z = x[t].double() @ gu[i].double().t()
            a = torch.nn.functional.silu(z[:f]) * z[f:]
            assert _err(y[t * top + c], a @ down[i].double().t()) < 2 * TOL  # (two products)
