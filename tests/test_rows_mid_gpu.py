"""Products of some ten to a few hundred rows on row-major bf16 weights (csrc/hybrid/rows_mid.hip): tile edges, ragged columns,
K splits, strided rows, rows by expert with empty and full ones, every activation, against 64-bit sums of the same operands."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF16 = torch.bfloat16


def _tol(k):
    # exact products, 32 at a time in an fp32 chain of k / 32: 6.0e-9 sqrt(k) of the result measured (K 2048, 4096, 7168: 2.7e-7, 3.95e-7, 5.3e-7),
    # half as much again for short sums of few numbers, and the result's own rounding with an add behind it
    return 9e-9 * k ** 0.5 + 1.2e-7


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


def _operands(m, n, k, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(m, k, generator=g, device=DEV),
            (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF16))


def _act64(y, act, limit, alpha):
    if act == hy.ACT_RELU2:
        return y.clamp_min(0).square()
    if act == hy.ACT_SOFTCAP:
        return limit * torch.tanh(y / limit)
    if not hy.act_gated(act):
        return y
    g, u = y.chunk(2, -1)
    if act == hy.ACT_SWIGLU:
        return torch.nn.functional.silu(g) * u
    if act == hy.ACT_GELU_GLU:
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    g = g.clamp(max=limit)
    return g * torch.sigmoid(alpha * g) * (u.clamp(-limit, limit) + 1)


@pytest.mark.parametrize("m,n,k", [(9, 4, 1024), (16, 64, 1088), (17, 68, 1024), (25, 36, 128), (31, 2048, 192), (33, 516, 640),
                                   (48, 132, 2048), (64, 36, 4096), (65, 20, 128), (97, 132, 320), (128, 64, 4096), (129, 256, 256),
                                   (200, 2048, 2048), (255, 1028, 192), (256, 64, 128), (257, 96, 128)])
def test_one_matrix(m, n, k):
    x, w = _operands(m, n, k)
    assert hy.ext().rows_mid_takes(m, w, hy.ACT_NONE) == (m <= 255)
    want = x.to(BF16).double() @ w.double().t()
    assert _err(hy.linear(x, w), want) < _tol(k)
    wide = torch.full((m, k + 12), float("nan"), device=DEV)  # (rows 16 bytes and an odd distance apart, and off 16 bytes)
    for at in (4, 3):
        wide[:, at:at + k] = x
        assert _err(hy.linear(wide[:, at:at + k], w), want) < _tol(k)
    res = torch.randn(m, n, device=DEV)
    want2 = res.double() + want
    assert _err(hy.linear_add_(res, x, w), want2) < _tol(k)


@pytest.mark.parametrize("k,n", [(2048, 2048), (4096, 4096), (7168, 4096)])
def test_up_to_64_rows_are_summed_in_64_bits(k, n):
    """Products of bf16 numbers are exact in fp32, so the error against 64 bits is the sums' alone: no more than the few-row products
    have that take such rows at other sizes (their test: 7.6e-8) for rows by expert, sorted or as many each, whose every four products meet in 64
    bits; for dense rows, eight products, 8.9e-8 to 9.4e-8 measured where four fp32 chains had 1.3e-7 and more."""
    g = torch.Generator(device=DEV).manual_seed(k)
    w = (torch.randn(8, n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    for r in (9, 16, 33, 64):
        x = torch.randn(r, k, generator=g, device=DEV).to(BF16)
        want = x.double() @ w[0].double().t()
        for a in (x, x.float()):
            assert _err(hy.linear(a, w[0]), want) < 1.1e-7, (r, a.dtype)
        if r <= 16:
            each = torch.randn(4, r, k, generator=g, device=DEV).to(BF16)
            assert _err(hy.stacked_linear(each, w[:4]), torch.stack([each[i].double() @ w[i].double().t() for i in range(4)])) < 7.6e-8, r
    for r in (40, 64):
        x = torch.randn(r, k, generator=g, device=DEV).to(BF16)
        ex = torch.randint(0, 8, (r,), generator=g, device=DEV)
        order = torch.argsort(ex, stable=True).to(torch.int32)
        offs = torch.tensor([int((ex < i).sum()) for i in range(9)], dtype=torch.int32, device=DEV)
        out = torch.full((r, n), float("nan"), device=DEV)
        hy.ext().linear_rows(x.float(), order, w, out, order, offs, None, r, hy.ACT_NONE, 0.0, 1.0, None, None, 0.0)
        assert _err(out, torch.stack([w[int(ex[i])].double() @ x[i].double() for i in range(r)])) < 7.6e-8, r


@pytest.mark.parametrize("act", [hy.ACT_RELU2, hy.ACT_SWIGLU, hy.ACT_CLAMP_GLU, hy.ACT_SOFTCAP, hy.ACT_GELU_GLU])
@pytest.mark.parametrize("m,n,k", [(9, 20, 1024), (40, 68, 2048), (70, 516, 192), (250, 32, 640), (256, 48, 128)])
def test_activations(act, m, n, k):
    x, w = _operands(m, 2 * n if hy.act_gated(act) else n, k, 1)
    want = _act64(x.to(BF16).double() @ w.double().t(), act, 1.3, 1.702)
    # (an activation amplifies the sums' error by its slope over its size; 16 covers these at sums around 1)
    assert _err(hy.linear(x, w, act=act, limit=1.3, alpha=1.702), want) < 16 * _tol(k)


@pytest.mark.parametrize("counts", [[0, 70, 0, 1], [16, 17, 33, 64], [0, 0, 0, 100], [112, 96, 129, 111], [9, 31, 32, 8]])
@pytest.mark.parametrize("n,k", [(36, 128), (260, 2048), (64, 704)])
@pytest.mark.parametrize("rows", ["f32", "bf16"])
def test_rows_by_expert(counts, n, k, rows):
    e, r = len(counts), sum(counts)
    g = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn(r, k, generator=g, device=DEV)
    w = (torch.randn(e, 2 * n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(DEV)
    src, dst = (torch.randperm(r, generator=g, device=DEV).to(torch.int32) for _ in range(2))
    a = x.to(BF16) if rows == "bf16" else x
    ops = hy.ext()
    for act, ww in ((hy.ACT_SWIGLU, w), (hy.ACT_NONE, w[:, :n].contiguous())):
        odt = BF16 if rows == "bf16" and act == hy.ACT_SWIGLU else torch.float32
        out = torch.full((r, n), float("nan"), device=DEV, dtype=odt)
        ops.linear_rows(a, src, ww, out, dst, offs, None, r, act, 0.0, 1.0, None, None, 0.0)
        want = torch.empty(r, n, dtype=torch.float64, device=DEV)
        for i in range(e):
            at = slice(int(offs[i]), int(offs[i + 1]))
            want[dst[at].long()] = _act64(x.to(BF16)[src[at].long()].double() @ ww[i].double().t(), act, 0, 1)
        assert _err(out, want) < (2.0 ** -8 if odt == BF16 else 16 * _tol(k))


@pytest.mark.parametrize("rows", ["f32", "bf16"])
@pytest.mark.parametrize("act", [hy.ACT_NONE, hy.ACT_SWIGLU])
def test_rows_of_experts_without_weights_are_left_alone(rows, act):
    """Rows behind the last offset (identity experts) keep what the output holds, with a K split as without one."""
    for n, k in ((64, 4096), (64, 128), (4096, 1024)):
        g = torch.Generator(device=DEV).manual_seed(k)
        x = torch.randn(100, k, generator=g, device=DEV).to(BF16)
        w = (torch.randn(2, 2 * n if hy.act_gated(act) else n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
        offs = torch.tensor([0, 30, 77], dtype=torch.int32, device=DEV)
        dst = torch.randperm(100, generator=g, device=DEV).to(torch.int32)
        out = torch.full((100, n), 7.0, device=DEV)
        hy.ext().linear_rows(x if rows == "bf16" else x.float(), None, w, out, dst, offs, None, 100, act, 0.0, 1.0, None, None, 0.0)
        assert (out[dst[77:].long()] == 7.0).all(), (n, k)
        for lo, hi, i in ((0, 30, 0), (30, 77, 1)):
            assert _err(out[dst[lo:hi].long()], _act64(x[lo:hi].double() @ w[i].double().t(), act, 0, 1)) < 16 * _tol(k)


def test_a_row_that_is_no_number_stays_in_its_row_and_replays_repeat():
    m, n, k = 70, 132, 2048
    x, w = _operands(m, n, k, 3)
    clean = hy.linear(x, w)
    x[5, 3], x[69, 0] = float("nan"), float("inf")
    y = hy.linear(x, w)
    keep = [i for i in range(m) if i not in (5, 69)]
    assert torch.equal(y[keep], clean[keep]) and y[5].isnan().all() and not y[69].isfinite().any()
    x[5, 3], x[69, 0] = 1.0, 1.0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = hy.linear(x, w)
    for i in range(3):
        x.add_(0.5)
        want = hy.linear(x, w)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
