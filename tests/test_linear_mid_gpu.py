"""The tiles of mid-sized batches on packed weights (csrc/kernels/linear_mid.hip): every form with and without a K split, at the edges of
its row tiles and with ragged columns, each epilogue, against 64-bit sums of the same operands; and what the dispatch sends there."""
import pytest
import torch

from jax_llama_amd import ops
from jax_llama_amd.models.weights import PackedLinear
from jax_llama_amd.ops import autotune, reference as ref

pytestmark = pytest.mark.gpu
DEV, BF16 = "cuda", torch.bfloat16


def _tol(k):
    # exact products, summed 32 at a time in fp32 chains of eight: 9e-8 of the result measured (K 2048 to 14336), as much again for the slabs of
    # a split, a residual and the row statistic; the chains' sums in 32 bits where there are many, at most 1.1e-9 sqrt(k) more
    return 1.8e-7 + 1.1e-9 * k ** 0.5


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


def _operands(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device=DEV).to(BF16)
    w = (torch.randn(n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    return x, w, PackedLinear.from_dense(w, torch.device(DEV)).weight


@pytest.mark.parametrize("tile", autotune.MID_TILES)
@pytest.mark.parametrize("m,n,k", [(17, 32, 128), (32, 96, 256), (33, 544, 2048), (64, 64, 1024), (65, 160, 256), (97, 96, 768),
                                   (128, 1056, 1024), (129, 32, 384), (256, 288, 512)])
@pytest.mark.parametrize("splits", [1, 2, 3])
def test_every_form(tile, m, n, k, splits):
    t = k // 64
    if -(-t // -(-t // splits)) != splits or (tile == 35 and t % (2 * splits)):  # (as the plan: whole stages; form 35 takes two at a time)
        pytest.skip("no such split")
    e = ops.ext()
    x, w, pw = _operands(m, n, k)
    y = x.double() @ w.double().t()
    scaled = y * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-5)
    ws = torch.full((splits * m * (n + 1),), float("nan"), device=DEV) if splits > 1 else None
    for eps, want in ((-1.0, y), (1e-5, scaled)):
        out, low = torch.full((m, n), float("nan"), device=DEV), torch.full((m, n), float("nan"), device=DEV, dtype=BF16)
        e.gemm(x, pw, n, k, out, 0, True, None, splits, ws, eps, tile, None, None)
        e.gemm(x, pw, n, k, low, 0, True, None, splits, ws, eps, tile, None, None)
        assert _err(out, want) < _tol(k) and torch.equal(low, out.to(BF16))
        pairs = want.view(m, n // 32, 2, 16)
        glu = (torch.nn.functional.silu(pairs[:, :, 0]) * pairs[:, :, 1]).reshape(m, n // 2)
        act = torch.full((m, n // 2), float("nan"), device=DEV, dtype=BF16)
        pack = ops.packed_empty(m, n // 2, DEV).fill_(0) if m <= 64 and n % 64 == 0 else None
        e.gemm(x, pw, n, k, act, 2, True, None, splits, ws, eps, tile, pack, None)
        assert _err(act, glu) < 2.0 ** -8
        if pack is not None:
            assert torch.equal(ref.unpack_act(pack.cpu(), m), act.cpu())
    h, mirror = torch.randn(m, n, device=DEV), torch.empty(m, n, device=DEV, dtype=BF16)
    want = h.double() + y
    e.gemm(x, pw, n, k, h, 1, True, mirror, splits, ws, -1.0, tile, None, None)
    assert _err(h, want) < _tol(k) and torch.equal(mirror, h.to(BF16))


@pytest.mark.parametrize("m,n,k,before", [(64, 6144, 4096, 1.9e-7), (128, 6144, 4096, 1.27e-7), (64, 4096, 4096, 1.37e-7), (100, 4096, 4096, 1.15e-7),
                                          (64, 28672, 4096, 1.9e-7), (128, 28672, 4096, 2.72e-7), (48, 4096, 14336, 1.87e-7), (128, 4096, 14336, 1.88e-7),
                                          (64, 1280, 8192, 1.39e-7), (128, 1280, 8192, 1.47e-7)])
def test_sums_are_no_less_exact_than_what_they_replaced(m, n, k, before):
    """By the plan, without a norm: the products of bf16 numbers are exact, so the error is the sums' alone; before: what the GEMVs and the
    tiles with K splits had at these sizes."""
    e = ops.ext()
    splits, tile = e.linear_mid_plan(m, n, k)
    assert tile in autotune.MID_TILES
    x, w, pw = _operands(m, n, k)
    out = torch.full((m, n), float("nan"), device=DEV)
    ws = torch.full((splits * m * (n + 1),), float("nan"), device=DEV) if splits > 1 else None
    e.gemm(x, pw, n, k, out, 0, True, None, splits, ws, -1.0, tile, None, None)
    assert _err(out, x.double() @ w.double().t()) < before


@pytest.mark.parametrize("m,heads,kv,k", [(33, 8, 2, 256), (96, 32, 8, 512), (128, 8, 2, 4096), (40, 30, 2, 1024)])
def test_rope_and_cache(m, heads, kv, k, monkeypatch):
    """Their epilogue, with the K split that the plan takes and without one, against the oracle."""
    monkeypatch.setattr(ops, "GEMV_VARIANT", ops.TILED)
    dh, t = 128, 50
    n = (heads + 2 * kv) * dh
    assert ops.ext().linear_mid_plan(m, n, k)[1] in autotune.MID_TILES
    x, w, _ = _operands(m, n, k)
    table, pos = ref.rope_table(dh, 256, 500000.0), torch.randint(0, 200, (m,), dtype=torch.int32)
    kc = torch.zeros(m, kv, t, dh, dtype=BF16)
    vc = torch.zeros_like(kc)
    kg, vg = kc.to(DEV), vc.to(DEV)
    want = ref.linear_qkv_rope(x.cpu(), w.cpu(), 1e-5, table, pos, kc, vc, 11, 1, heads, kv, dh)
    got = ops.linear_qkv_rope(x, PackedLinear.from_dense(w, torch.device(DEV)), 1e-5, table.to(DEV), pos.to(DEV), kg, vg,
                              torch.tensor([11], dtype=torch.int32, device=DEV), 1, heads, kv, dh)
    for a, b in ((got, want), (kg, kc), (vg, vc)):  # (one bf16 rounding here, two in the oracle)
        torch.testing.assert_close(a.float().cpu(), b.float(), rtol=2.0 ** -6, atol=2.0 ** -6)


def test_what_the_dispatch_sends_here_and_replays():
    e = ops.ext()
    for m, n, k, mid in ((16, 4096, 4096, False), (17, 4096, 4096, True), (128, 4096, 4096, True), (256, 4096, 4096, True), (257, 4096, 4096, False),
                         (64, 4096, 96, False), (64, 4104, 4096, False), (64, 4096, 64, False), (96, 128256, 4096, True), (97, 128256, 4096, False)):
        assert (e.linear_mid_plan(m, n, k)[1] in autotune.MID_TILES) == mid, (m, n, k)
    m, n, k = 100, 4096, 2048
    x, w, pw = _operands(m, n, k)
    lin = PackedLinear.from_dense(w, torch.device(DEV))
    ops.linear(x, lin, rms_eps=1e-5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.linear(x, lin, rms_eps=1e-5)
    for i in range(3):
        x.add_(0.5)
        want = ops.linear(x, lin, rms_eps=1e-5)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
    x[7, 5] = float("nan")
    y = ops.linear(x, lin, rms_eps=1e-5)
    keep = [i for i in range(m) if i != 7]
    assert torch.equal(y[keep], out[keep]) and y[7].isnan().all()
