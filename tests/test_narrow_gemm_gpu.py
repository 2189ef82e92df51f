"""Narrow outputs of more rows than the plan tuner measures: K split so that their few tiles fill the chip (csrc/kernels/gemm.hip)."""
import pytest
import torch

from jax_llama_amd import ops
from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,splits", [(4097, 16, 128, 1), (4097, 16, 512, 4), (4160, 64, 4096, 8), (5000, 256, 4096, 2), (5000, 272, 4096, 1),
                                          (12001, 48, 2080, 5), (33000, 64, 1024, 1)])
def test_narrow_output(m, n, k, splits):
    assert ops.ext().gemm_ksplit(m, n, k) == splits
    g = torch.Generator(device="cuda").manual_seed(n)
    x, w = torch.randn(m, k, generator=g, device="cuda").bfloat16(), (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()
    want = x.double() @ w.double().t()
    # exact products, k fp32 additions
    assert float(((hy.linear(x, w).double() - want).abs() / (x.double().abs() @ w.double().abs().t())).max()) < k * 2.0 ** -24


@pytest.mark.parametrize("m,n,k,rest,split", [(4352, 4096, 2048, 256, 8), (4353, 4096, 4096, 257, 8), (8192 + 1, 4096, 1792, 1, 7), (4608, 4112, 14336, 768, 256 // (3 * 17)),
                                              (4097, 4096, 1024, 0, 1), (18432, 2048, 2048, 0, 1), (17000, 2048, 2048, 616, 8), (8192, 4096, 4096, 0, 1), (6656, 4096, 4096, 0, 1)])
@pytest.mark.parametrize("mirrored", [True, False])
def test_rows_behind_the_whole_rounds(m, n, k, rest, split, mirrored):
    """The rows whose tiles start a mostly empty round have K split, in a launch of their own; all rows against 64 bits."""
    e = ops.ext()
    assert e.gemm_tail(m, n, k, True) == (rest, split)
    g = torch.Generator(device="cuda").manual_seed(m)
    x, w = torch.randn(m, k, generator=g, device="cuda").bfloat16(), (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).bfloat16()
    pw, h = hy._packed_weight(w), torch.randn(m, n, generator=g, device="cuda")
    was, mirror = h.clone(), torch.zeros(m, n, dtype=torch.bfloat16, device="cuda") if mirrored else None
    ops.linear_residual(x, pw, h, mirror=mirror)
    y = ops.linear(x, pw, out_dtype=torch.float32)
    rows = torch.cat([torch.arange(0, 64), torch.arange(m - rest - 64, m - rest + 64).clamp(max=m - 1), torch.arange(m - 64, m)]).unique().cuda()
    want, size = x[rows].double() @ w.double().t(), x[rows].double().abs() @ w.double().abs().t()
    tol = (k + 2) * 2.0 ** -24 * size + 2.0 ** -24 * (was[rows].double().abs() + size)
    assert bool(((h[rows].double() - was[rows].double() - want).abs() <= tol).all()) and bool(((y[rows].double() - want).abs() <= tol).all())
    if mirrored:
        assert torch.equal(mirror, h.bfloat16())
