"""fp32 products on the bf16 matrix cores (csrc/kernels/gemm_f32x3.h) with enough tiles for the wide form, and at the edges of both."""
import pytest
import torch

from jax_llama_amd import ops
from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m,n,k", [(1, 16644, 8), (127, 33028, 40), (129, 8196, 520), (640, 9004, 96), (1000, 4100, 2080), (257, 260, 1032)])
@pytest.mark.parametrize("act", [hy.ACT_NONE, hy.ACT_SWIGLU])
def test_wide_tiles(m, n, k, act):
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x, w = torch.randn(m, k, generator=g, device=DEV), torch.randn(n, k, generator=g, device=DEV) * k ** -0.5
    y, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # a product leaves out 2^-24 of itself; the 24 roundings of a step of 32 are of the step's sum, one per step of the whole
    bound = 2.0 ** -24 * (1 + 24 + (k + 31) // 32 + 16) * size
    if act == hy.ACT_NONE:
        assert float(((ops.linear_f32(x, w).double() - y).abs() / bound).max()) < 1
        got = [hy.linear(x, w)]
    else:
        got, y, size = [hy.linear(x, w, act=act)], torch.nn.functional.silu(y[:, :n // 2]) * y[:, n // 2:], size
        bound = bound[:, :n // 2] * (1.1 * (x.double() @ w.double().t()).abs()[:, n // 2:]) + bound[:, n // 2:] * (
            x.double() @ w.double().t()).abs()[:, :n // 2] + 2e-6 * y.abs() + 1e-6
    for o in got:
        assert float(((o.double() - y).abs() / bound).max()) < 1


@pytest.mark.parametrize("row,col", [(0, 0), (127, 255), (128, 256), (129, 8195)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 1e-41])
def test_wide_tile_with_a_number_the_split_does_not_hold(row, col, bad):
    g = torch.Generator().manual_seed(row + col)
    x, w = torch.randn(130, 264, generator=g), torch.randn(8196, 264, generator=g)
    x[row, 263], w[col, 3] = bad, bad
    want, got = x @ w.t(), ops.linear_f32(x.to(DEV), w.to(DEV)).cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    ok = torch.isfinite(want)
    assert float((got - want)[ok].abs().max()) < 2.0 ** -24 * 2 * 264 * float((x.abs()[ok.any(1)].nan_to_num(0, 0, 0)).max() * 4)
