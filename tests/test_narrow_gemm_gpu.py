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
