"""A prompt's products on row-major bf16 weights (csrc/hybrid/rows_gemm.hip): tiles of 128 to 256 rows at their edges, with ragged columns,
gated and not, rows by expert with few, many and no rows, against 64-bit sums of the same operands."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV, BF16, F32 = "cuda", torch.bfloat16, torch.float32


def _err(got, want):
    return float((got.double() - want).norm() / want.norm())


def _check(counts, n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    r, e = sum(counts), len(counts)
    x = torch.randn(r, k, generator=g, device=DEV).to(BF16)
    w = (torch.randn(e, 2 * n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    offs = torch.tensor([0] + list(counts)).cumsum(0).to(torch.int32).to(DEV) if e > 1 else None
    src, dst = (torch.randperm(r, generator=g, device=DEV).to(torch.int32) for _ in range(2)) if e > 1 else (None, None)
    bounds = [0] + torch.tensor(counts).cumsum(0).tolist()
    for act, ww in ((hy.ACT_SWIGLU, w), (hy.ACT_NONE, w[:, :n].contiguous())):
        odt = BF16 if act else F32
        out = torch.full((r, n), float("nan"), device=DEV, dtype=odt)
        hy.ext().linear_rows(x, src, ww if e > 1 else ww[0], out, dst, offs, None, r, act, 0.0, 1.0, None, None, 0.0)
        want = torch.empty(r, n, dtype=torch.float64, device=DEV)
        for i in range(e):
            at = slice(bounds[i], bounds[i + 1])
            y = (x[src[at].long()] if e > 1 else x).double() @ ww[i].double().t()
            if act:
                a, b = y.chunk(2, -1)
                y = torch.nn.functional.silu(a) * b
            want[dst[at].long() if e > 1 else slice(None)] = y
        # fp32: exact products, 32 at a time in one chain of k / 32: 6.0e-9 sqrt(k) of the result measured, half as much again
        assert _err(out, want) < (2.0 ** -8 if act else 9e-9 * k ** 0.5), act


# (of 11264 gated columns the choice moves through 128-, 160-, 192- and 256-row tiles)
@pytest.mark.parametrize("rows", [257, 384, 385, 600, 639, 641, 768, 777, 1000, 1537])
def test_one_matrix(rows):
    _check([rows], 5632 if rows % 2 else 5636, 1024 if rows < 700 else 2048, rows)


@pytest.mark.parametrize("counts", [[128, 129, 127, 256], [160, 161, 0, 320], [192, 193, 191, 385], [0, 0, 700, 1], [513, 511, 512, 2000]])
@pytest.mark.parametrize("n,k", [(2820, 1024), (260, 1088)])
def test_rows_by_expert(counts, n, k):
    _check(counts, n, k, 7)


@pytest.mark.parametrize("per", [64, 65, 70, 104, 105])
def test_where_the_tiles_for_fewer_rows_end(per):
    _check([per - 3, per + 3, per, per], 8200, 1024, per)
    _check([per - 3, per + 3, per, per], 512, 1024, per)


@pytest.mark.parametrize("k", [1024, 1088, 1152])  # every phase of the rows' three slots
def test_largest_tiles(k):
    """256 x 256 tiles (rounds enough for them), their last row tile nearly empty, and the activations outside the two fast loops."""
    rows, n = 2050, 30000
    g = torch.Generator(device=DEV).manual_seed(k)
    x = torch.randn(rows, k, generator=g, device=DEV).to(BF16)
    w = (torch.randn(2 * n, k, generator=g, device=DEV) * k ** -0.5).to(BF16)
    y = x.double() @ w.double().t()
    gate, up = y.chunk(2, -1)
    gc, uc = gate.clamp(max=1.5), up.clamp(-1.5, 1.5)
    for act, ww, want in ((hy.ACT_SWIGLU, w, torch.nn.functional.silu(gate) * up), (hy.ACT_NONE, w, y),
                          (hy.ACT_CLAMP_GLU, w, gc * torch.sigmoid(1.7 * gc) * (uc + 1)), (hy.ACT_RELU2, w, y.clamp(min=0) ** 2)):
        out = torch.full((rows, want.shape[1]), float("nan"), device=DEV)
        hy.ext().linear_rows(x, None, ww, out, None, None, None, rows, act, 1.5, 1.7, None, None, 0.0)
        # the product's error as above; each of these activations grows a relative error at most about twice
        assert _err(out, want) < (1 if act == hy.ACT_NONE else 2) * 9e-9 * k ** 0.5 + 2.0 ** -22, act
