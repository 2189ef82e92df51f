"""Per-head norms in groups of lanes (attn_prep in csrc/hybrid/attn_bias.hip, gated_rmsnorm in delta_rule.hip) against the CPU ops, at
the edges of the groups and where the separate kernel runs (odd sizes, unaligned rows)."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"
# a norm's statistic, root and three products round by 2^-24 each, the sum of n squares by at most log2(n) + 2 of it
TOL = 16 * 2.0 ** -24


@pytest.mark.parametrize("dim,vdim", [(4, 4), (60, 64), (64, 64), (68, 128), (128, 64), (128, 128), (132, 256), (256, 4), (256, 260), (66, 64)])
@pytest.mark.parametrize("h,g,pad", [(1, 1, 0), (6, 2, 4), (5, 5, 3)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("own", [True, False])
def test_attn_prep(dim, vdim, h, g, pad, dt, own):
    b, s, s0, t = 2, 7, 3, 9  # (the last token of a row has no slot left)
    gen = torch.Generator().manual_seed(dim * h)
    proj = torch.randn(b * s, h * dim + g * (dim + vdim) + pad, generator=gen)
    pos = torch.arange(b * s, dtype=torch.int32) * 400
    kw = dict(temp_coef=0.1, temp_every=512, q_w=torch.randn(dim, generator=gen), k_w=torch.randn(dim, generator=gen), norm_v=h != 5)
    out = []
    for dev in ("cpu", DEV):
        n = s if dev == DEV else s - 1
        kc, vc = torch.zeros(b, g, t, dim, dtype=dt, device=dev), torch.zeros(b, g, t, vdim, dtype=dt, device=dev)
        rows = torch.arange(b * s).reshape(b, s)[:, :n].reshape(-1)
        cols = h * dim + (g * (dim + vdim) if own else 0)
        q = hy.attn_prep(proj[rows].to(dev)[:, :cols], pos[rows].to(dev), torch.tensor([s0], dtype=torch.int32, device=dev), b, n, h, g, dim, vdim,
                         kc if own else None, vc if own else None, 1e-5, **{k: v.to(dev) if torch.is_tensor(v) else v for k, v in kw.items()})
        out.append([x.float().cpu() for x in (q[:, :s - 1], kc, vc)])
    for want, got in zip(*out):
        assert float(((got - want).abs() / want.abs().clamp_min(1e-6)).max()) <= (TOL if want is out[0][0] or dt == torch.float32 else 2.0 ** -7)


@pytest.mark.parametrize("vdim", [4, 64, 68, 128, 200, 256, 260, 66])
@pytest.mark.parametrize("m,h", [(1, 1), (5, 3), (300, 6)])
@pytest.mark.parametrize("act", [hy.GATE_SILU, hy.GATE_SIGMOID, hy.GATE_NONE])
@pytest.mark.parametrize("dt,col", [(torch.float32, 0), (torch.bfloat16, 4), (torch.float32, 3)])
def test_gated_rmsnorm(vdim, m, h, act, dt, col):
    gen = torch.Generator().manual_seed(vdim + m)
    o, gate = torch.randn(m, h, vdim, generator=gen), torch.randn(m, h * vdim + 8, generator=gen)[:, col:col + h * vdim]
    w = torch.randn(h * vdim if m == 5 else vdim, generator=gen)
    want = hy.gated_rmsnorm(o, None if act == hy.GATE_NONE else gate, w, 1e-5, act, gain=0.5)
    wide = torch.full((m, h * vdim + 8), 7.0, dtype=dt, device=DEV)
    hy.gated_rmsnorm(o.to(DEV), None if act == hy.GATE_NONE else gate.to(DEV), w.to(DEV), 1e-5, act, gain=0.5, out=wide[:, col:col + h * vdim])
    got = wide.float().cpu()
    assert bool((got[:, :col] == 7).all()) and bool((got[:, col + h * vdim:] == 7).all())
    got = got[:, col:col + h * vdim]
    assert float(((got - want).abs() / want.abs().clamp_min(1e-6)).max()) <= (TOL if dt == torch.float32 else 2.0 ** -8 + TOL)


@pytest.mark.parametrize("vdim,m,h", [(64, 1365, 3), (64, 1366, 3), (60, 4096, 1), (4, 820, 5)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_gated_rmsnorm_of_many_narrow_heads(vdim, m, h, dt):
    """Heads of up to 64 numbers on either side of the 4096 heads from which they run in groups of lanes."""
    test_gated_rmsnorm(vdim, m, h, hy.GATE_SILU, dt, 4)


@pytest.mark.parametrize("m,d", [(256, 264), (300, 1024), (256, 4096), (257, 8200), (256, 200)])
@pytest.mark.parametrize("nsum", [1, 2])
def test_residual_as_an_operand(m, d, nsum):
    """The stream rounded by the kernel that adds to it: what rounding it afterwards gives, again after another addition."""
    gen = torch.Generator(device=DEV).manual_seed(d)
    r, plain = (hy.Residual(torch.ones(m, d, device=DEV)) for _ in range(2))
    assert torch.equal(r.operand(torch.bfloat16), r.x.bfloat16())
    for _ in range(2):
        y, w = torch.randn(m * nsum, d, generator=gen, device=DEV), torch.randn(d, generator=gen, device=DEV)
        r.add(y, w, 1e-5, nsum, 0.5)
        plain.add(y, w, 1e-5, nsum, 0.5)
        rows = r.operand(torch.bfloat16)
        assert rows.dtype == torch.bfloat16 and torch.equal(rows, plain.value().bfloat16()) and r.operand(torch.bfloat16) is rows
        assert torch.equal(r.value(), plain.x) and r.operand(torch.float32).dtype == torch.float32
        for x in (r, plain):
            x.value().mul_(0.5)  # (a block that adds to the stream in place)
        assert torch.equal(r.operand(torch.bfloat16), plain.x.bfloat16())
    assert hy.Residual(torch.ones(3, 8, device=DEV)).operand(torch.bfloat16).dtype == torch.float32
