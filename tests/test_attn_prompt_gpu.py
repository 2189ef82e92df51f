"""Prompt attention over bf16 caches (csrc/hybrid/attn_bias.hip): many rows at once, whose waves share staged keys or take a query
tile each, against the rows in small groups, whose query tiles are split by their keys; both against the CPU op."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"
HOW = {"plain": {}, "bias": dict(softcap=20.0, bias=40), "chunk": dict(chunk=24, head_scale=True), "sink": dict(sink=True),
       "window": dict(window=37, keep_first=5), "wide": dict(window=70, keep_first=40), "gate": dict(gate_cols=True)}


# query tiles of 32 in all: at most 512 four ways, 1536 two ways, one way above (key widths 64 and 128; both 64: 1024 four ways, one way
# above); 1024 for other widths
@pytest.mark.parametrize("b,s,s0,h,g,dim,vdim", [(20, 97, 0, 8, 2, 128, 128), (33, 65, 63, 8, 4, 64, 64), (20, 127, 130, 8, 8, 64, 128),
                                                 (66, 33, 1, 8, 2, 128, 64), (50, 129, 0, 8, 2, 128, 128), (97, 40, 31, 8, 1, 64, 64),
                                                 (13, 300, 57, 16, 4, 128, 128), (65, 34, 3, 8, 2, 80, 64)])
@pytest.mark.parametrize("how", list(HOW))
def test_all_rows_as_a_few(b, s, s0, h, g, dim, vdim, how):
    torch.manual_seed(1)
    t = s0 + s + 5
    q, kc, vc = torch.randn(b, s, h, dim), torch.randn(b, g, t, dim).bfloat16(), torch.randn(b, g, t, vdim).bfloat16()
    kw = dict(HOW[how])
    if "bias" in kw: kw["bias"] = torch.randn(kw["bias"], h)
    if "head_scale" in kw: kw["head_scale"] = torch.rand(h) + 0.5
    if "sink" in kw: kw["sink"] = torch.randn(h)
    gate = torch.randn(b * s, h * vdim) if "gate_cols" in kw else None
    slot = torch.tensor([s0], dtype=torch.int32, device=DEV)
    dev = {k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()}

    def run(r0, r1):
        more = {} if gate is None else dict(gate=gate[r0 * s:r1 * s].to(DEV))
        return hy.attn_bias(q[r0:r1].to(DEV), kc[r0:r1].to(DEV), vc[r0:r1].to(DEV), slot, dim ** -0.5, **dev, **more).float().cpu()
    whole, group = run(0, b), max(1, 512 // (h * ((s + 31) // 32)))
    small = torch.cat([run(r, min(b, r + group)) for r in range(0, b, group)])
    # the weights' two bf16 parts hold them to 2**-17, whatever maximum they are taken against
    top = float(vc.float().abs().max())
    assert float((whole - small.view_as(whole)).abs().max()) <= 4 * 2.0 ** -17 * top
    want = hy.attn_bias(q[:1].bfloat16().float(), kc[:1], vc[:1], s0, dim ** -0.5, **kw, **({} if gate is None else dict(gate=gate[:s])))
    got = whole.view(b, -1)[0].view_as(want)
    assert float((got - want).abs().max()) <= 4 * 2.0 ** -17 * top + 2e-5


# heads of one query tile: directly from 257 tiles on over at most 256 keys, else four ways; heads of 64 x 64 on either side of 1024 tiles
@pytest.mark.parametrize("b,s,s0,h,g,dim,vdim", [(33, 2, 0, 8, 2, 128, 128), (33, 32, 224, 8, 4, 64, 64), (33, 32, 225, 8, 4, 64, 128), (33, 9, 5, 8, 4, 80, 64), (300, 5, 60, 8, 8, 128, 64),
                                                 (64, 33, 3, 8, 2, 64, 64), (65, 33, 3, 8, 2, 64, 64)])
@pytest.mark.parametrize("how", ["bias", "sink", "window"])
def test_a_head_s_only_tile(b, s, s0, h, g, dim, vdim, how):
    """With the slot on the host, which decides between the forms, and on the device; both as the CPU op on the last row."""
    t = s0 + s + 200
    q, kc, vc = torch.randn(b, s, h, dim).bfloat16().float(), torch.randn(b, g, t, dim).bfloat16(), torch.randn(b, g, t, vdim).bfloat16()
    kw = {"bias": dict(softcap=20.0, bias=torch.randn(40, h)), "sink": dict(sink=torch.randn(h)), "window": dict(window=37, keep_first=5)}[how]
    dev = {k: v.to(DEV) if torch.is_tensor(v) else v for k, v in kw.items()}
    want = hy.attn_bias(q[-1:], kc[-1:], vc[-1:], s0, dim ** -0.5, **kw)
    top = float(vc.float().abs().max())
    both = [hy.attn_bias(q.to(DEV), kc.to(DEV), vc.to(DEV), slot, dim ** -0.5, **dev).cpu()
            for slot in (s0, torch.tensor([s0], dtype=torch.int32, device=DEV))]
    assert float((both[0] - both[1]).abs().max()) <= 4 * 2.0 ** -17 * top  # (the weights' two parts, as above)
    for got in both:
        assert float((got.view(b, s, -1)[-1] - want.view(s, -1)).abs().max()) <= 4 * 2.0 ** -17 * top + 2e-5
