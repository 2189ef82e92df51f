"""One token per row through the kernels that fuse a decode step's launches (csrc/hybrid/attn_step.hip), against the separate ops
on the CPU, at the edges of their key splits and caches."""
import pytest
import torch

from jax_llama_amd.ops import hybrid as hy

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF16 = torch.bfloat16


def _rand(*shape, dt=torch.float32, std=1.0):
    return (torch.randn(*shape) * std).to(dt)


def _close(a, b, tol, what):
    a, b = a.float().cpu(), b.float().cpu()
    assert a.shape == b.shape, what
    err = float((a - b).abs().max() / b.abs().max().clamp_min(1e-6))
    assert err <= tol, f"{what}: relative error {err:.3e} > {tol:.1e}"


def _to(x):
    return None if x is None else x.to(DEV)


SHAPES = [  # rows, heads, key heads, key width, value width, cache length, slot
    (1, 4, 2, 64, 64, 40, 0), (1, 4, 1, 128, 128, 200, 63), (2, 4, 2, 128, 64, 200, 64), (3, 2, 2, 64, 128, 200, 65),
    (1, 16, 4, 128, 128, 2112, 2080), (1, 8, 2, 128, 128, 2112, 2111), (1, 2, 1, 128, 128, 1100, 1023), (1, 2, 1, 64, 64, 1100, 1024),
    (5, 4, 4, 128, 128, 64, 1), (1, 2, 1, 64, 64, 1, 0), (60, 4, 2, 64, 64, 130, 100), (1, 30, 10, 64, 128, 2600, 2570), (2, 2, 1, 128, 128, 90, 90)]


@pytest.mark.parametrize("b,h,g,dim,vdim,t,slot", SHAPES)
@pytest.mark.parametrize("kind", ["norm", "norm-shared", "rope", "rope-chunk", "rope-sink"])
@pytest.mark.parametrize("dt", [BF16, torch.float32])
def test_attention_of_one_token(b, h, g, dim, vdim, t, slot, kind, dt):
    """Projection to head output, and the cache row written (none when the cache is full: slot == t), as the separate ops; the
    tickets are back at zero, so that a second step on the same buffers gives the same."""
    own = kind != "norm-shared"
    if not own and slot >= t:
        slot = t - 1
    cols = h * dim + (g * (dim + vdim) if own else 0)
    proj = _rand(b, cols + 8)[:, :cols]
    kc, vc = _rand(b, g, t, dim, dt=dt), _rand(b, g, t, vdim, dt=dt)
    pos = torch.full((b,), slot, dtype=torch.int32) + torch.arange(b, dtype=torch.int32)
    slot_t, full = torch.tensor([slot], dtype=torch.int32), slot >= t
    scale, kr, vr = dim ** -0.5, kc.clone(), vc.clone()
    args = dict(softcap=0.0, bias=None, sink=None, chunk=0, head_scale=None)
    out = None
    if kind.startswith("norm"):
        args.update(softcap=20.0, bias=_rand(50, h))
        q = hy.attn_prep(proj, pos, min(slot, t - 1), b, 1, h, g, dim, vdim, kr if own else None, vr if own else None, 1e-5, 0.1, 7)
        how = dict(norm=(1e-5, 0.1, 7))
    else:
        freq, vf = hy.rotary_freqs(1e4, dim // 2, "cpu"), (None if kind == "rope-sink" else hy.rotary_freqs(1e4, vdim, "cpu"))
        cb = _rand(cols)
        args.update(head_scale=torch.rand(h) + 0.5, chunk=64 if kind == "rope-chunk" else 0, sink=_rand(h) if kind == "rope-sink" else None)
        q = hy.rope_prep(proj, cb, pos, min(slot, t - 1), b, 1, h, g, dim, vdim, kr, vr, freq, vf)
        out = torch.zeros(b, h * vdim + 24, device=DEV)[:, 8:8 + h * vdim]
        how = dict(rope=(cb.to(DEV), freq.to(DEV), _to(vf), 0.7))
    if full:
        kr, vr = kc.clone(), vc.clone()  # the token's own key is dropped
    kd, vd, tickets = kc.to(DEV), vc.to(DEV), torch.zeros(b * h * 32, dtype=torch.int32, device=DEV)
    for _ in range(2):
        kd.copy_(kc), vd.copy_(vc)
        got = hy.attn_step(proj.to(DEV).as_strided((b, cols), (cols, 1)) if proj.is_contiguous() else _strided(proj), pos.to(DEV),
                           slot_t.to(DEV), tickets, h, own, kd, vd, scale, **{k: _to(v) if torch.is_tensor(v) else v for k, v in args.items()},
                           out=out, **how)
        assert got is not None
        # the output over the cache as this step left it: the last bit of a prepared key in 32 bits may round it to either of two
        # neighbouring bf16 numbers
        a = hy.attn_bias(q, kd.cpu(), vd.cpu(), min(slot, t - 1), scale, args["softcap"], args["bias"], sink=args["sink"],
                         chunk=args["chunk"], head_scale=args["head_scale"])
        if not kind.startswith("norm"):
            a = hy.rotate_heads(a, pos, vf, h, sign=-1.0, gain=0.7)
        _close(got, a, 2e-5, "output")
        tol = (2.0 ** -7 if dt == BF16 else 2e-6) if own else 0.0
        _close(kd, kr, tol, "keys"), _close(vd, vr, tol, "values")
        keep = torch.arange(t) != slot
        assert torch.equal(kd.cpu()[:, :, keep], kc[:, :, keep]) and torch.equal(vd.cpu()[:, :, keep], vc[:, :, keep])
        assert not tickets.any()


def _strided(x):
    big = torch.zeros(x.shape[0], x.shape[1] + 8, device=DEV)
    big[:, :x.shape[1]] = x.to(DEV)
    return big[:, :x.shape[1]]


@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("d", [256, 264, 2048, 2056, 4096])
def test_inputs_of_a_token_shift_in_one_launch(m, d):
    """Products of the normed row and of its blends with the row before it, as the norm, the blend and the products one by one; odd
    widths, a capped part, a part of one column, and more columns than are resident at once."""
    x, gain, prev, mu = _rand(m, d), torch.rand(d) + 0.5, _rand(m, d), torch.rand(3, d)
    parts = [(_rand(n, d, dt=BF16, std=d ** -0.5), j, cap) for n, j, cap in ((70, -1, 0.0), (1, 2, 0.0), (8200, 0, 0.0), (33, 1, 1.0), (4, 2, 0.5))]
    h = hy.RmsInput(x.to(DEV), gain.to(DEV), 1e-5)
    got = hy.shifted_linears(h, prev.to(DEV), mu.to(DEV), [(w.to(DEV), j, c) for w, j, c in parts])
    assert got is not None
    row = hy.rms_rows(x, gain, 1e-5)
    _close(got[1], row, 2e-6, "row")
    for y, (w, j, cap) in zip(got[0], parts):
        v = got[1].cpu() if j < 0 else hy.token_shift(got[1].cpu(), prev.clone(), mu, m, 1)[j]
        ref = hy.linear(v, w)
        # (a blend's last bit in 32 bits may round it to either of two bf16 neighbours: one number of d, 2^-8 of it)
        _close(y, cap * torch.tanh(ref / cap) if cap else ref, 2e-5 + 2.0 ** -8 * d ** -0.5, f"part of {w.shape[0]}")


@pytest.mark.parametrize("dt", [BF16, torch.float32])
@pytest.mark.parametrize("b,h,dim,rank,width", [(1, 3, 64, 64, 200), (2, 2, 64, 4, 64), (1, 4, 128, 36, 5000), (3, 2, 20, 60, 40), (1, 2, 256, 64, 512)])
def test_time_mix_of_one_token_takes_its_decay_product(dt, b, h, dim, rank, width):
    hd = (h, dim)
    r, k, v = (_rand(b, *hd) for _ in range(3))
    z, w2, w0, u, gate, w = torch.tanh(_rand(b, rank)), _rand(h * dim, rank, dt=dt, std=rank ** -0.5), _rand(*hd) - 2.0, _rand(*hd), _rand(b, h * dim), torch.rand(h * dim)
    st, prev, row = _rand(b, h, dim, dim), _rand(b, width), _rand(b, width)
    s_dev, p_dev = st.to(DEV), prev.to(DEV)
    got = hy.timemix_memory(*(t.to(DEV) for t in (r, k, v)), (z.to(DEV), w2.to(DEV)), w0.to(DEV), u.to(DEV), s_dev, b, 1, gate.to(DEV), w.to(DEV),
                            1e-5, 0.7, carry=(p_dev, row.to(DEV)))
    want = hy.timemix_memory(r, k, v, (z, w2), w0, u, st, b, 1, gate, w, 1e-5, 0.7, carry=(prev, row))
    _close(got, want, 2e-5, "output"), _close(s_dev, st, 2e-5, "state")
    assert torch.equal(p_dev.cpu(), row) and torch.equal(prev, row)


@pytest.mark.parametrize("m,before", [(1, 194), (1, 1), (2, 67), (1, 64)])
@pytest.mark.parametrize("moved", [False, True])
def test_time_mix_behind_a_part_of_any_width(m, before, moved):
    """The decay product's input from the joint launch behind a matrix whose row count is no multiple of four, and as a view that
    does not start on 16 bytes: the same as from memory of its own."""
    d, hd, rank = 256, (2, 64), 64
    x, gain, prev, mu = _rand(m, d), torch.rand(d) + 0.5, _rand(m, d), torch.rand(2, d)
    w_also, w1, w2 = _rand(before, d, dt=BF16), _rand(rank, d, dt=BF16, std=d ** -0.5), _rand(128, rank, dt=BF16, std=rank ** -0.5)
    outs, _ = hy.shifted_linears(hy.RmsInput(x.to(DEV), gain.to(DEV), 1e-5), prev.to(DEV), mu.to(DEV),
                                 [(w_also.to(DEV), -1, 0.0), (w1.to(DEV), 1, 1.0)])
    z = outs[1]
    if moved:
        z = torch.zeros(m * rank + 2, device=DEV)[2:].view(m, rank).copy_(z)
    r, k, v, w0, u, gate, w = _rand(m, *hd), _rand(m, *hd), _rand(m, *hd), _rand(*hd) - 2.0, _rand(*hd), _rand(m, 128), torch.rand(128)
    st = _rand(m, 2, 64, 64)
    s_dev, s_own = st.to(DEV), st.to(DEV)
    args = [t.to(DEV) for t in (w0, u)]
    got = hy.timemix_memory(*(t.to(DEV) for t in (r, k, v)), (z, w2.to(DEV)), *args, s_dev, m, 1, gate.to(DEV), w.to(DEV), 1e-5)
    want = hy.timemix_memory(*(t.to(DEV) for t in (r, k, v)), (z.clone(), w2.to(DEV)), *args, s_own, m, 1, gate.to(DEV), w.to(DEV), 1e-5)
    _close(got, want.cpu(), 2e-5, "output"), _close(s_dev, s_own.cpu(), 2e-5, "state")


@pytest.mark.parametrize("b,h,g,dim,vdim", [(1, 4, 1, 128, 128), (2, 4, 2, 64, 64), (3, 3, 3, 40, 20), (1, 16, 4, 128, 128), (2, 6, 2, 200, 64),
                                            (1, 2, 1, 64, 256), (1, 2, 1, 256, 64), (70, 4, 2, 64, 64)])
def test_delta_rule_of_one_token_from_its_projection(b, h, g, dim, vdim):
    """Three tokens one after the other (the carried convolution inputs move on once per token, whichever head comes last) as the
    separate ops on the CPU; the tickets are back at zero."""
    c = 2 * g * dim + h * vdim
    conv_w, tail, st = _rand(c, 4, std=0.6), _rand(b, c, 3), _rand(b, h, dim, vdim)
    a_log, dt, w = torch.rand(h) - 1.0, _rand(h), torch.rand(vdim) + 0.5
    s_dev, t_dev, tickets = st.to(DEV), tail.to(DEV), torch.zeros(b * g * 128, dtype=torch.int32, device=DEV)
    for _ in range(3):
        proj = _rand(b, c + h * vdim + 2 * h)
        got = hy.delta_step(proj.to(DEV), b, h, g, dim, vdim, conv_w.to(DEV), t_dev, a_log.to(DEV), dt.to(DEV), s_dev, w.to(DEV), 1e-5, tickets)
        q, k, v, beta, decay = hy.delta_prep(proj, b, 1, h, g, dim, vdim, conv_w, tail, a_log, dt)
        want = hy.delta_memory(q, k, v, beta, decay, st, b, 1, proj[:, c:c + h * vdim], w, 1e-5)
        assert got is not None
        _close(got, want, 2e-5, "output"), _close(s_dev, st, 2e-5, "state")
        assert torch.equal(t_dev.cpu(), tail) and not tickets.any()


@pytest.mark.parametrize("b,v", [(1, 1), (2, 63), (17, 5000), (1, 12288), (3, 32001), (64, 20000), (65, 13000), (256, 12289), (1, 128256)])
def test_greedy_choice_and_bookkeeping_in_one_launch(b, v):
    """Partials of logits with ties, infinities and rows of NaN, the choice over them and the loop's state, as the two launches."""
    from jax_llama_amd import ops
    logits = torch.randint(-3, 4, (b, v)).float()
    logits[0, v // 2:] = float("nan")
    if b > 2:
        logits[1], logits[2] = float("nan"), float("-inf")
        logits[2, v - 1] = float("inf")
    lg = logits.to(DEV)
    length, cl, eos, pad = 9, 6, 2, 77
    state = lambda: dict(finished=(torch.arange(b) % 5 == 3).int().to(DEV), sequences=torch.zeros(b, length, dtype=torch.int32, device=DEV),  # noqa: E731
                         cur_len=torch.tensor([cl], dtype=torch.int32, device=DEV), tokens=torch.zeros(b, 1, dtype=torch.int32, device=DEV),
                         positions=torch.arange(b, dtype=torch.int32, device=DEV), slot=torch.tensor([11], dtype=torch.int32, device=DEV))
    one, two = state(), state()
    ops.ext().decode_update(ops.argmax(lg)[0], *two.values(), pad, eos)
    part = ops.ArgmaxParts.of(lg).part
    for p in (part, torch.cat([part, torch.tensor([float("-inf"), 0.0], device=DEV).expand(b, 70, 2)], 1).contiguous()):  # (a wave, the workgroup)
        one = state()
        ops.ext().argmax_next(p, *one.values(), pad, eos)
        assert all(torch.equal(one[k], two[k]) for k in one)
    assert ops.ArgmaxParts.of(torch.zeros(257, 8, device=DEV)) is None


@pytest.mark.parametrize("m", [1, 2])
@pytest.mark.parametrize("d,v", [(256, 4096), (264, 4101), (2048, 32000), (4096, 5000)])
@pytest.mark.parametrize("pending,cap", [(True, 0.0), (False, 3.0), (True, 3.0)])
def test_greedy_choice_inside_the_output_product(m, d, v, pending, cap):
    """The same token, and the same residual stream, as the product written out and its argmax (a cap that ties many columns too)."""
    from jax_llama_amd import ops
    w, gain, x, y = _rand(v, d, dt=BF16).to(DEV), (torch.rand(d) + 0.5).to(DEV), _rand(m, d).to(DEV), _rand(2 * m, d).to(DEV)
    res = []
    for _ in range(2):
        r = hy.Residual(x.clone())
        if pending:
            r.add(y, gain, 1e-5, nsum=2, ysc=0.5)
        res.append(r)
    logits = hy.head_linear(res[0], gain, 1e-5, w, cap)
    got = hy.head_argmax(res[1], gain, 1e-5, w, cap)
    part = got.part.cpu()
    best = [max(((float(a), -int(i)) for a, i in zip(part[r, :, 0], part[r, :, 1].view(torch.int32)))) for r in range(m)]
    assert [-i for _, i in best] == ops.argmax(logits)[0].tolist()
    assert torch.equal(torch.tensor([a for a, _ in best]), logits.max(1).values.cpu()) and torch.equal(res[0].x, res[1].x)


@pytest.mark.parametrize("b", [32, 33])
def test_time_mix_of_many_rows_takes_its_decay_product_apart(b):
    """On either side of the pairs from which the decay product is a launch of its own."""
    test_time_mix_of_one_token_takes_its_decay_product(BF16, b, 64, 20, 12, 24)
