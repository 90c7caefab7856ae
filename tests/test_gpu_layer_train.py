"""The fused layer of a training step and its kernels: the norm between the
layouts and its backward against float64, the transposition and the batch sum
bit for bit, and a layer's and a model's outputs and gradients against float64
and, over more forms of the call, against the op-by-op path."""
import copy

import pytest
import torch

from helpers import lm_state64
from oracle import lm_ref as LR

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


# one token; ragged tiles of 32 tokens, element-wise rows (odd lengths); channel
# counts of one chunk, past a 64-chunk group, and the largest of each tile size
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,seqlen,ch", [(1, 1, 8), (2, 33, 64), (3, 100, 1000), (2, 77, 512),
                                              (1, 64, 1024), (1, 50, 2048)])
def test_norm_between_layouts(cuda, dtype, batch, seqlen, ch):
    from ssm_mamba_amd import layout as LY
    ch = min(ch, 1024) if dtype == torch.float32 else ch
    g = torch.Generator().manual_seed(ch + seqlen)
    x = torch.randn(batch, seqlen, ch, generator=g).to(dtype)
    w = (0.3 * torch.randn(ch, generator=g)).to(dtype)
    dh = torch.randn(batch, ch, seqlen, generator=g).to(dtype)
    dres = torch.randn(batch, seqlen, ch, generator=g).to(dtype)
    d = lambda t: t.to(cuda)
    assert LY.norm_tc_supported(d(x), d(w))
    h, h_tm, rstd, xr = LY.norm_tc(d(x), d(w), 1e-6, token_major=True)
    assert torch.equal(LY.norm_tc(d(x), d(w), 1e-6)[0], h)
    assert torch.equal(h.transpose(1, 2), h_tm)
    dx, dw = LY.norm_tc_backward(xr, d(w), rstd, d(dh), d(dres))
    dx0, _ = LY.norm_tc_backward(xr, d(w), rstd, d(dh), None)
    again = LY.norm_tc_backward(xr, d(w), rstd, d(dh), d(dres))
    assert torch.equal(dx, again[0]) and torch.equal(dw, again[1])
    x64, w64 = x.double().requires_grad_(True), w.double().requires_grad_(True)
    r = x64 * torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-6) * (1.0 + w64)
    g64 = dh.double().transpose(1, 2)
    rx, rw = torch.autograd.grad(r, [x64, w64], g64)
    # one rounding of the result; in float32 the rsqrt and the sums on top
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -19
    assert bool(((h_tm.cpu().double() - r).abs() <= u * r.abs()).all())
    # sums of |terms|: g xh over the channels, dh xh over the tokens
    rs = torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-6)
    xh, gw = x.double() * rs, (g64 * (1.0 + w.double())).abs()
    size = rs * (gw + xh.abs() * (gw * xh.abs()).mean(-1, keepdim=True))
    for got, ref, sz in ((dx, rx + dres.double(), size + dres.double().abs()), (dx0, rx, size),
                         (dw, rw, (g64 * xh).abs().sum((0, 1)))):
        err = (got.cpu().double() - ref).abs()
        assert bool((err <= u * ref.abs() + 64 * 2.0 ** -24 * sz).all())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,rows,cols", [(1, 1, 1), (3, 65, 130), (2, 64, 72), (2, 96, 40),
                                              (5, 200, 64)])
def test_transpose_and_batch_sum(cuda, dtype, batch, rows, cols):
    from ssm_mamba_amd import layout as LY
    g = torch.Generator().manual_seed(rows * cols)
    x = torch.randn(batch, rows, cols, generator=g).to(dtype).to(cuda)
    assert torch.equal(LY.transposed(x), x.transpose(1, 2).contiguous())
    part = x[:, : rows // 2 + 1]  # read through its batch stride
    assert torch.equal(LY.transposed(part), part.transpose(1, 2).contiguous())
    ref = torch.zeros(rows, cols, device=cuda)
    for b in range(batch):
        ref = ref + x[b].float()
    ref = ref.to(dtype)
    assert torch.equal(LY.batch_sum(x), ref)
    assert torch.equal(LY.batch_sum(x, transpose=True), ref.t())


def _block(dtype, model_dim, conv_bias, seed, nstate=16):
    from ssm_mamba_amd.causal_lm import Block
    torch.manual_seed(seed)
    blk = Block(model_dim=model_dim, dropout_rate=0.0, conv_bias=conv_bias, state_dim=nstate)
    with torch.no_grad():
        blk.norm.weight.normal_(0.0, 0.3)
        blk.ssm.D.normal_(1.0, 0.1)
    return blk.cuda().to(dtype).train()


def _grads(blk, x, dout, dlast, h0, lengths, fused):
    from ssm_mamba_amd import layer_train as LT
    keep = LT.supported
    if not fused:
        LT.supported = lambda *a: False
    try:
        assert blk._fused(x) == fused
        out, last = blk(x, lengths=lengths, ssm_hiddens=h0)
        names, ps = zip(*blk.named_parameters())
        got = torch.autograd.grad([out, last], [x, h0, *ps], [dout, dlast])
    finally:
        LT.supported = keep
    return {"out": out.detach(), "last": last.detach(), **dict(zip(["x", "h0", *names], got))}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,seqlen,model_dim,conv_bias", [
    (2, 37, 64, False),    # odd length: element-wise rows in every kernel
    (1, 100, 72, True),    # one batch row: the plain out-projection product
    (3, 256, 256, False),
])
def test_block_gradients(cuda, dtype, batch, seqlen, model_dim, conv_bias):
    """Against the op-by-op path: the two round the same intermediate tensors
    to the layer's dtype, so they differ by float32 sums in other orders, in
    bf16 amplified to single roundings of those tensors."""
    blk = _block(dtype, model_dim, conv_bias, seed=seqlen)
    g = torch.Generator().manual_seed(model_dim)
    r = lambda *s: torch.randn(*s, generator=g).to(cuda)
    x = r(batch, seqlen, model_dim).to(dtype).requires_grad_(True)
    h0 = (0.1 * r(batch, 2 * model_dim, 16)).requires_grad_(True)
    lengths = torch.randint(1, seqlen + 1, (batch,), generator=g).to(cuda)
    dout, dlast = r(batch, seqlen, model_dim).to(dtype), r(batch, 2 * model_dim, 16)
    a = _grads(blk, x, dout, dlast, h0, lengths, True)
    b = _grads(blk, x, dout, dlast, h0, lengths, False)
    for k in a:
        assert a[k].dtype == b[k].dtype and a[k].shape == b[k].shape, k
        rel = float((a[k].double() - b[k].double()).norm() / b[k].double().norm())
        assert rel <= (2.0 ** -6 if dtype == torch.bfloat16 else 2.0 ** -18), (k, rel)


@pytest.mark.parametrize("dtype", DTYPES)
def test_block_gradients_of_a_graph(cuda, dtype):
    """With create_graph the gradients come from the op-by-op forms: the same
    values, up to roundings of the layer's intermediate tensors."""
    blk = _block(dtype, 64, False, seed=7)
    g = torch.Generator().manual_seed(8)
    x = torch.randn(2, 40, 64, generator=g).to(dtype).to(cuda).requires_grad_(True)
    dout = torch.randn(2, 40, 64, generator=g).to(dtype).to(cuda)
    ps = [x, *blk.parameters()]
    for a, b in zip(torch.autograd.grad(blk(x)[0], ps, dout, create_graph=True),
                    torch.autograd.grad(blk(x)[0], ps, dout)):
        assert a.dtype == b.dtype
        a = a.detach()
        rel = float((a.double() - b.double()).norm() / b.double().norm())
        assert rel <= (2.0 ** -6 if dtype == torch.bfloat16 else 2.0 ** -18), rel


def test_block_second_derivatives_and_frozen_parameters(cuda):
    """create_graph differentiates the op-by-op form: the second derivatives of
    the op-by-op layer, whose terms through the scan's and the conv's own
    gradients are left out on both paths (float64 checks of the norm's and the
    products' second derivatives: tests/test_layer_dispatch.py).  Parameters and
    inputs that need no gradient get none."""
    from ssm_mamba_amd import layer_train as LT
    blk = _block(torch.float32, 64, False, seed=3)
    x0 = torch.randn(2, 40, 64, generator=torch.Generator().manual_seed(4)).to(cuda)

    def penalty(fused):
        keep = LT.supported
        if not fused:
            LT.supported = lambda *a: False
        try:
            x = x0.clone().requires_grad_(True)
            out, _ = blk(x)
            gx, = torch.autograd.grad(out.pow(2).sum(), x, create_graph=True)
            return torch.autograd.grad(gx.pow(2).sum(), [x, blk.norm.weight, blk.ssm.out_proj.weight,
                                                         blk.ssm.input_proj.weight])
        finally:
            LT.supported = keep

    for u, v in zip(penalty(True), penalty(False)):
        assert float((u - v).norm() / v.norm()) <= 1e-5
    blk.ssm.input_proj.weight.requires_grad_(False)
    blk.norm.weight.requires_grad_(False)
    blk(x0)[0].sum().backward()
    assert blk.ssm.input_proj.weight.grad is None and blk.norm.weight.grad is None
    assert all(p.grad is not None for n, p in blk.named_parameters() if p.requires_grad)


# fewer and more elements than a workgroup, one state, no D, mixed stored types
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dim,nstate,with_d,mixed", [(1, 1, True, False), (300, 1, True, False),
                                                      (70, 16, False, False), (257, 64, True, True)])
def test_scan_params(cuda, dtype, dim, nstate, with_d, mixed):
    from ssm_mamba_amd import layout as LY
    g = torch.Generator().manual_seed(dim)
    log_A = torch.randn(dim, nstate, generator=g).to(dtype).to(cuda)
    D = torch.randn(dim, generator=g).to(dtype).to(cuda) if with_d else None
    bias = torch.randn(dim, generator=g).to(torch.float32 if mixed else dtype).to(cuda)
    A, D32, b32 = LY.scan_params(log_A, D, bias)
    ref = -torch.exp(log_A.double())
    assert A.dtype == torch.float32
    assert bool(((A.double() - ref).abs() <= 2.0 ** -22 * ref.abs()).all())
    assert (D32 is None) == (D is None) and (D is None or torch.equal(D32, D.float()))
    assert torch.equal(b32, bias.float())
    grads = [torch.randn(t.shape, generator=g).to(cuda) if t is not None else None for t in (A, D32, b32)]
    for want in ((1, 1, 1), (0, 1, 0), (1, 0, 0)):
        use = [x if w else None for x, w in zip(grads, want)]
        got = LY.scan_params_backward(A, (log_A, D, bias), use)
        exp = [None if use[0] is None else use[0] * A, use[1], use[2]]
        for o, e, t in zip(got, exp, (log_A, D, bias)):
            assert (o is None) == (e is None)
            assert o is None or (o.dtype == t.dtype and torch.equal(o, e.to(t.dtype)))


def test_norm_hooks_and_overridden_layers_keep_being_called(cuda):
    """A layer whose norm has hooks, or whose class has a forward of its own,
    does not take the fused kernels."""
    from ssm_mamba_amd.causal_lm import Block, Mamba
    x = torch.randn(1, 40, 64, generator=torch.Generator().manual_seed(5)).to(cuda)
    blk = _block(torch.float32, 64, False, seed=6)
    assert blk._fused(x)
    seen = []
    handle = blk.norm.register_full_backward_hook(lambda *a: seen.append("norm"))
    blk(x.clone().requires_grad_(True))[0].sum().backward()
    handle.remove()
    assert seen == ["norm"] and blk._fused(x)

    class OwnMixer(Mamba):
        def forward_cm(self, *a, **k):
            seen.append("mixer")
            return super().forward_cm(*a, **k)

    class OwnBlock(Block):
        def forward_cm(self, *a, **k):
            seen.append("block")
            return super().forward_cm(*a, **k)

    blk.ssm.__class__ = OwnMixer
    blk(x)
    blk.ssm.__class__, blk.__class__ = Mamba, OwnBlock
    blk(x)
    assert seen == ["norm", "mixer", "block"]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,seqlen,ch", [(1, 33, 64), (2, 37, 1000)])
def test_residual_copy(cuda, dtype, batch, seqlen, ch):
    """The norm's copy of x, which the layer's output is summed into: x's bits
    in memory of its own, so a layer's input keeps its values."""
    from ssm_mamba_amd import layout as LY
    x = torch.randn(batch, seqlen, ch, generator=torch.Generator().manual_seed(ch)).to(dtype).to(cuda)
    w = torch.zeros(ch, dtype=dtype, device=cuda)
    h, _, _, xc = LY.norm_tc(x, w, 1e-6, copy=True)
    assert torch.equal(xc, x) and xc.data_ptr() != x.data_ptr()
    assert torch.equal(h, LY.norm_tc(x, w, 1e-6)[0])
    strided = x.transpose(0, 1).contiguous().transpose(0, 1)  # read through a copy already
    xc = LY.norm_tc(strided, w, 1e-6, copy=True)[3]
    assert torch.equal(xc, x) and xc.data_ptr() != strided.data_ptr()
    if ch != 64:
        return
    blk, keep = _block(dtype, ch, False, seed=9), x.clone()
    with torch.no_grad():
        out = blk(x)[0]
    again = blk(x)[0]
    assert torch.equal(x, keep) and torch.equal(blk(x.requires_grad_(True))[0], again)
    assert float((out - again.detach()).norm() / out.norm()) <= 2.0 ** -7


@pytest.mark.parametrize("frozen", [("norm", "ssm"), ("norm.weight", "ssm.input_proj.weight"),
                                    ("ssm.input_proj.weight", "ssm.log_A", "ssm.out_proj.weight"), ()])
def test_block_gradients_of_a_graph_on_data(cuda, frozen):
    """create_graph for a layer whose input needs no gradient (the first layer,
    a frozen embedding) and for subsets of frozen parameters."""
    blk = _block(torch.float32, 64, False, seed=11)
    for n, p in blk.named_parameters():
        p.requires_grad_(not n.startswith(frozen) if frozen else True)
    ps = [p for p in blk.parameters() if p.requires_grad]
    g = torch.Generator().manual_seed(12)
    x = torch.randn(2, 40, 64, generator=g).to(cuda)
    dout, dlast = (torch.randn(s, generator=g).to(cuda) for s in ((2, 40, 64), (2, 128, 16)))
    if not ps:
        x.requires_grad_(True)
        ps = [x]
    for a, b in zip(*(torch.autograd.grad(blk(x), ps, [dout, dlast], create_graph=c) for c in (True, False))):
        assert float((a.detach() - b).norm() / b.norm()) <= 2.0 ** -18


@pytest.mark.parametrize("strided", [lambda v: torch.stack([v, v], 1)[:, 0], lambda v: v[:1].expand(2)])
def test_block_with_strided_lengths(cuda, strided):
    """Lengths as a column of a tensor, or one expanded over the batch."""
    blk = _block(torch.float32, 64, False, seed=13)
    x = torch.randn(2, 40, 64, generator=torch.Generator().manual_seed(14)).to(cuda)
    lengths = strided(torch.tensor([31, 40], device=cuda))
    got, want = (blk(x, lengths=v, use_cache=True) for v in (lengths, lengths.contiguous()))
    assert not lengths.is_contiguous() and all(torch.equal(a, b) for a, b in zip(got, want))
    ps = list(blk.parameters())
    for a, b in zip(*(torch.autograd.grad(list(o), ps, [torch.ones_like(t) for t in o]) for o in (got, want))):
        assert torch.equal(a, b)


def test_wrapped_mixer_is_called(cuda):
    """A mixer behind a wrapper that passes its attributes on runs op by op,
    with and without autograd and in the decode step."""
    from tests.test_layer_dispatch import _Delegate
    blk = _block(torch.float32, 64, False, seed=15)
    x = torch.randn(12, 40, 64, generator=torch.Generator().manual_seed(16)).to(cuda)
    want = blk(x)[0].detach()
    blk.ssm = _Delegate(blk.ssm)
    assert float((blk(x)[0].detach() - want).norm() / want.norm()) <= 2.0 ** -18
    with torch.no_grad():
        got = blk(x, use_cache=True)[0]
        step = blk.step(x[:, -1].contiguous())
    assert float((got - want).norm() / want.norm()) <= 2.0 ** -18 and step.shape == (12, 64)


def test_frozen_layer_saves_nothing(cuda):
    """With gradients enabled and none wanted, a layer's scan saves no states
    (seqlen / 16 of them) and the results are the same."""
    blk = _block(torch.float32, 64, False, seed=17)
    x = torch.randn(2, 4096, 64, generator=torch.Generator().manual_seed(18)).to(cuda)
    peak = []
    for wanted in (True, False):
        blk.requires_grad_(wanted)
        out = [t.detach().clone() for t in blk(x, use_cache=True)]
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        res = blk(x)
        peak.append((out, torch.cuda.max_memory_allocated() - base))
        assert res[0].requires_grad == wanted
        del res
    (a, most), (b, least) = peak
    assert all(float((u - v).norm() / v.norm()) <= 2.0 ** -20 for u, v in zip(a, b))
    # the states, the ungated output and the token-major norm
    assert most - least >= 2 * 256 * 16 * 128 * 4 // 2


@pytest.mark.parametrize("autocast", [False, True])
@pytest.mark.parametrize("batch", [1, 2])
def test_bf16_layer_op_by_op_makes_no_transposed_products(cuda, batch, autocast):
    """A layer with projection biases, or under autocast, trains op by op: no
    bfloat16 batched product with a transposed right operand either way, and
    gradients against the float32 layer's (which float64 checks elsewhere)."""
    from ssm_mamba_amd.causal_lm import Block
    from tests.test_layer_dispatch import _NoTransposedRight
    torch.manual_seed(19)
    blk = Block(model_dim=64, dropout_rate=0.0, bias=True).cuda()
    x = torch.randn(batch, 40, 64, device=cuda)
    low = blk if autocast else copy.deepcopy(blk).bfloat16()
    xl = x if autocast else x.bfloat16()
    assert not low._fused(xl)
    with _NoTransposedRight() as seen:
        with torch.autocast("cuda", torch.bfloat16, enabled=autocast):
            out = low(xl)[0]
        got = torch.autograd.grad(out.float().pow(2).sum(), list(low.parameters()))
    assert seen.count
    want = torch.autograd.grad(blk(x)[0].pow(2).sum(), list(blk.parameters()))
    for (n, p), a, b in zip(low.named_parameters(), got, want):
        assert a.dtype == p.dtype
        # a chain of a dozen bfloat16 roundings, each of 2^-9 relative
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 2.0 ** -5, n


def _ref64(p, x, nstate, h0, lengths, use_cache, scale):
    """The layer in float64: (out, last state, conv window)."""
    y, last, ctx = LR.mamba_forward(p, LR.rms_norm(x, p["norm.weight"]), nstate,
                                    p["ssm.delta_proj.weight"].shape[1], h0=h0, lengths=lengths,
                                    use_cache=use_cache)
    return x + (y if scale is None else y * scale), last, ctx


def _with_mask(blk, scale, dev):
    """Dropout with a given mask in place of a drawn one."""
    if scale is not None:
        blk.dropout.p = 0.25
        blk.dropout.forward = lambda v, s=scale.to(dev): v * s.to(v.dtype)


def _mask(shape, g):
    return (torch.rand(shape, generator=g) >= 0.25).double() / 0.75


# one and several batch rows, odd and whole rows; 8 to 64 states; without a first
# state the last state's gradient still counts; the caches of a prefill; dropout
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batch,seqlen,model_dim,nstate,h0,pads,use_cache,drop", [
    (2, 37, 64, 16, False, True, True, False),
    (1, 100, 72, 32, True, False, False, True),
    (3, 64, 40, 64, False, False, True, True),
    (2, 130, 64, 8, True, True, False, True),
])
def test_layer_against_float64(cuda, dtype, batch, seqlen, model_dim, nstate, h0, pads, use_cache, drop):
    """Outputs, caches and every gradient of the fused layer.  float32: norm-wise
    2^-16, the float32 sums over up to 128 channels and 130 steps and their
    exponentials.  bfloat16: no further from float64 than the op-by-op layer by
    more than half (they round as many tensors, at other places) and one
    rounding."""
    blk = _block(dtype, model_dim, True, seed=nstate, nstate=nstate)
    g = torch.Generator().manual_seed(seqlen)
    r = lambda *s: torch.randn(*s, generator=g)
    x, dout, dlast = r(batch, seqlen, model_dim).to(dtype), r(batch, seqlen, model_dim).to(dtype), \
        r(batch, 2 * model_dim, nstate)
    first = 0.1 * r(batch, 2 * model_dim, nstate) if h0 else None
    lengths = torch.randint(5, seqlen + 1, (batch,), generator=g) if pads else None
    scale = _mask((batch, seqlen, model_dim), g) if drop else None
    _with_mask(blk, scale, cuda)
    names = ["x"] + (["h0"] if h0 else []) + [n for n, _ in blk.named_parameters()]

    def run(fused):
        from ssm_mamba_amd import layer_train as LT
        keep = LT.supported
        s = blk.dropout.forward if drop else None
        if not fused:
            LT.supported = lambda *a: False
            if drop:  # the op-by-op layer drops channel-major
                blk.dropout.forward = lambda v: s(v.transpose(1, 2)).transpose(1, 2)
        try:
            leaves = [t.detach().to(cuda).requires_grad_(True) for t in (x, first) if t is not None]
            xg, hg = leaves[0], leaves[1] if h0 else None
            assert blk._fused(xg) == fused
            out, last = blk(xg, lengths=None if lengths is None else lengths.to(cuda),
                            ssm_hiddens=hg, use_cache=use_cache)
            grads = torch.autograd.grad([out, last], [*leaves, *blk.parameters()],
                                        [dout.to(cuda), dlast.to(cuda)])
        finally:
            LT.supported = keep
            if drop:
                blk.dropout.forward = s
        res = dict(zip(names, grads), out=out, last=last)
        if use_cache:
            res["window"] = blk.ssm._conv_context
            assert torch.equal(blk.ssm._ssm_hiddens, last)
        return res

    p = {n: t.detach().double().cpu().requires_grad_(True) for n, t in blk.named_parameters()}
    x64 = x.double().requires_grad_(True)
    f64 = first.double().requires_grad_(True) if h0 else None
    out, last, ctx = _ref64(p, x64, nstate, f64, lengths, use_cache, scale)
    grads = torch.autograd.grad([out, last], [t for t in (x64, f64) if t is not None] + list(p.values()),
                                [dout.double(), dlast.double()])
    want = dict(zip(names, grads), out=out.detach(), last=last.detach())
    if use_cache:
        want["window"] = ctx.detach()
    err = lambda got: {k: float((got[k].detach().double().cpu() - w).norm() / w.norm())
                       for k, w in want.items()}
    got = err(run(True))
    if dtype == torch.float32:
        assert max(got.values()) <= 2.0 ** -16, got
    else:
        ops = err(run(False))
        for k in got:
            assert got[k] <= 1.5 * ops[k] + 2.0 ** -9, (k, got[k], ops[k])


@pytest.mark.parametrize("pads", [False, True])
def test_model_training_step_against_float64(cuda, pads):
    """CausalLM.forward with gradients in its default form (no projection
    biases, dropout on): logits and every parameter's gradient."""
    from ssm_mamba_amd.causal_lm import CausalLM, CausalLMConfig
    torch.manual_seed(21)
    m = CausalLM(CausalLMConfig(vocab_size=31, model_dim=64, num_layers=3)).cuda().train()
    with torch.no_grad():
        for n, t in m.named_parameters():
            if n.endswith("norm.weight"):
                t.normal_(0.0, 0.3)
    g = torch.Generator().manual_seed(22)
    ids = torch.randint(3, 31, (2, 45), generator=g)
    lengths = torch.tensor([45, 30]) if pads else None
    r = torch.randn(2, 45, 31, generator=g)
    masks = [_mask((2, 45, 64), g) for _ in m.layers]
    for layer, s in zip(m.layers, masks):
        _with_mask(layer, s, cuda)
        assert layer._fused(m.embedding(ids.to(cuda)))
    sd = lm_state64(m)
    for v in sd.values():
        v.requires_grad_(True)
    x = sd["embedding.weight"][ids]
    for i, s in enumerate(masks):
        p = LR.layer_params(sd, i)
        x = _ref64(p, x, 16, None, lengths, False, s)[0]
    want = LR.rms_norm(x, sd["norm.weight"]) @ sd["lm_head.weight"].t()
    names = [n for n, _ in m.named_parameters()]
    grads = torch.autograd.grad(want, [sd[n] for n in names], r.double())
    got = m(ids.to(cuda), None if lengths is None else lengths.to(cuda))
    mine = torch.autograd.grad(got, list(m.parameters()), r.to(cuda))
    for n, a, b in zip(["logits", *names], [got, *mine], [want, *grads]):
        rel = float((a.detach().double().cpu() - b.detach()).norm() / b.detach().norm())
        assert rel <= 2.0 ** -16, (n, rel)
