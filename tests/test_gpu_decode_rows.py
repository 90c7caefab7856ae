"""The decode step past the GEMV kernels' batches (9 to 64 rows, on the matrix
cores): the linear kernel against float64, and a layer's step against the
op-by-op path and the oracle's step chain."""
import pytest
import torch

from helpers import lm_state64
from oracle import lm_ref as LR

pytestmark = pytest.mark.gpu


# batch tiles of 16 and their edges; out_dim at the edges of the 16-row tiles
# and of the dispatch (16 waves up to 2048 rows, two tiles from 16384);
# in_dim below one K step, past a step's end, and one K group per wave
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("batch,out_dim,in_dim", [
    (9, 1, 8), (16, 37, 64), (17, 300, 1032), (32, 2049, 1024), (33, 2048, 2048), (64, 96, 4096),
    (31, 16400, 72),
])
def test_rows_linear(cuda, dtype, norm, batch, out_dim, in_dim):
    from ssm_mamba_amd import decode as DEC
    g = torch.Generator().manual_seed(out_dim + in_dim + batch)
    W = torch.randn(out_dim, in_dim, generator=g).to(dtype)
    x = torch.randn(batch, in_dim, generator=g).to(dtype)
    nw = (0.3 * torch.randn(in_dim, generator=g)).to(dtype) if norm else None
    b = torch.randn(out_dim, generator=g).to(dtype)
    res = torch.randn(batch, out_dim, generator=g).to(dtype)
    d = lambda t: None if t is None else t.to(cuda)
    with torch.no_grad():
        assert DEC.rows_supported(d(W), d(x), d(nw))
        assert not DEC.rows_supported(d(W), d(x)[:8], d(nw))
        got = DEC.rows_linear(d(W), d(x), d(nw), 1e-6, d(b), d(res)).double().cpu()
        again = DEC.rows_linear(d(W), d(x), d(nw), 1e-6, d(b), d(res)).double().cpu()
    v = x.double()
    if norm:
        v = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-6) * (1.0 + nw.double())
    ref = v @ W.double().t() + b.double() + res.double()
    size = v.abs() @ W.double().abs().t() + b.double().abs() + res.double().abs()
    # the result's rounding, the float32 sum of in_dim terms (64 units covers
    # the pairwise waves), and with the norm in bf16 one rounding of each
    # normalised activation
    u = 2.0 ** -24 if dtype == torch.float32 else 2.0 ** -8
    tol = u * ref.abs() + (64 * 2.0 ** -24 + (2.0 ** -8 if norm and dtype != torch.float32 else 0.0)) * size
    assert bool(((got - ref).abs() <= tol).all())
    assert torch.equal(got, again)


def make_model(seed, **kw):
    """A two-layer CausalLM with every norm weight and bias randomised."""
    from ssm_mamba_amd.causal_lm import CausalLM, CausalLMConfig
    torch.manual_seed(seed)
    m = CausalLM(CausalLMConfig(num_layers=2, dropout_rate=0.0, **kw)).float()
    with torch.no_grad():
        for name, p in m.named_parameters():
            if name.endswith("norm.weight") or (name.endswith(".bias") and "delta_proj" not in name):
                p.normal_(0.0, 0.3)
    return m.eval(), m.config


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch,model_dim,kw", [
    (9, 64, dict(bias=True, conv_bias=True)),
    (16, 72, dict(bias=False, conv_bias=False, conv_kernel=2)),   # rank 5: element-wise step sizes
    (33, 256, dict(bias=True, conv_bias=False, conv_kernel=7)),
    (64, 128, dict(bias=False, conv_bias=True, state_dim=8)),
])
def test_rows_block_step(cuda, dtype, batch, model_dim, kw):
    from ssm_mamba_amd import decode as DEC
    m, cfg = make_model(50 + batch, vocab_size=61, model_dim=model_dim, **kw)
    m = m.to(cuda, dtype)
    sd = lm_state64(m)
    g = torch.Generator().manual_seed(batch)
    ids = torch.randint(3, cfg.vocab_size, (batch, 7), generator=g)
    toks = torch.randint(3, cfg.vocab_size, (4, batch), generator=g)
    outs = {}
    for fused in (True, False):
        DEC.ENABLED = fused
        try:
            with torch.no_grad():
                m(ids.to(cuda), use_cache=True)
                x = torch.zeros(batch, model_dim, device=cuda, dtype=dtype)
                assert DEC.rows_step_supported(m.layers[0].ssm, x, m.layers[0].norm.weight) == fused
                outs[fused] = [m.step(t.to(cuda)).double().cpu() for t in toks]
                outs[(fused, "state")] = torch.stack([l.ssm._ssm_hiddens.double() for l in m.layers]).cpu()
                outs[(fused, "ctx")] = torch.stack([l.ssm._conv_context.double() for l in m.layers]).cpu()
        finally:
            DEC.ENABLED = True
    _, caches = LR.lm_forward(sd, ids, use_cache=True)
    refs = []
    for t in toks:
        ref, caches = LR.lm_step(sd, t, caches)
        refs.append(ref)
    # no further from float64 than the op-by-op step, within one rounding of
    # the largest value (the two round intermediate tensors at other places)
    u = 2.0 ** -20 if dtype == torch.float32 else 2.0 ** -8
    pairs = [(outs[True][i], outs[False][i], r) for i, r in enumerate(refs)]
    pairs += [(outs[(True, "state")], outs[(False, "state")], torch.stack([c[1] for c in caches])),
              (outs[(True, "ctx")], outs[(False, "ctx")], torch.stack([c[0] for c in caches]))]
    for new, old, ref in pairs:
        assert float((new - ref).abs().max()) <= float((old - ref).abs().max()) + u * float(ref.abs().max())
