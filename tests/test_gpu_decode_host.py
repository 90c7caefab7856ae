"""The native host side of a decode step (``_ext/decode_step``): the same
launches as the Python one for the batch sizes at the edges of each kernel's
range, and no answer of its own for layers that are not exactly the package's."""
from array import array

import pytest
import torch
import torch.nn.utils.parametrize as P
from torch import nn

pytestmark = pytest.mark.gpu


def _model(cuda, dtype, batch, model_dim=64, layers=2, **kw):
    from ssm_mamba_amd.causal_lm import CausalLM, CausalLMConfig
    torch.manual_seed(5)
    m = CausalLM(CausalLMConfig(vocab_size=32, model_dim=model_dim, num_layers=layers,
                                device="cuda", **kw)).to(cuda, dtype).eval()
    _caches(m, batch, dtype)
    return m


def _caches(m, batch, dtype):
    g = torch.Generator(device="cuda").manual_seed(6)
    for l in m.layers:
        s = l.ssm
        s._conv_context = torch.randn(batch, s.inner_dim, s.conv_kernel - 1, device="cuda",
                                      generator=g).to(dtype)
        s._ssm_hiddens = torch.randn(batch, s.inner_dim, s.state_dim, device="cuda", generator=g)


def _native(m, x):
    from ssm_mamba_amd import causal_lm as CL, decode as DEC
    return DEC.plain_block_step(m.layers[0], x, CL._LAYER_CLASSES)


def _run(m, x):
    out = m.layers[0].step(x)
    s = m.layers[0].ssm
    return out, s._conv_context.clone(), s._ssm_hiddens.clone()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch", [1, 4, 8, 9, 64, 65])
@pytest.mark.parametrize("kw", [dict(), dict(bias=True, conv_bias=True, state_dim=8, conv_kernel=3),
                                dict(model_dim=160, delta_rank=24, state_dim=64)])
def test_same_step(cuda, monkeypatch, dtype, batch, kw):
    from ssm_mamba_amd import decode as DEC
    m = _model(cuda, dtype, batch, **kw)
    x = torch.randn(batch, m.config.model_dim, device=cuda).to(dtype)
    with torch.no_grad():
        assert (_native(m, x) is not None) == (batch <= 64)
        for fold in (True, False):
            monkeypatch.setattr(DEC, "FOLD_XPROJ", fold)
            _caches(m, batch, dtype)
            got = _run(m, x)
            with monkeypatch.context() as mp:
                mp.setattr(DEC, "plain_block_step", lambda *a: None)
                _caches(m, batch, dtype)
                want = _run(m, x)
            for a, b in zip(got, want):
                assert torch.equal(a, b)


@pytest.mark.parametrize("batch", [1, 4, 5])
def test_layer_rows(cuda, batch):
    from ssm_mamba_amd import causal_lm as CL, decode as DEC
    m = _model(cuda, torch.bfloat16, batch, model_dim=128, layers=3)
    x = torch.zeros(batch, 128, device=cuda, dtype=torch.bfloat16)
    with torch.no_grad():
        rows = DEC.plain_layer_rows(m.layers, x, CL._LAYER_CLASSES)
        assert (rows is not None) == DEC.layers_supported(m.layers, x) == (batch <= 4)
        if rows is not None:
            assert rows == array("q", [0 if t is None else t.data_ptr() for l in m.layers
                                       for t in DEC._layer_tensors(l)]).tobytes()
            m.layers[2].norm.eps = 1e-5
            assert DEC.plain_layer_rows(m.layers, x, CL._LAYER_CLASSES) is None


class _Scaled(nn.Module):
    def forward(self, w):
        return w * 2


class _Sub(nn.Linear):
    @property
    def scale(self):
        return 1


def _subclass(m):
    m.layers[0].ssm.out_proj.__class__ = _Sub


def _parametrized(m):
    P.register_parametrization(m.layers[0].ssm.out_proj, "weight", _Scaled())


def _tensor_subclass(m):
    class T(torch.Tensor):
        pass
    m.layers[0].ssm._ssm_hiddens = m.layers[0].ssm._ssm_hiddens.as_subclass(T)


def _strided(m):
    w = m.layers[0].ssm.out_proj.weight
    w.data = w.data.t().contiguous().t()


def _mixed(m):
    m.layers[0].ssm.log_A.data = m.layers[0].ssm.log_A.data.double()


def _cache_shape(m):
    m.layers[0].ssm._ssm_hiddens = m.layers[0].ssm._ssm_hiddens[:, :, :8]


def _no_cache(m):
    m.layers[0].ssm._conv_context = None


@pytest.mark.parametrize("change", [_subclass, _parametrized, _tensor_subclass, _strided, _mixed,
                                    _cache_shape, _no_cache])
def test_left_to_the_general_checks(cuda, change):
    m = _model(cuda, torch.float32, 2)
    x = torch.randn(2, 64, device=cuda)
    with torch.no_grad():
        assert _native(m, x) is not None
        change(m)
        assert _native(m, x) is None
    m = _model(cuda, torch.float32, 2)
    assert _native(m, x) is None  # gradients wanted
    with torch.no_grad():
        assert _native(m, x.double()) is None and _native(m, x.cpu()) is None
        assert _native(m, x.t().contiguous().t()) is None


def test_hooked_norm_and_autocast(cuda):
    """Past 8 rows a hooked norm or autocast keeps the op-by-op step."""
    m = _model(cuda, torch.float32, 16)
    x = torch.randn(16, 64, device=cuda)
    with torch.no_grad():
        assert _native(m, x) is not None
        with torch.autocast("cuda", torch.bfloat16):
            assert _native(m, x) is None
        m.layers[0].norm.register_forward_hook(lambda *a: None)
        assert _native(m, x) is None
        assert _native(m, x[:2]) is None  # the caches hold 16 rows


def test_norm_with_a_forward_of_its_own(cuda):
    """Past 8 rows a forward set on the norm, or a hook on all modules, keeps
    being called by the layer's step and by the model's head."""
    seen = []

    def check(m, x, calls):
        with torch.no_grad():
            _caches(m, 16, torch.float32)
            want = [m.layers[0].step(x), m._head(x)]
            undo = calls()
            seen.clear()
            assert _native(m, x) is None
            _caches(m, 16, torch.float32)
            got = [m.layers[0].step(x), m._head(x)]
            undo()
        assert len(seen) >= 2
        assert all(float((a - b).norm() / b.norm()) <= 2.0 ** -18 for a, b in zip(got, want))

    m = _model(cuda, torch.float32, 16)
    x = torch.randn(16, 64, device=cuda)

    def on_the_object():
        norms = (m.layers[0].norm, m.norm)
        for n in norms:
            n.forward = lambda v, f=n.forward, **kw: (seen.append(n), f(v, **kw))[1]
        return lambda: [delattr(n, "forward") for n in norms]

    def on_all_modules():
        return nn.modules.module.register_module_forward_hook(lambda mod, *a: seen.append(mod)).remove

    check(m, x, on_the_object)
    check(m, x, on_all_modules)


def test_mixer_with_a_step_of_its_own(cuda):
    """Past 8 rows a layer's step calls the mixer's step where a subclass or the
    object has one."""
    from ssm_mamba_amd.causal_lm import Mamba

    class Own(Mamba):
        def step(self, x):
            return super().step(x) + 1.0

    m = _model(cuda, torch.float32, 16)
    x = torch.randn(16, 64, device=cuda)
    ssm = m.layers[0].ssm

    def run():
        _caches(m, 16, torch.float32)
        return m.layers[0].step(x)

    with torch.no_grad():
        want = run() + 1.0
        ssm.__class__ = Own
        got = [run()]
        ssm.__class__ = Mamba
        ssm.step = lambda v, f=ssm.step: f(v) + 1.0
        got.append(run())
        assert _native(m, x) is None
    for a in got:
        assert float((a - want).norm() / want.norm()) <= 2.0 ** -18


def test_weight_with_operators_of_its_own(cuda):
    """Past 8 rows a projection or head whose weight is a tensor subclass without
    memory of its own takes torch's operators."""
    from tests.test_layer_dispatch import _wrap_weight
    m = _model(cuda, torch.float32, 16, tie_embeddings=False)
    x = torch.randn(16, 64, device=cuda)
    with torch.no_grad():
        want = [m.layers[0].step(x), m._head(x), m.layers[0](x[:, None].expand(16, 40, 64))[0]]
        _caches(m, 16, torch.float32)
        _wrap_weight(m.lm_head)
        _wrap_weight(m.layers[0].ssm.out_proj)
        got = [m.layers[0].step(x), m._head(x), m.layers[0](x[:, None].expand(16, 40, 64))[0]]
    for a, b in zip(got, want):
        assert float((a - b).norm() / b.norm()) <= 2.0 ** -18
