"""Host logic of the fused training layer, on the CPU: the op-by-op gradients
that create_graph takes, and which layers the fused kernels may stand in for."""
from types import SimpleNamespace

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils._pytree import tree_map

from ssm_mamba_amd import layer_train as LT


def _op_by_op(fn, inputs, grads, needs=None):
    needs = needs or [isinstance(t, torch.Tensor) and t.requires_grad for t in inputs]
    return LT._grads_op_by_op(SimpleNamespace(needs_input_grad=needs), fn, inputs, grads)


@pytest.mark.parametrize("wants", [(True, True, True), (False, True, True), (False, False, True),
                                   (True, False, False), (False, True, False), (False, False, False)])
def test_norm_gradients_of_a_graph_with_parts_frozen(wants):
    """All three outputs of NormInProjFn carry a gradient, whichever of its
    inputs need one: the residual output of an input that needs none takes no
    part.  Values and second derivatives against autograd in float64 (the form's
    products are float32: 1e-5)."""
    g = torch.Generator().manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)
    x, nw, w = (t.requires_grad_(k) for t, k in zip((r(2, 5, 8), r(8), r(12, 8)), wants))
    dxs, dz, dres = r(2, 6, 5), r(2, 6, 5), r(2, 5, 8)
    got = _op_by_op(LT.NormInProjFn._op_by_op, (x, nw, w, 1e-6), (dxs, dz, dres))
    assert [t is not None for t in got[:3]] == list(wants)

    def ref():
        h = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * (1.0 + nw)
        p = h @ w.t()
        return (p * torch.cat([dxs, dz], 1).transpose(1, 2)).sum() + (x * dres).sum()

    live = [t for t, k in zip((x, nw, w), wants) if k]
    if not live:
        return
    want = torch.autograd.grad(ref(), live, create_graph=True)
    got = [t for t in got if t is not None]
    close = lambda a, b: bool((a.detach().double() - b.detach()).norm() <= 1e-5 * b.detach().norm())
    assert all(close(a, b) for a, b in zip(got, want))
    total = lambda gs: sum(t.double().pow(2).sum() for t in gs)
    if wants[0] or sum(wants) > 1:  # otherwise linear in what is left
        second = torch.autograd.grad(total(got), live)
        assert all(close(a, b) for a, b in zip(second, torch.autograd.grad(total(want), live)))


@pytest.mark.parametrize("strided", [lambda v: torch.stack([v, v], 1)[:, 0], lambda v: v[:1].expand(2)])
def test_lengths_reach_the_scan_contiguous(monkeypatch, strided):
    """The scan's kernels take a dense lengths vector; a layer takes a column of
    a tensor or one length expanded over the batch, forward and backward."""
    seen = []

    def forward(u, A, B, C, D, delta, bias, h0, length, side, **kw):
        seen.append(length)
        return torch.zeros_like(u), torch.zeros(2, 1, A.shape[1], A.shape[0])

    def backward(u, A, B, C, D, delta, bias, h, h0, dout, dlast, length, side, **kw):
        seen.append(length)
        return [torch.zeros_like(t) for t in (u, A, B, C, D, delta, bias)] + [None, torch.zeros_like(u)]

    monkeypatch.setattr(LT.selective_scan, "forward", forward)
    monkeypatch.setattr(LT.selective_scan, "backward", backward)
    monkeypatch.setattr(LT._lay, "batch_sum",
                        lambda x, transpose=False, out=None: x.sum(0).t() if transpose else x.sum(0))
    r = lambda *s: torch.randn(*s).requires_grad_(True)
    lengths = strided(torch.tensor([3, 5]))
    out, _ = LT.SsmFn.apply(r(2, 8, 5), r(2, 8, 5), r(6, 8), r(8, 2), r(8, 2), r(8), r(8), None,
                            lengths, "left")
    out.sum().backward()
    assert len(seen) == 2
    assert all(t.is_contiguous() and torch.equal(t, lengths) for t in seen)


class _Delegate(torch.nn.Module):
    """A wrapper that passes every attribute on, as torch.compile's does."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(super().__getattr__("inner"), name)


def _block(monkeypatch, **kw):
    """A layer that takes the fused kernels, as far as its tensors go."""
    from ssm_mamba_amd.causal_lm import Block
    monkeypatch.setattr(LT._lay, "norm_tc_supported", lambda x, w: True)
    return Block(model_dim=16, dropout_rate=0.0, **kw), torch.zeros(1, 4, 16)


@pytest.mark.parametrize("wrap", [_Delegate, torch.compile])
def test_wrapped_mixer(monkeypatch, wrap):
    blk, x = _block(monkeypatch)
    assert blk._fused(x)
    blk.ssm = wrap(blk.ssm)
    assert not blk._fused(x)


def test_methods_set_on_the_object(monkeypatch):
    for who in ("block", "mixer"):
        blk, x = _block(monkeypatch)
        obj = blk if who == "block" else blk.ssm
        obj.forward_cm = lambda *a, **k: None
        assert not blk._fused(x)


def test_missing_projection(monkeypatch):
    blk, x = _block(monkeypatch)
    blk.ssm.conv = None
    assert not blk._fused(x)
    del blk.ssm.conv
    assert not blk._fused(x)


class _ChannelMajorOnly(torch.nn.Module):
    def forward_cm(self, x, **kw):
        return x + 1.0, None


def test_model_asks_its_layers_for_forward_cm(monkeypatch):
    """A layer in CausalLM.layers needs forward_cm and no more, and a forward of
    a subclass or of the object is not what a model calls."""
    from ssm_mamba_amd.causal_lm import Block, CausalLM, CausalLMConfig
    monkeypatch.setattr(LT._lay, "norm_tc_supported", lambda x, w: True)
    called = []

    def forward_cm(self, x, **kw):
        called.append("forward_cm")
        return x, None

    def forward(self, *a, **kw):
        called.append("forward")

    class OwnForward(Block):
        pass

    OwnForward.forward = forward
    m = CausalLM(CausalLMConfig(vocab_size=11, model_dim=16, num_layers=2, dropout_rate=0.0))
    ids = torch.randint(3, 11, (2, 5))
    monkeypatch.setattr(Block, "forward", lambda self, x, **kw: (x, None))
    assert m(ids).shape == (2, 5, 11)        # (plain layers: Block.forward)
    monkeypatch.setattr(Block, "forward_cm", forward_cm)
    m.layers[1].__class__ = OwnForward
    m(ids)
    m.layers[1].__class__ = Block
    m.layers[1].forward = forward.__get__(m.layers[1])
    m(ids)
    assert called == ["forward_cm"] * 4
    m.layers = torch.nn.ModuleList([_ChannelMajorOnly()])
    assert m(ids).shape == (2, 5, 11)


def _global(register):
    return lambda m: getattr(torch.nn.modules.module, register)(lambda *a: None)


@pytest.mark.parametrize("change", [
    _global("register_module_forward_hook"), _global("register_module_forward_pre_hook"),
    _global("register_module_full_backward_hook"),
    lambda m: m.register_forward_hook(lambda *a: None),
    lambda m: m.register_forward_pre_hook(lambda *a: None),
    lambda m: m.register_full_backward_hook(lambda *a: None),
    lambda m: setattr(m, "forward", type(m).forward.__get__(m)),
    lambda m: setattr(m, "__class__", type("Own", (type(m),), {})),
])
def test_plain_module_calls(change):
    """A kernel may stand in for a module's call only where the call is its
    class's forward and nothing else."""
    from ssm_mamba_amd import decode as DEC
    from ssm_mamba_amd.causal_lm import RMSNorm
    for m in (RMSNorm(8), torch.nn.Linear(8, 8)):
        cls = type(m)
        assert DEC.plain(m, cls)
        handle = change(m)
        try:
            assert not DEC.plain(m, cls)
        finally:
            if handle is not None:
                handle.remove()
    assert DEC.plain(RMSNorm(8), RMSNorm)


class _NoTransposedRight(TorchDispatchMode):
    """Counts batched products and refuses a bfloat16 one whose right operand
    is a transposed view."""
    count = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        name = func.overloadpacket.__name__.rstrip("_")
        if name in ("bmm", "baddbmm"):
            right = args[1 if name == "bmm" else 2]
            self.count += 1
            bad = right.shape[2] > 1 and right.stride(2) != 1
            assert not (bad and right.dtype == torch.bfloat16), (name, right.shape, right.stride())
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("add", [None, "bias", "residual"])
def test_products_of_a_bf16_layer_op_by_op(batch, add):
    """Forward, backward and the backward of create_graph make no bfloat16
    batched product with a transposed right operand; values against float64,
    within one rounding of each batch row's product and of their sum."""
    from ssm_mamba_amd.causal_lm import _proj_cm
    g = torch.Generator().manual_seed(batch)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().requires_grad_(True)
    w, xs, dout = r(6, 8), r(batch, 12, 7), r(batch, 6, 7).detach()
    a = {None: None, "bias": r(6), "residual": r(batch, 6, 7)}[add]
    live = [t for t in (w, xs, a) if t is not None]
    kw = {} if a is None else {add: a}
    with _NoTransposedRight() as seen:
        for graph in (False, True):
            out = _proj_cm(w, xs[:, :8], **kw)
            got = torch.autograd.grad(out, live, dout, create_graph=graph)
            if graph:
                torch.autograd.grad(sum(t.float().pow(2).sum() for t in got), live, allow_unused=True)
    assert seen.count
    w64, x64, a64 = (None if t is None else t.detach().double().requires_grad_(True) for t in (w, xs, a))
    ref = w64 @ x64[:, :8]
    if a64 is not None:
        ref = ref + (a64[None, :, None] if add == "bias" else a64)
    want = torch.autograd.grad(ref, [t for t in (w64, x64, a64) if t is not None], dout.double())
    for p, q in ((out, ref), *zip(got, want)):
        assert float((p.double() - q).detach().norm()) <= 2.0 ** -7 * float(q.detach().norm())


class _Wrapped(torch.Tensor):
    """A weight that holds another tensor and no memory of its own, as a
    quantized or sharded one does."""

    @staticmethod
    def __new__(cls, held):
        return torch.Tensor._make_wrapper_subclass(cls, held.shape, dtype=held.dtype, device=held.device)

    def __init__(self, held):
        self.held = held

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        held = lambda t: t.held if isinstance(t, _Wrapped) else t
        if func is torch.ops.aten.detach.default:
            return _Wrapped(args[0].held)
        return func(*tree_map(held, args), **tree_map(held, kwargs or {}))


def _wrap_weight(module):
    module.weight = torch.nn.Parameter(_Wrapped(module.weight.detach()), requires_grad=False)


@pytest.mark.parametrize("part", ["norm", "ssm.out_proj", "ssm.ssm_param_proj", "ssm.conv"])
def test_weights_with_operators_of_their_own(monkeypatch, part):
    blk, x = _block(monkeypatch)
    assert blk._fused(x)
    _wrap_weight(blk.get_submodule(part))
    assert not blk._fused(x)
