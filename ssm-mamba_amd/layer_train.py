"""The training forward and backward of one ``Block`` (``modules/block.py:78-90``
with ``modules/mamba.py:82-187``) as four autograd functions over the HIP
kernels: norm and in-projection, the conv (``CausalConv1dFn``), the x- and
step-size projections with the scan, and the out-projection with the residual.

Against one torch op per line, what each function's backward saves is passes
over memory: the norm's chain of float32 elementwise kernels, the transpositions
around the layer, the additions of gradients that meet (the residual's into the
norm's backward, the scan's du into the x-projection's product), the zero-filled
gradients of slices.  The weight gradients are batched products per batch row of
contiguous operands, each rounded to the layer's type as torch's are, and their
sum over the batch in float32, rounded again.  With one batch row there is nothing to sum, and plain products take the transposed
views: nine of a step's launches less (1 x 186 x 136, bf16: 842 us a step before,
822 now; 1 x 4096 x 1024: 844 and 819).

``supported`` says which layers and inputs take this path; every other one runs
op by op (``Block.forward_cm``).  When a backward is itself being differentiated
(create_graph), the functions of this module fall back to differentiating their
op-by-op form.  The scan and the conv in it are the operators' own functions,
whose gradients are native kernels: constants to a second differentiation, whose
terms through them are left out, as they are op by op.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import decode as _dec
from . import layout as _lay
from . import selective_scan
from .ops import selective_scan_fn
from .utils.tensor_utils import ensure_contiguous


def _bmm(w: torch.Tensor, x: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """w @ x per batch row, for one (m, k) weight (or its transposed view) and
    contiguous (batch, k, n) x; added to ``out`` in place when given."""
    w = w.expand(x.shape[0], *w.shape)
    return torch.bmm(w, x) if out is None else out.baddbmm_(w, x)


def _wgrad(g: torch.Tensor, x_tm: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Sum over the batch of g @ x_tm, for contiguous (batch, m, n) and (batch,
    n, k); one batch row is the product itself, with no sum to launch."""
    if g.shape[0] == 1:
        return torch.mm(g[0], x_tm[0]) if out is None else torch.mm(g[0], x_tm[0], out=out)
    return _lay.batch_sum(torch.bmm(g, x_tm), out=out)


def _product(w: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """w @ x of the op-by-op forms, in float32: autograd's derivative by w is a
    batched product whose right operand is a transposed view, and such products
    in bfloat16 (torch.bmm and baddbmm) have faulted the GPU.  Plain products
    (torch.mm) and transposed left operands have not."""
    return torch.bmm(w.float().expand(x.shape[0], *w.shape), x.float()).type_as(x)


def _grads_op_by_op(ctx, fn, inputs, grads):
    """Gradients of fn(*inputs) as differentiable torch ops (create_graph).  The
    function's every output takes a gradient when any of its inputs needs one;
    the op-by-op form's only where an input it comes from does."""
    res = [None] * len(ctx.needs_input_grad)
    with torch.enable_grad():
        outs = fn(*inputs)
        pairs = [(o, g) for o, g in zip(outs, grads) if g is not None and o.requires_grad]
        want = [i for i, t in enumerate(inputs)
                if isinstance(t, torch.Tensor) and t.requires_grad and ctx.needs_input_grad[i]]
        if not pairs or not want:
            return tuple(res)
        got = torch.autograd.grad([o for o, _ in pairs], [inputs[i] for i in want],
                                  [g for _, g in pairs], create_graph=True, allow_unused=True)
    for i, g in zip(want, got):
        res[i] = g
    return tuple(res)


class ProductFn(torch.autograd.Function):
    """w @ x (+ addend, of any shape that expands to the result) per batch row
    for a bfloat16 layer that runs op by op: torch's own product, whose
    derivative by w takes x transposed by a copy (see ``_product``).  The
    function and the copies cost a float32 layer with projection biases, where
    both forms can be timed, 3 to 10% (1 x 186 x 1024: 1311 -> 1358 us a step; 4 x
    2048 x 1024: 3508 -> 3632)."""

    @staticmethod
    def forward(ctx, w, x, addend):
        ctx.save_for_backward(w, x)
        if addend is None:
            return _bmm(w, x)
        ctx.addend_shape = addend.shape
        w = w.expand(x.shape[0], *w.shape)
        return torch.baddbmm(addend.expand(x.shape[0], w.shape[1], x.shape[2]), w, x)

    @staticmethod
    def _op_by_op(w, x):
        return (_product(w, x),)

    @staticmethod
    def backward(ctx, g):
        w, x = ctx.saved_tensors
        need_w, need_x, need_a = ctx.needs_input_grad
        da = g.sum_to_size(ctx.addend_shape) if need_a else None
        if torch.is_grad_enabled():
            return (*_grads_op_by_op(ctx, ProductFn._op_by_op, (w, x), (g,))[:2], da)
        g = g.contiguous()
        dw = None
        if need_w:
            dw = torch.mm(g[0], x[0].t()) if g.shape[0] == 1 \
                else torch.bmm(g, _lay.transposed(x)).sum(0)
        return dw, _bmm(w.t(), g) if need_x else None, da


class NormInProjFn(torch.autograd.Function):
    """(xs, z, x) of token-major x: the two halves of W_in @ rmsnorm(x),
    channel-major, and x itself (``copy``: a copy) for the residual, whose
    gradient then enters the norm's backward."""

    @staticmethod
    def forward(ctx, x, norm_weight, w_in, eps, copy):
        h, h_tm, rstd, xr = _lay.norm_tc(x, norm_weight, eps, copy=copy,
                                         token_major=any(ctx.needs_input_grad))
        inner = w_in.shape[0] // 2
        xs, z = _bmm(w_in[:inner], h), _bmm(w_in[inner:], h)
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(x, norm_weight, w_in, h_tm, rstd)
        ctx.eps = eps
        return xs, z, xr if copy else x.view_as(x)

    @staticmethod
    def _op_by_op(x, norm_weight, w_in, eps):
        xf = x.transpose(1, 2).float()
        h = (xf * torch.rsqrt(xf.pow(2).mean(1, keepdim=True) + eps)
             * (1.0 + norm_weight.float())[:, None]).type_as(x).contiguous()
        inner = w_in.shape[0] // 2
        return _product(w_in[:inner], h), _product(w_in[inner:], h), x.view_as(x)

    @staticmethod
    def backward(ctx, dxs, dz, dres):
        x, norm_weight, w_in, h_tm, rstd = ctx.saved_tensors
        if torch.is_grad_enabled():
            return _grads_op_by_op(ctx, NormInProjFn._op_by_op, (x, norm_weight, w_in, ctx.eps),
                                   (dxs, dz, dres))
        need_x, need_nw, need_w = ctx.needs_input_grad[:3]
        inner = w_in.shape[0] // 2
        halves = [(slice(0, inner), dxs), (slice(inner, 2 * inner), dz)]
        halves = [(s, g.contiguous()) for s, g in halves if g is not None]
        dw = None
        if need_w:
            dw = torch.empty(w_in.shape, dtype=w_in.dtype, device=w_in.device)
            if len(halves) < 2:
                dw.zero_()
            for s, g in halves:
                _wgrad(g, h_tm, out=dw[s])
        dx = dnw = None
        if need_x or need_nw:
            dh = None
            for s, g in halves:
                dh = _bmm(w_in[s].t(), g, dh)
            if dh is None:
                dx = dres
            else:
                xr = _lay.aligned(x)
                dx, dnw = _lay.norm_tc_backward(xr, norm_weight, rstd, dh, dres)
        return dx if need_x else None, dnw if need_nw else None, dw, None, None


class SsmFn(torch.autograd.Function):
    """(y, last state) from the conv output xc and the gate z, channel-major:
    params = W_x xc, delta = W_dt params[:R], and the gated scan with B and C
    read from params (``modules/mamba.py:141-182``)."""

    @staticmethod
    def forward(ctx, xc, z, w_x, w_dt, log_A, D, dt_bias, h_init, lengths, side):
        rank, nstate = w_dt.shape[1], log_A.shape[1]
        params = _bmm(w_x, xc)
        delta = _bmm(w_dt, params[:, :rank])
        A32, D32, b32 = _lay.scan_params(log_A, D, dt_bias)
        h0 = None if h_init is None else h_init.float().contiguous()
        lengths = ensure_contiguous(lengths)
        # (no gradient wanted, as in a frozen layer: no states and no ungated output)
        grad = any(ctx.needs_input_grad)
        y = torch.empty_like(xc) if grad else None
        out, h = selective_scan.forward(
            xc, A32, params[:, rank:rank + nstate], params[:, rank + nstate:], D32, delta, b32, h0,
            lengths, side, z=z, save_chunks=grad, out_ungated=y)
        if not grad:
            return out, h
        ctx.set_materialize_grads(False)
        ctx.save_for_backward(xc, z, w_x, w_dt, log_A, D, dt_bias, h_init, lengths, params, delta, y,
                              h, A32, D32, b32)
        ctx.side = side
        return out, selective_scan.last_state(h)

    @staticmethod
    def _op_by_op(xc, z, w_x, w_dt, log_A, D, dt_bias, h_init, lengths, side):
        rank, nstate = w_dt.shape[1], log_A.shape[1]
        A = -torch.exp(log_A.float())
        params = _product(w_x, xc)
        delta = _product(w_dt, params[:, :rank])
        return selective_scan_fn(xc, delta, A, params[:, rank:rank + nstate],
                                 params[:, rank + nstate:], D, z=z, delta_bias=dt_bias,
                                 return_last_state=True, h_init=h_init, length=lengths,
                                 padding_side=side)

    @staticmethod
    def backward(ctx, dout, dlast):
        (xc, z, w_x, w_dt, log_A, D, dt_bias, h_init, lengths, params, delta, y, h, A32, D32,
         b32) = ctx.saved_tensors
        if torch.is_grad_enabled():
            return _grads_op_by_op(ctx, SsmFn._op_by_op,
                                   (xc, z, w_x, w_dt, log_A, D, dt_bias, h_init, lengths, ctx.side),
                                   (dout, dlast))
        need = ctx.needs_input_grad
        rank, nstate = w_dt.shape[1], log_A.shape[1]
        f32 = lambda t: None if t is None else t.float().contiguous()
        if dout is None:
            dout = torch.zeros_like(xc)
        du, dA, dB, dC, dD, ddelta, dbias, dh0, dz = selective_scan.backward(
            xc, A32, params[:, rank:rank + nstate], params[:, rank + nstate:], D32, delta,
            b32, h, f32(h_init), dout.contiguous(), f32(dlast), lengths, ctx.side, z=z,
            out_ungated=y)
        dlog_A, dD, dbias = _lay.scan_params_backward(
            A32, (log_A, D, dt_bias), [g if n else None for g, n in zip((dA, dD, dbias), need[4:7])])
        dw_dt = dw_x = None
        one = xc.shape[0] == 1
        if need[3]:
            # (one batch row: a plain product, which takes the transposed views)
            dw_dt = torch.mm(ddelta[0], params[0, :rank].t()) if one \
                else _wgrad(ddelta, _lay.transposed(params[:, :rank]))
        if need[0] or need[2]:
            dparams = torch.cat([_bmm(w_dt.t(), ddelta), dB, dC], dim=1)
            if need[2]:
                dw_x = torch.mm(dparams[0], xc[0].t()) if one \
                    else _lay.batch_sum(torch.bmm(xc, _lay.transposed(dparams)), transpose=True)
            if need[0]:
                du = _bmm(w_x.t(), dparams, du)
        return (du if need[0] else None, dz, dw_x, dw_dt, dlog_A, dD, dbias, dh0, None,
                None)


class OutProjFn(torch.autograd.Function):
    """Token-major W_out @ y of channel-major y, added to ``residual`` in place
    when given."""

    @staticmethod
    def forward(ctx, y, w_out, residual):
        ctx.save_for_backward(y, w_out)
        if residual is not None:
            ctx.mark_dirty(residual)
        return out_proj(y, w_out, residual)

    @staticmethod
    def _op_by_op(y, w_out, residual):
        out = _product(w_out, y).transpose(1, 2)
        return (out if residual is None else residual + out,)

    @staticmethod
    def backward(ctx, dout):
        y, w_out = ctx.saved_tensors
        need = ctx.needs_input_grad
        if torch.is_grad_enabled():
            dy, dw, _ = _grads_op_by_op(ctx, OutProjFn._op_by_op, (y, w_out, None), (dout,))
            return dy, dw, dout if need[2] else None
        dout = dout.contiguous()
        if y.shape[0] == 1:  # plain products, which take the transposed views
            dt = dout[0].t()
            dy = torch.mm(w_out.t(), dt)[None] if need[0] else None
            return dy, torch.mm(dt, y[0].t()) if need[1] else None, dout if need[2] else None
        dy = _bmm(w_out.t(), _lay.transposed(dout)) if need[0] else None
        dw = _lay.batch_sum(torch.bmm(y, dout), transpose=True) if need[1] else None
        return dy, dw, dout if need[2] else None


def out_proj(y: torch.Tensor, w_out: torch.Tensor, residual: Optional[torch.Tensor]) -> torch.Tensor:
    """(batch, seq_len, out) = y^T W_out^T for channel-major y, in ``residual``
    itself plus its values when given (out of place the product's library call
    starts with a copy of it).  The batched product takes W_out^T as a
    contiguous copy; one batch row is a plain product and takes the views."""
    if y.shape[0] == 1:
        a, b = y[0].t(), w_out.t()
        if residual is None:
            return torch.mm(a, b)[None]
        residual[0].addmm_(a, b)
        return residual
    wt = _lay.transposed(w_out[None]).expand(y.shape[0], w_out.shape[1], w_out.shape[0])
    return torch.bmm(y.transpose(1, 2), wt) if residual is None \
        else residual.baddbmm_(y.transpose(1, 2), wt)


def supported(block, x: torch.Tensor) -> bool:
    """Whether token-major x through ``block`` takes the fused layer: float32 or
    bfloat16 on the GPU with every projection weight a plain tensor in x's
    dtype, no projection biases, a width the norm kernel takes, no autocast."""
    w = block.norm.weight
    if torch.is_autocast_enabled() or not _dec.plain_tensor(w) or not _lay.norm_tc_supported(x, w):
        return False
    # read where nn.Module keeps them: a weight that is not a plain parameter
    # (parametrized, computed by a hook) is not there and takes the other path
    mods, dtype, dev = block.ssm._modules, x.dtype, x.device
    for name in _PROJECTIONS:
        params = getattr(mods.get(name), "_parameters", {})
        p = params.get("weight")
        if p is None or p.dtype != dtype or p.device != dev or not _dec.plain_tensor(p):
            return False
        if name in _NO_BIAS and params.get("bias") is not None:
            return False
    return True


_PROJECTIONS = ("input_proj", "conv", "ssm_param_proj", "delta_proj", "out_proj")
_NO_BIAS = ("input_proj", "out_proj")
