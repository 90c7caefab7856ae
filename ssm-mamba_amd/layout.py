"""Host side of the kernels between token-major activations (batch, seq_len,
channels), the layout of the reference's ``Block`` (``modules/block.py:78-90``),
and the channel-major layout the conv and scan kernels stream
(``ssm_rms_norm_tc_*``, ``ssm_transpose`` and ``ssm_batch_sum`` of
include/ssm_mamba.h).  No autograd here."""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _native as N
from .decode import plain_tensor

DTYPES = {torch.float32: N.SSM_F32, torch.bfloat16: N.SSM_BF16}
_MAX_CHANNELS = {torch.float32: 1024, torch.bfloat16: 2048}


def norm_tc_supported(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Whether ``norm_tc`` takes token-major x (batch, seq_len, channels)."""
    if not (x.is_cuda and x.dim() == 3 and x.dtype in DTYPES and x.numel() > 0):
        return False
    c = x.shape[2]
    return (weight.dtype == x.dtype and weight.device == x.device and weight.is_contiguous()
            and tuple(weight.shape) == (c,) and c * x.element_size() % 16 == 0
            and c <= _MAX_CHANNELS[x.dtype] and weight.data_ptr() % 16 == 0)


def aligned(x: torch.Tensor) -> torch.Tensor:
    """x contiguous at a 16-byte aligned address."""
    x = x.contiguous()
    return x if x.data_ptr() % 16 == 0 else x.clone()


def norm_tc(x: torch.Tensor, weight: torch.Tensor, eps: float, token_major: bool = False,
            copy: bool = False):
    """(h (batch, channels, seq_len), h token-major or None, 1 / rms (batch,
    seq_len) float32 or None, x as read) of RMSNorm(x) for token-major x;
    ``token_major`` asks for the two that a backward needs, ``copy`` for an x
    as read that is the caller's to write."""
    given, x = x, aligned(x)
    batch, seqlen, ch = x.shape
    h = torch.empty(batch, ch, seqlen, dtype=x.dtype, device=x.device)
    h_tm = torch.empty_like(x) if token_major else None
    rstd = torch.empty(batch, seqlen, dtype=torch.float32, device=x.device) if token_major else None
    x_copy = torch.empty_like(x) if copy and x is given else None
    with N.on(x.device):
        N.check(N.lib().ssm_rms_norm_tc_fwd(
            batch, seqlen, ch, DTYPES[x.dtype], x.data_ptr(), weight.data_ptr(), float(eps),
            h.data_ptr(), None if h_tm is None else h_tm.data_ptr(),
            None if rstd is None else rstd.data_ptr(), _ptr(x_copy), N.stream(x.device)))
    return h, h_tm, rstd, x if x_copy is None else x_copy


def norm_tc_backward(x: torch.Tensor, weight: torch.Tensor, rstd: torch.Tensor, dh: torch.Tensor,
                     dres: Optional[torch.Tensor]):
    """(dx, dweight) of ``norm_tc`` for dh (batch, channels, seq_len); dres, the
    gradient of a residual use of x, is added to dx."""
    batch, seqlen, ch = x.shape
    dh = dh.contiguous()
    dres = None if dres is None else aligned(dres)
    dx, dw = torch.empty_like(x), torch.empty_like(weight)
    lib = N.lib()
    ws = torch.empty(lib.ssm_rms_norm_tc_bwd_workspace_bytes(batch, seqlen, ch), dtype=torch.uint8,
                     device=x.device)
    with N.on(x.device):
        N.check(lib.ssm_rms_norm_tc_bwd(
            batch, seqlen, ch, DTYPES[x.dtype], x.data_ptr(), weight.data_ptr(), rstd.data_ptr(),
            dh.data_ptr(), None if dres is None else dres.data_ptr(), dx.data_ptr(), dw.data_ptr(),
            ws.data_ptr(), ws.numel(), N.stream(x.device)))
    return dx, dw


def transposed(x: torch.Tensor) -> torch.Tensor:
    """x.transpose(1, 2).contiguous() for x (batch, rows, cols) whose matrices
    are contiguous (a slice along dim 1 of a contiguous tensor is read in place
    through its batch stride)."""
    batch, rows, cols = x.shape
    if not (x.is_cuda and x.dtype in DTYPES and x.numel() > 0) or batch > 65535 \
            or rows > 65535 * 64:
        return x.transpose(1, 2).contiguous()
    if x.stride(2) != 1 or x.stride(1) != cols or (batch > 1 and x.stride(0) < rows * cols):
        x = x.contiguous()
    out = torch.empty(batch, cols, rows, dtype=x.dtype, device=x.device)
    with N.on(x.device):
        N.check(N.lib().ssm_transpose(batch, rows, cols, DTYPES[x.dtype], x.data_ptr(),
                                      0 if batch == 1 else x.stride(0), out.data_ptr(),
                                      N.stream(x.device)))
    return out


def batch_sum(x: torch.Tensor, transpose: bool = False,
              out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x.sum(0), or its transpose, for contiguous x (batch, rows, cols), its
    elements added in float32 and the sum rounded once; into ``out`` (contiguous) when given."""
    batch, rows, cols = x.shape
    x = x.contiguous()
    if out is None:
        out = torch.empty((cols, rows) if transpose else (rows, cols), dtype=x.dtype, device=x.device)
    with N.on(x.device):
        N.check(N.lib().ssm_batch_sum(batch, rows, cols, DTYPES[x.dtype], x.data_ptr(),
                                      int(transpose), out.data_ptr(), N.stream(x.device)))
    return out


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _one_type(log_A: torch.Tensor, *others: Optional[torch.Tensor]) -> bool:
    """Whether the stored parameters (dim, nstate), (dim,), (dim,) are what the
    scan_params kernels take."""
    return (log_A.is_cuda and log_A.dtype in DTYPES and log_A.dim() == 2 and log_A.numel() > 0
            and log_A.is_contiguous() and all(map(plain_tensor, (log_A, *others)))
            and all(t is None or (t.dtype == log_A.dtype and t.device == log_A.device
                                  and t.is_contiguous() and tuple(t.shape) == log_A.shape[:1])
                    for t in others))


def scan_params(log_A: torch.Tensor, D: Optional[torch.Tensor],
                bias: Optional[torch.Tensor]) -> Tuple[torch.Tensor, ...]:
    """(A = -exp(log_A), D, bias) contiguous in float32: float32 D and bias are
    the tensors given."""
    if not _one_type(log_A, D, bias):
        f32 = lambda t: None if t is None else t.float().contiguous()
        return -torch.exp(log_A.float().contiguous()), f32(D), f32(bias)
    dim, nstate = log_A.shape
    cast = log_A.dtype != torch.float32
    new = lambda t: torch.empty(t.shape, dtype=torch.float32, device=t.device)
    A = new(log_A)
    D32, b32 = ((None if t is None else new(t)) if cast else t for t in (D, bias))
    with N.on(log_A.device):
        N.check(N.lib().ssm_scan_params_fwd(
            dim, nstate, DTYPES[log_A.dtype], log_A.data_ptr(), _ptr(D) if cast else None,
            _ptr(bias) if cast else None, A.data_ptr(), _ptr(D32) if cast else None,
            _ptr(b32) if cast else None, N.stream(log_A.device)))
    return A, D32, b32


def scan_params_backward(A: torch.Tensor, stored, grads):
    """Gradients of the stored (log_A, D, bias) from those of ``scan_params``'s
    results (float32, or None where none is wanted), in the stored types."""
    dA, dD, db = grads
    log_A, D, bias = stored
    if not _one_type(log_A, D, bias):
        to = lambda g, t: None if g is None else g.to(t.dtype)
        return to(None if dA is None else dA * A, log_A), to(dD, D), to(db, bias)
    cast = log_A.dtype != torch.float32
    new = lambda g, t: None if g is None else torch.empty_like(t)
    out = (new(dA, log_A), *((new(dD, D), new(db, bias)) if cast else (dD, db)))
    if dA is not None or cast:
        dim, nstate = log_A.shape
        with N.on(A.device):
            N.check(N.lib().ssm_scan_params_bwd(
                dim, nstate, DTYPES[log_A.dtype], A.data_ptr(), _ptr(dA), _ptr(dD) if cast else None,
                _ptr(db) if cast else None, _ptr(out[0]), _ptr(out[1]) if cast else None,
                _ptr(out[2]) if cast else None, N.stream(A.device)))
    return out
