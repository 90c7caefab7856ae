"""Conv1d rows that are not whole 16-byte pieces: lengths at the edges of a
lane's 8 positions, a wave's 512 and a workgroup's 2048, rows at every element
alignment, and rows beside non-finite ones."""
import pytest
import torch
import torch.nn.functional as F

from oracle import lm_ref as LR
from tests.helpers import assert_close
from tests.test_gpu_conv1d import _wgrad_magnitude

pytestmark = pytest.mark.gpu


def _offset(t, n):
    """The same values at an address n elements past an allocation's start."""
    flat = torch.empty(t.numel() + n, dtype=t.dtype, device=t.device)
    flat[n:] = t.reshape(-1)
    return flat[n:].view(t.shape)


def _passes(x, w, b, dy):
    from ssm_mamba_amd.causal_conv1d import causal_conv1d_fn
    x, w, b = (t.detach().requires_grad_(True) for t in (x, w, b))
    out = causal_conv1d_fn(x, w, b)
    return [out.detach(), *torch.autograd.grad(out, [x, w, b], dy)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("seqlen", [1, 7, 9, 12, 511, 513, 519, 1004, 2047, 2049, 2060, 4097])
def test_row_remainders(cuda, dtype, width, seqlen):
    g = torch.Generator().manual_seed(10 * seqlen + width)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype)
    x, w, b, dy = r(2, 3, seqlen), 0.5 * r(3, 1, width), 0.5 * r(3), r(2, 3, seqlen)
    print(f"case L={seqlen} width={width} {dtype}", flush=True)
    want = _passes(*(t.to(cuda) for t in (x, w, b, dy)))
    x64, w64, b64 = (t.double().requires_grad_(True) for t in (x, w, b))
    ref = F.silu(LR.causal_conv(x64, w64, b64))
    rx, rw, rb = torch.autograd.grad(ref, [x64, w64, b64], dy.double())
    assert_close(want[0], ref.detach(), dtype, "out")
    assert_close(want[1], rx, dtype, "dx")
    mw, mb = _wgrad_magnitude(x, w, b, dy, True)
    assert_close(want[2], rw, dtype, "dweight", mw)
    assert_close(want[3], rb, dtype, "dbias", mb)
    # the same bits at other row starts
    for off in (1, 2, 3):
        got = _passes(_offset(x.to(cuda), off), w.to(cuda), b.to(cuda), _offset(dy.to(cuda), off))
        assert all(torch.equal(p, q) for p, q in zip(want, got)), off


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqlen", [37, 2047, 2050])
def test_rows_beside_non_finite_ones(cuda, dtype, seqlen):
    g = torch.Generator().manual_seed(seqlen)
    r = lambda *s: torch.randn(*s, generator=g).to(dtype).to(cuda)
    x, w, b, dy = r(1, 9, seqlen), r(9, 1, 4), r(9), r(1, 9, seqlen)
    want = _passes(x, w, b, dy)
    x[:, 1::2], dy[:, 1::2] = float("nan"), float("inf")
    got = _passes(x, w, b, dy)
    assert torch.equal(got[0][:, ::2], want[0][:, ::2]) and torch.equal(got[1][:, ::2], want[1][:, ::2])
    assert torch.equal(got[2][::2], want[2][::2]) and torch.equal(got[3][::2], want[3][::2])
