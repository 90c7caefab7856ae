"""Scan rows that are not whole 16-byte pieces: every element alignment of the
row starts, lengths at the edges of the 4-step pieces and 16-step tiles, channel
counts that leave a wave's last rows empty, and rows beside non-finite ones."""
import pytest
import torch

from tests.helpers import make_case, to_dev
from tests.test_gpu_scan import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqlen", [1, 2, 3, 6, 15, 17, 18, 271, 533])
@pytest.mark.parametrize("dim", [1, 63, 81])
def test_row_remainders(cuda, dtype, seqlen, dim):
    run_case(cuda, 3, dim, seqlen, 16, dtype, seed=seqlen + dim, h_init=True, dlast=True,
             with_z=seqlen != 533, padding_side="left" if seqlen % 2 else "right",
             length=torch.tensor([seqlen, seqlen // 2, 0]) if seqlen > 6 else None)


def _offset(t, n):
    """The same values at an address n elements past an allocation's start."""
    flat = torch.empty(t.numel() + n, dtype=t.dtype, device=t.device)
    flat[n:] = t.reshape(-1)
    return flat[n:].view(t.shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqlen", [37, 530])
def test_start_and_neighbours(cuda, dtype, seqlen):
    """Start addresses one to three elements off and rows between non-finite
    ones: the finite rows' results are those of the case without either."""
    from ssm_mamba_amd import selective_scan as ss
    d = to_dev(make_case(2, 67, seqlen, 16, dtype, seed=3, with_z=True), cuda)
    dy = torch.randn(2, 67, seqlen, generator=torch.Generator().manual_seed(4)).to(dtype).to(cuda)
    bad = torch.zeros(2, 67, 1, dtype=torch.bool, device=cuda)
    bad[:, 1::2] = True

    def run(off, value):
        rows = [torch.where(bad, value, t) if value is not None else t
                for t in (d["u"], d["delta"], d["z"], dy)]
        u, delta, z, g = (_offset(t, off) for t in rows)
        y = _offset(torch.zeros_like(d["u"]), off)
        B, C = _offset(d["B"], off), _offset(d["C"], off)
        print(f"case L={seqlen} {dtype} offset={off} value={value}", flush=True)
        out, h = ss.forward(u, d["A"], B, C, d["D"], delta, d["delta_bias"], None, None, "right",
                            z=z, delta_softplus=True, out_ungated=y)
        res = ss.backward(u, d["A"], B, C, d["D"], delta, d["delta_bias"], h, None, g, None, None,
                          "right", z=z, delta_softplus=True, out_ungated=y)
        return [out, y, res[0], res[5], res[8]]

    want = run(0, None)
    keep = ~bad.expand_as(dy)
    for off, value in ((1, None), (2, None), (3, None), (1, float("inf")), (0, float("nan"))):
        for a, b in zip(want, run(off, value)):
            assert torch.isfinite(a).all()
            assert torch.equal(a[keep], b[keep])
