"""The role-split scan kernels past 16 states: state counts at the edges of their
32- and 64-state forms and of a wave's state pairs, in one segment and split
into several with summary parts, aligned and not."""
import pytest
import torch

from tests.test_gpu_scan import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nstate", [17, 31, 33, 48, 63, 64])
@pytest.mark.parametrize("batch,dim,seqlen,side,length", [
    (2, 70, 33, "right", None),          # three tiles, one segment, element-wise rows
    (1, 130, 528, "left", [401]),        # split, padded inside a segment
    (3, 64, 777, "right", [777, 0, 130]),  # ragged last segment
])
def test_state_counts(cuda, dtype, nstate, batch, dim, seqlen, side, length):
    run_case(cuda, batch, dim, seqlen, nstate, dtype, seed=nstate + seqlen, h_init=seqlen != 33,
             dlast=True, with_z=nstate % 2 == 1, padding_side=side,
             length=None if length is None else torch.tensor(length))


def _inputs(cuda, batch, dim, seqlen, nstate):
    g = torch.Generator(device=cuda).manual_seed(nstate)
    r = lambda *s: torch.randn(s, generator=g, device=cuda)
    A = -torch.arange(1, nstate + 1, device=cuda).float().repeat(dim, 1)
    return dict(u=r(batch, dim, seqlen), delta=r(batch, dim, seqlen), z=r(batch, dim, seqlen), A=A,
                B=r(batch, nstate, seqlen), C=r(batch, nstate, seqlen), D=r(dim), bias=r(dim) - 4.0,
                h0=0.1 * r(batch, dim, nstate))


def _near(a, b, bits, name):
    rel = float((a.double() - b.double()).norm() / b.double().norm())
    assert rel <= 2.0 ** -bits, (name, rel)


# one row of B past 2 GiB (64 states), and 16 rows of the output past 2 GiB (3):
# the role-split kernels' 32-bit ranges end there
@pytest.mark.parametrize("nstate,seqlen,dim", [(64, (1 << 23) + 24, 3), (3, (1 << 25) + 20, 2)])
def test_general_forward_with_few_states(cuda, nstate, seqlen, dim):
    """The general forward and its summaries, which serve what the role-split
    kernels' ranges do not reach, against two role-split calls over the halves
    of the sequence, the second from the first's last state."""
    from ssm_mamba_amd import selective_scan as ss
    c = _inputs(cuda, 1, dim, seqlen, nstate)

    def run(s, h0):
        cut = {k: c[k][:, :, s].contiguous() for k in ("u", "delta", "B", "C", "z")}
        y = torch.empty_like(cut["u"])
        out, h = ss.forward(cut["u"], c["A"], cut["B"], cut["C"], c["D"], cut["delta"], c["bias"], h0,
                            z=cut["z"], out_ungated=y)
        last = ss.forward(cut["u"], c["A"], cut["B"], cut["C"], c["D"], cut["delta"], c["bias"], h0,
                          z=cut["z"], save_chunks=False)[1]
        return out, y, h, last

    print(f"general forward {nstate} states, {dim} x {seqlen}", flush=True)
    out, y, h, last = run(slice(0, seqlen), c["h0"])
    half = 1 << (seqlen.bit_length() - 2)
    a = run(slice(0, half), c["h0"])
    b = run(slice(half, seqlen), a[3])
    # one float32 update after another, the error of a step decaying with it
    for name, got, want in (("out", out, torch.cat([a[0], b[0]], 2)), ("y", y, torch.cat([a[1], b[1]], 2)),
                            ("h", h, torch.cat([a[2], b[2]], 1)), ("last", last, b[3])):
        _near(got, want, 18, name)


# the dB / dC partials of all batch rows past 2 GiB, one row's not; every form by
# state count, whole and ragged rows
@pytest.mark.parametrize("nstate,batch,seqlen", [(64, 4, (1 << 20) + 8), (20, 13, (1 << 20) + 3),
                                                 (5, 52, (1 << 20) + 8)])
def test_general_backward_with_few_states(cuda, nstate, batch, seqlen):
    """The general backward and its summaries against role-split calls of one
    batch row each."""
    from ssm_mamba_amd import selective_scan as ss
    dim = 3
    c = _inputs(cuda, batch, dim, seqlen, nstate)
    g = torch.Generator(device=cuda).manual_seed(1)
    dout = torch.randn(batch, dim, seqlen, generator=g, device=cuda)
    dlast = torch.randn(batch, dim, nstate, generator=g, device=cuda)
    length = torch.randint(1, seqlen + 1, (batch,), generator=g, device=cuda)
    y = torch.empty_like(dout)
    _, h = ss.forward(c["u"], c["A"], c["B"], c["C"], c["D"], c["delta"], c["bias"], c["h0"], length,
                      "left", z=c["z"], out_ungated=y)

    def run(s):
        return ss.backward(c["u"][s], c["A"], c["B"][s], c["C"][s], c["D"], c["delta"][s], c["bias"], h[s],
                           c["h0"][s], dout[s], dlast[s], length[s], "left", z=c["z"][s], out_ungated=y[s])

    print(f"general backward {nstate} states, {batch} x {dim} x {seqlen}", flush=True)
    names = ["du", "dA", "dB", "dC", "dD", "ddelta", "dbias", "dh0", "dz"]
    got = dict(zip(names, run(slice(0, batch))))
    summed = ("dA", "dD", "dbias")
    want = {k: torch.zeros_like(got[k], dtype=torch.float64) for k in summed}
    for b in range(batch):
        for k, t in zip(names, run(slice(b, b + 1))):
            if k in summed:
                want[k] += t.double()
            else:
                _near(got[k][b:b + 1], t, 17, f"{k} of row {b}")
    # sums of 2^16 terms a segment, one after the other: 2^-24 of the running
    # sum each, 2^-16 of it at random signs, and eight times that
    for k in summed:
        _near(got[k], want[k], 13, k)
