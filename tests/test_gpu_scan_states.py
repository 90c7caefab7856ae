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
