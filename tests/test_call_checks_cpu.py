"""What the Python entry points refuse before they call the library, on the
CPU: arrays that are no tensors, and rows of no columns (a view of no columns
has a valid address: the library would read in_dim elements from it)."""
import numpy as np
import pytest
import torch

import xtern


class Weights:
    in_dim, out_dim, handle = 4, 2, None


ONES = torch.ones(3)
CALLS = {
    "linear_f32": lambda x: xtern.linear_f32(Weights, x),
    "linear_f32 out": lambda x: xtern.linear_f32(Weights, x, out=torch.zeros(3, 2)),
    "linear_f32_noalloc": lambda x: xtern.linear_f32_noalloc(Weights, x, out=torch.zeros(3, 2)),
    "linear_q": lambda x: xtern.linear_q(Weights, x, ONES),
    "linear_q_rowsum": lambda x: xtern.linear_q_rowsum(Weights, x, ONES, ONES, out=torch.zeros(3, 2)),
    "linear_multi_f32": lambda x: xtern.linear_multi_f32([Weights], x, outs=[torch.zeros(3, 2)]),
    "linear_multi_q": lambda x: xtern.linear_multi_q([Weights], x, ONES),
    "quantize_i8": lambda x: xtern.quantize_i8(x),
    "quantize_i8_rowsum": lambda x: xtern.quantize_i8_rowsum(x),
}


@pytest.mark.parametrize("name", list(CALLS))
def test_arrays_and_host_tensors(name):
    for x in (np.zeros((3, 4), np.float32), np.zeros(4, np.float32), torch.zeros(3, 4), torch.zeros(2, 3, 4)):
        with pytest.raises(xtern.XternError, match="must be a CUDA"):
            CALLS[name](x)


@pytest.mark.parametrize("name", list(CALLS))
def test_rows_of_no_columns(name):
    for x in (torch.zeros(3, 0), torch.zeros(3, 4)[:, :0], torch.zeros(0), torch.zeros(2, 3, 0)):
        with pytest.raises(RuntimeError, match="cannot reshape"):
            CALLS[name](x)
