"""Which calls of the product entry points reach a kernel of the engine, which the library and which are
refused: on the CPU, with tensors that have a device and a shape but no data."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from pylon_amd.kernels import ops


def empty(*shape, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device="cuda:0")


@pytest.mark.parametrize("act", ["relu2", "capped", "none", "tanh"])
@pytest.mark.parametrize("rows", [8, 100, 300])
def test_what_is_no_gate_is_refused(rows, act):
    with FakeTensorMode(), pytest.raises(KeyError):
        ops.linear_glu(empty(rows, 256), empty(512, 256), out_dtype=torch.bfloat16, act=act)
