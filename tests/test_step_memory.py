"""Start-up asks for the memory of the step that takes the most, which need not be the largest one."""
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from pylon_amd.engine.runner import rows_to_measure
from pylon_amd.kernels import ops

UNITS = 256
SHAPES = {"4b": ((2560, 4096), (2560, 9728)), "8b": ((4096, 4096), (4096, 12288)), "32b": ((5120, 8192), (5120, 25600)),
          "deep and shallow": ((2560, 1280), (2560, 14592)), "no whole chunks": ((2560, 4104), (2562, 4096))}


@pytest.mark.parametrize("most", [1, 128, 129, 255, 2048, 2055, 2111, 4200])
@pytest.mark.parametrize("shape", SHAPES)
def test_no_step_takes_more_than_the_measured_ones(shape, most):
    products = SHAPES[shape]
    measured = rows_to_measure(products, most, UNITS)
    assert measured[0] == most and len(measured) <= 12 and measured == sorted(set(measured), reverse=True)
    taken = {rows: [ops.residual_bytes(rows, n, k, UNITS) for n, k in products] for rows in range(1, most + 1)}
    for rows, mine in taken.items():
        assert any(more >= rows and all(a >= b for a, b in zip(taken[more], mine)) for more in measured), rows


def test_a_portion_below_the_largest_step_takes_more():
    """2,048 prompt tokens beside 63 decoding requests: float sums of ranges of K are more bytes for fewer rows."""
    for shape, rows in (("8b", 2048), ("32b", 1792)):
        products = SHAPES[shape]
        assert rows in rows_to_measure(products, 2111, UNITS)
        assert sum(ops.residual_bytes(rows, n, k, UNITS) for n, k in products) > \
            2 * sum(ops.residual_bytes(2111, n, k, UNITS) for n, k in products)


def test_products_whose_results_grow_with_the_rows_take_one_step():
    assert rows_to_measure((), 2111, UNITS) == [2111] and rows_to_measure(SHAPES["4b"], 0, UNITS) == []


# as the parts' entry point allocates it: partial sums, one bfloat16 result, operands that the library takes
@pytest.mark.parametrize("rows, n, k", [(8, 2560, 4096), (128, 2560, 9728), (129, 4096, 12288), (2048, 4096, 12288),
                                        (2049, 4096, 12288), (300, 2562, 4096), (2048, 2560, 4096)])
def test_the_bytes_are_those_of_the_result(monkeypatch, rows, n, k):
    real = ops._lib.call
    monkeypatch.setattr(ops, "_raw_device", lambda: 0)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_watched", lambda x, weight: False)
    monkeypatch.setattr(ops._lib, "compute_units", lambda: UNITS)
    monkeypatch.setattr(ops._lib, "call", lambda name, *args: real(name, *args) if name.endswith("_plan") else None)
    with FakeTensorMode(), warnings.catch_warnings():
        warnings.simplefilter("ignore")  # data pointers of tensors without data
        x, w = (torch.empty(r, k, dtype=torch.bfloat16, device="cuda:0") for r in (rows, n))
        got = ops.linear_into_residual(x, w, out_dtype=torch.bfloat16)
    assert got.numel() * got.element_size() == ops.residual_bytes(rows, n, k, UNITS)
