"""The tiled bfloat16 product of prompt portions (``ops.gemm_wide``): every tile at its edges and with
every activation against float64, the rule that picks a tile, and the products that are led to it."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TILES = [(64, 64), (128, 128), (128, 128), (128, 192), (128, 192), (96, 256), (256, 128), (128, 256),
         (160, 256), (256, 256)]


@pytest.fixture(scope="module")
def ops():
    from pylon_amd.kernels import ops

    return ops


def draw(seed, rows, k, pad=0):
    gen = torch.Generator(DEV).manual_seed(seed)
    return torch.randn(rows, k + pad, generator=gen, device=DEV).to(torch.bfloat16)[:, :k]


def wanted(x, w, epilogue):
    v = x.double() @ w.double().T
    if epilogue == "none":
        return v
    if epilogue == "relu2":
        return v.clamp(min=0) ** 2
    g, u = v.chunk(2, 1)
    if epilogue == "silu":
        return g * torch.sigmoid(g) * u
    if epilogue == "gelu_tanh":
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


def close(got, want):
    """One rounding to bfloat16 (seven bits behind the leading one: at most 2^-8 of the value), and float32
    sums and an activation ahead of it (2^-16 of the largest value)."""
    room = want.abs() * 1.01 * 2.0 ** -8 + want.abs().max() * 2.0 ** -16
    return bool(((got.double() - want).abs() <= room).all())


# K: one chunk (fewer than any tile keeps in flight), a few, more than all that are in flight
@pytest.mark.parametrize("k", [64, 128, 320, 704])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_every_tile_at_its_edges(ops, tile, k):
    rows, cols = TILES[tile]
    for m, n in ((rows, cols), (rows + 1, cols - 4), (2 * rows - 3, cols + 4), (5, 3 * cols + 12)):
        x, w = draw(m, m, k, 8), draw(n + k, n, k, 64)
        got = ops.gemm_wide(x, w, tile=tile)
        assert close(got, wanted(x, w, "none")), (m, n)
        assert torch.equal(got, ops.gemm_wide(x, w, tile=(tile + 3) % len(TILES))), (m, n)  # one order of sums


@pytest.mark.parametrize("epilogue", ["silu", "relu2", "gelu_tanh", "capped"])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_every_activation(ops, tile, epilogue):
    rows, cols = TILES[tile]
    m, n, k = rows + 7, cols + 4, 192
    x, w = draw(1, m, k), draw(2, 2 * n, k, 64) * 0.2
    got = ops.gemm_wide(x, w, epilogue=epilogue, alpha=1.702, offset=1.0, limit=7.0, tile=tile)
    assert close(got, wanted(x, w, epilogue))


def test_the_rule_names_a_tile_that_fills_the_chip():
    from pylon_amd.kernels import library

    tile, us = ctypes.c_int(), ctypes.c_float()
    for m, n, k, gated, expected in ((2048, 12288, 4096, 1, (256, 256)), (2048, 4096, 12288, 0, (256, 128)),
                                     (2048, 9728, 2560, 1, (160, 256)), (100, 2560, 4096, 0, (64, 64)),
                                     (656, 5120, 25600, 0, (128, 128))):
        assert library.load().pylon_gemm_wide_plan(m, n, k, gated, 256, ctypes.byref(tile), ctypes.byref(us)) == 0
        assert TILES[tile.value] == expected, (m, n, k, tile.value, us.value)


@pytest.mark.parametrize("rows", [65, 128, 129, 300, 1537])
def test_products_that_are_led_to_it(ops, rows):
    """Each dispatcher beside its own answer for rows it leads elsewhere or takes apart: K of no whole
    chunks, rows off a 16-byte boundary, odd strides of the result."""
    x, w = draw(rows, rows, 256), draw(3, 600, 256) * 0.1
    for k in (256, 248):  # 248: the library
        a, b = x[:, :k], w[:, :k]
        assert close(ops.linear(a, b), wanted(a, b, "none"))
        twice = k == 248  # the library rounds before the activation
        for got, want in ((ops.linear_glu(a, b, out_dtype=torch.bfloat16), wanted(a, b, "silu")),
                          (ops.linear_glu(a, b, out_dtype=torch.bfloat16, act="gelu_tanh"), wanted(a, b, "gelu_tanh")),
                          (ops.linear_relu2(a, b, out_dtype=torch.bfloat16), wanted(a, b, "relu2")),
                          (ops.linear_capped(a, b, alpha=1.702, offset=1.0, limit=7.0, out_dtype=torch.bfloat16),
                           wanted(a, b, "capped"))):
            assert close(got, want) or (twice and (got.double() - want).abs().max() <= 2e-2 * want.abs().max())
    for got, epilogue in ((ops.linear(x, w), "none"), (ops.linear_relu2(x, w, out_dtype=torch.bfloat16), "relu2"),
                          (ops.linear_glu(x, w, out_dtype=torch.bfloat16), "silu"),
                          (ops.linear_capped(x, w, alpha=1.702, offset=1.0, limit=7.0, out_dtype=torch.bfloat16), "capped")):
        assert torch.equal(got, ops.gemm_wide(x, w, epilogue=epilogue, alpha=1.702, offset=1.0, limit=7.0))
    into = torch.empty(rows, 600, dtype=torch.bfloat16, device=DEV)
    assert ops.linear(x, w, out=into) is into and close(into, wanted(x, w, "none"))
    assert close(ops.linear(x, w[:599]), wanted(x, w[:599], "none"))  # columns that are no multiple of 4: the library
    shifted = torch.zeros(rows * 256 + 1, dtype=torch.bfloat16, device=DEV)[1:].view(rows, 256).copy_(x)
    assert close(ops.linear(shifted, w), wanted(x, w, "none"))
    assert ops.linear(x, w, out_dtype=torch.float32).dtype == torch.float32


def test_infinities_stay_in_their_rows_and_columns(ops):
    x, w = draw(5, 100, 128), draw(6, 72, 128)
    x[3, 5], w[9, 0] = float("inf"), float("nan")
    got = ops.gemm_wide(x, w)
    keep = torch.ones(100, 72, dtype=torch.bool, device=DEV)
    keep[3], keep[:, 9] = False, False
    assert torch.isfinite(got[keep]).all() and torch.isnan(got[:, 9]).all() and not torch.isfinite(got[3]).any()


@pytest.mark.parametrize("tile", range(len(TILES)))
def test_operands_that_end_where_their_memory_ends(ops, tile):
    """Loads ahead of the last chunks of K fetch nothing: the last rows of both operands are the last bytes of
    allocations of their own (whole multiples of 2 MB, above what the allocator shares out)."""
    torch.cuda.empty_cache()
    x = draw(1, 5120, 1024).contiguous()
    w = draw(2, 5120, 1024).contiguous()
    got = ops.gemm_wide(x, w, tile=tile)
    again = ops.gemm_wide(torch.cat([x, x[:8]]), torch.cat([w, w[:8]]), tile=tile)  # with memory behind them
    assert torch.equal(got, again[:5120, :5120])
    assert close(got[-300:], wanted(x[-300:], w, "none"))


# one non-zero term a sum, so that the sums are exact and the gate alone is compared: up to 128 rows it is the
# same expf and division as in the activation kernels, to the bit; beyond, the hardware's functions (2^-22, and
# 2^-24 of the exponent's argument, ahead of the rounding)
@pytest.mark.parametrize("rows", [65, 128, 129])
@pytest.mark.parametrize("epilogue", ["silu", "gelu_tanh", "capped"])
def test_a_gate_keeps_its_precision_up_to_128_rows(ops, rows, epilogue):
    half, k, constants = 16384, 64, dict(alpha=1.702, offset=1.0, limit=7.0)
    gen = torch.Generator(DEV).manual_seed(rows)
    x = torch.zeros(rows, k, device=DEV)
    x[torch.arange(rows), torch.arange(rows) % k] = 2.0 * torch.rand(rows, generator=gen, device=DEV) + 1.0
    x, w = x.to(torch.bfloat16), draw(7, 2 * half, k) * 3
    sums = torch.mm(x, w.t(), out_dtype=torch.float32)
    if epilogue == "capped":
        got = ops.linear_capped(x, w, out_dtype=torch.bfloat16, **constants)
        behind = ops.gated_act(sums, out_dtype=torch.bfloat16, **constants)
    else:
        got = ops.linear_glu(x, w, out_dtype=torch.bfloat16, act=epilogue)
        behind = ops.silu_gate(sums, out_dtype=torch.bfloat16, act=epilogue)
    assert torch.equal(got, ops.gemm_wide(x, w, epilogue=epilogue, **constants))
    if rows <= 128:
        assert torch.equal(got, behind)
    else:
        torch.testing.assert_close(got, behind, rtol=2.0 ** -7, atol=1e-30)


@pytest.mark.parametrize("rows", [100, 300])  # the exact gate and the hardware's
@pytest.mark.parametrize("limit", [0.0, -1.0])
def test_a_gate_without_caps(ops, rows, limit):
    x, w = draw(1, rows, 192), draw(2, 160, 192) * 0.5
    got = ops.gemm_wide(x, w, epilogue="capped", alpha=0.7, offset=0.25, limit=limit)
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    assert g.abs().max() > 10  # more than the other tests' cap
    assert close(got, g * torch.sigmoid(0.7 * g) * (u + 0.25))
