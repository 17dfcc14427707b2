"""The tiled bfloat16 product's float sums of ranges of K, its tiles of 160 and 192 columns, and its launches in two."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TILES = [(64, 64), (128, 128), (128, 128), (128, 192), (128, 192), (96, 256), (256, 128), (128, 256), (160, 256), (256, 256),
         (128, 160), (256, 160), (256, 192), (192, 256)]


@pytest.fixture(scope="module")
def ops():
    from pylon_amd.kernels import ops

    return ops


def draw(seed, rows, k, pad=0):
    gen = torch.Generator(DEV).manual_seed(seed)
    return torch.randn(rows, k + pad, generator=gen, device=DEV).to(torch.bfloat16)[:, :k]


# one chunk a range and ranges of unequal length; K of one chunk, a few, more than all that are in flight
@pytest.mark.parametrize("k, parts", [(64, 1), (128, 2), (320, 3), (704, 4), (704, 1), (1088, 8)])
@pytest.mark.parametrize("tile", range(len(TILES)))
def test_sums_of_ranges(ops, tile, k, parts):
    rows, cols = TILES[tile]
    for m, n in ((rows, cols), (rows + 1, cols - 4), (2 * rows - 3, cols + 4), (5, 3 * cols + 12)):
        x, w = draw(m, m, k, 8), draw(n + k, n, k, 64)
        got = ops.gemm_wide_parts(x, w, parts=parts, tile=tile)
        assert got.dtype == torch.float32
        chunks = k // 64
        for p, sums in enumerate(got if parts > 1 else got[None]):
            at = slice(chunks * p // parts * 64, chunks * (p + 1) // parts * 64)
            want = x[:, at].double() @ w[:, at].double().T
            # float32 sums of up to 1,088 exact products: 2^-24 of the running sum each, far below 2^-16 of the largest
            assert (sums.double() - want).abs().max() <= want.abs().max() * 2.0 ** -16, (m, n, p)
        assert torch.equal(got, ops.gemm_wide_parts(x, w, parts=parts, tile=(tile + 3) % len(TILES))), (m, n)


@pytest.mark.parametrize("tile", [10, 11, 12, 13])
def test_tiles_of_160_and_192_columns(ops, tile):
    rows, cols = TILES[tile]
    for k in (64, 128, 704):
        for m, n in ((rows, cols), (rows + 1, cols - 4), (2 * rows - 3, cols + 4), (5, 3 * cols + 12)):
            x, w = draw(m, m, k, 8), draw(n + k, n, k, 64)
            assert torch.equal(ops.gemm_wide(x, w, tile=tile), ops.gemm_wide(x, w, tile=1))
            assert torch.equal(ops.gemm_wide(x, w, epilogue="relu2", tile=tile), ops.gemm_wide(x, w, epilogue="relu2", tile=1))
    x, w = draw(1, 300, 192), draw(2, 2 * 260, 192, 64) * 0.2
    if cols % 64 == 0:
        assert torch.equal(ops.gemm_wide(x, w, epilogue="silu", tile=tile), ops.gemm_wide(x, w, epilogue="silu", tile=6))
    else:
        with pytest.raises(ops.KernelError):  # a gate tile and its up tile belong to one wave
            ops.gemm_wide(x, w, epilogue="silu", tile=tile)


# whole rounds in a launch of their own, the other columns, the last tile of them ragged, in another (whose up rows are as far
# from its gate rows as the whole matrix's); rows of whole tiles and ragged ones
@pytest.mark.parametrize("m, n, k, epilogue, ahead", [
    (1000, 9732, 1280, "silu", 6144), (2048, 9732, 576, "capped", 8192), (1000, 16516, 832, "none", 16384),
    (2040, 8368, 832, "relu2", 8192)])
def test_launches_in_two(ops, m, n, k, epilogue, ahead):
    from pylon_amd.kernels import library

    gated = epilogue in ("silu", "capped")
    (columns, first, rest), us = (ctypes.c_int() for _ in range(3)), ctypes.c_float()
    assert library.load().pylon_gemm_wide_launches(m, n, k, int(gated), 0, *map(ctypes.byref, (columns, first, rest, us))) == 0
    assert columns.value == ahead and (n - ahead) % TILES[rest.value][1] != 0
    x, w = draw(1, m, k), draw(2, 2 * n if gated else n, k, 64) * 0.2
    got = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    options = dict(epilogue=epilogue, alpha=1.702, offset=1.0, limit=7.0)
    ops.gemm_wide(x, w, out=got, **options)
    assert torch.equal(got, ops.gemm_wide(x, w, tile=6, **options))


def test_every_tile_has_the_same_sums_of_many_ranges(ops):
    """Whole tiles and ragged ones over all compute units, ranges of five, five and six chunks: the bits of the first tile,
    whose sums the tests above compare with 64 bits."""
    x, w = draw(1, 5120, 1024).contiguous(), draw(2, 5120, 1024).contiguous()
    for tile in range(len(TILES)):
        got = ops.gemm_wide_parts(x, w, parts=3, tile=tile)
        if tile == 0:
            first = got
        assert torch.equal(got, first)


def test_what_the_residual_norm_makes_of_parts(ops):
    """A deep product of a portion with its norm, against 64 bits: as close as with the product rounded first."""
    x, w = draw(3, 700, 9728), draw(4, 2560, 9728) * 0.02
    resid, gain = torch.randn(700, 2560, device=DEV), torch.rand(2560, device=DEV)
    delta = ops.linear_into_residual(x, w, out_dtype=torch.bfloat16)
    assert delta.dtype == torch.float32 and delta.dim() == 3
    want = resid.double() + x.double() @ w.double().T
    scaled = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-6) * gain.double()
    out = ops.add_rmsnorm(resid, delta, gain, 1e-6, torch.bfloat16)
    assert ((resid.double() - want).abs() <= want.abs() * 2.0 ** -22 + want.abs().max() * 2.0 ** -17).all()
    assert ((out.double() - scaled).abs() <= scaled.abs() * 1.01 * 2.0 ** -8 + scaled.abs().max() * 2.0 ** -16).all()


def test_arguments_that_are_refused(ops):
    from pylon_amd.kernels import library

    x, w = draw(1, 200, 256), draw(2, 64, 256)
    for parts, tile in ((5, 0), (0, 0), (9, 0), (2, -1), (2, len(TILES)), (1, -2)):  # four chunks: at most four ranges
        with pytest.raises(ops.KernelError):
            ops.gemm_wide_parts(x, w, parts=parts, tile=tile)
    with pytest.raises(ops.KernelError):
        ops.gemm_wide_parts(x, w[:62], parts=2, tile=0)
    with pytest.raises(ops.KernelError):
        ops.gemm_wide_parts(x[:, :200], w[:, :200], parts=2, tile=0)
    assert library.load().pylon_gemm_wide_parts_plan(0, 64, 64, 256, None, None, None) != 0
