"""The float32 product (``ops.gemm_tiled`` with float32 operands): every kernel it is made of at the
edges of their tiles, against a float64 product with the error bound of the order its sums are taken in,
and one value per element whatever rows share the launch."""
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
UNIT = 2.0 ** -24  # float32's unit roundoff


@pytest.fixture(scope="module")
def ops():
    from pylon_amd.kernels import ops

    return ops


def draw(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator(DEV).manual_seed(seed), device=DEV)


def within_bound(got, x, w, ranges=True):
    """A chain of at most n fused multiply-adds is off by at most n units of the sum of the products'
    magnitudes; each range of K is such a chain, and eight sums follow.  (Without ranges: one chain.)"""
    k = x.shape[1]
    chain = 64 * -(-(-(-k // 64)) // 8) + 8 if k >= 512 and ranges else k
    want = x.double() @ w.double().T
    room = 1.01 * chain * UNIT * (x.double().abs() @ w.double().abs().T)
    return bool(((got.double() - want).abs() <= room).all())


# rows: the streaming kernel's one and two row tiles, tiles of 32 and of 64; columns: part of a tile,
# several tiles a workgroup, workgroups of the last round; K: below the shortest that the kernels take, one
# chunk a range, uneven ranges, a part chunk
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 32, 33, 65, 511, 520])
@pytest.mark.parametrize("n, k", [(17, 508), (1, 512), (16, 516), (70, 576), (300, 1100), (20, 2560), (26000, 520)])
def test_against_float64(ops, rows, n, k):
    x, w = draw(rows, rows, k), draw(n + k, n, k)
    got = ops.gemm_tiled(x, w)
    assert within_bound(got, x, w)
    for first, last in ((0, 1), (rows // 2, rows), (rows - 1, rows)):  # the rows' own values, to the bit
        assert torch.equal(ops.gemm_tiled(x[first:last].contiguous(), w), got[first:last])


def test_tiles_of_64_agree_with_the_streaming_kernel(ops):
    x, w = draw(1, 700, 640), draw(2, 5000, 640)  # 11 x 79 tiles: three rounds of the chip
    got = ops.gemm_tiled(x, w)
    assert within_bound(got, x, w)
    for first, last in ((0, 20), (330, 400), (699, 700)):
        assert torch.equal(ops.gemm_tiled(x[first:last].contiguous(), w), got[first:last])


# sizes at which each of the tiles is chosen, one row and one column past whole tiles among them: 32 x 32, 32 x 64, 48 x
# 64, 48 x 64 by two teams, 64 x 64, 64 x 64 by two teams, 96 x 64; and the streaming kernel's narrower shares
@pytest.mark.parametrize("rows, n, k", [(97, 2560, 576), (100, 19455, 520), (181, 19457, 516), (270, 2561, 640),
                                        (32770, 70, 520), (360, 2497, 1100), (287, 19455, 576), (5, 5121, 520),
                                        (17, 2561, 8192), (16, 2561, 8188), (16, 2561, 8196), (1, 17, 8192)])
def test_every_tile_against_float64(ops, rows, n, k):
    x, w = draw(rows, rows, k), draw(n + k, n, k)
    got = ops.gemm_tiled(x, w)
    assert within_bound(got, x, w)
    for first, last in ((0, 1), (rows // 2, rows // 2 + 9), (rows - 1, rows)):  # the streaming kernel's bits
        assert torch.equal(ops.gemm_tiled(x[first:last].contiguous(), w), got[first:last])


def test_strided_rows_and_rows_that_are_not_aligned(ops):
    x, w = draw(3, 40, 600), draw(4, 50, 604)
    for cut in (600, 599):  # 16-byte pieces, and a K that has none (the general kernel)
        a, b = x[:, :cut], w[:, :cut]
        assert within_bound(ops.gemm_tiled(a, b), a, b, ranges=cut == 600)
        torch.testing.assert_close(ops.gemm_tiled(a, b).double(), a.double() @ b.double().T, rtol=0, atol=5e-4)
    shifted = draw(5, 40 * 600 + 1)[1:].view(40, 600)  # rows that begin off a 16-byte boundary
    assert within_bound(ops.gemm_tiled(shifted, w[:, :600]), shifted, w[:, :600], ranges=False)
    torch.testing.assert_close(ops.gemm_tiled(shifted, w[:, :600]).double(), shifted.double() @ w[:, :600].double().T,
                               rtol=0, atol=5e-4)


@pytest.mark.parametrize("rows", [3, 40])
def test_numbers_at_the_ends_of_the_range(ops, rows):
    x, w = torch.zeros(rows, 512, device=DEV), torch.zeros(5, 512, device=DEV)
    x[:, 0], w[0, 0], w[1, 0] = 1.0, 1e-40, 3e38  # a subnormal number stays what it is
    x[1, 1], w[2, 1] = float("inf"), 1.0
    w[3, 2] = float("nan")
    got = ops.gemm_tiled(x, w)
    assert got[0, 0].item() == w[0, 0].item() and got[0, 1].item() == w[1, 0].item()
    assert torch.isinf(got[1, 2]) and got[0, 2].item() == 0.0
    assert torch.isnan(got[0, 3]) and torch.isnan(got[1, 0]) and got[0, 4].item() == 0.0


def test_threads_with_launches_of_different_sizes(ops):
    """Every host thread its own stream and shape, each with launches of other sizes beside it."""
    shapes = [(3, 64, 512), (3, 26000, 512), (32, 26000, 512), (20, 300, 512)]
    operands = [(draw(m, m, k), draw(n, n, k)) for m, n, k in shapes]
    want = [ops.gemm_tiled(x, w) for x, w in operands]
    torch.cuda.synchronize()

    def work(i):
        x, w = operands[i]
        with torch.cuda.stream(torch.cuda.Stream()):
            got = [ops.gemm_tiled(x, w) for _ in range(40)]
            torch.cuda.current_stream().synchronize()
            return all(torch.equal(g, want[i]) for g in got)

    with ThreadPoolExecutor(len(shapes)) as pool:
        assert all(pool.map(work, range(len(shapes))))
