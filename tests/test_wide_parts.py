"""Products of prompt portions with K cut into ranges, and projections of long portions: the rules, and what the parts'
entry points launch for them."""
import ctypes
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from pylon_amd.engine import layer_run
from pylon_amd.kernels import library, ops, plan


@pytest.mark.parametrize("rows", [129, 300, 512, 513, 640, 1024, 1500, 2048, 2112])
@pytest.mark.parametrize("n, k", [(2560, 4096), (2560, 9728), (5120, 25600), (4096, 4096), (1024, 512), (64, 64), (512, 1024)])
def test_ranges_of_k_are_whole_and_long(rows, n, k):
    parts, tile = ops.wide_parts(rows, n, k, 256)
    assert 1 <= parts <= 4 and (parts > 1) == (tile >= 0)
    assert parts == 1 or k // 64 >= 8 * parts


def test_deep_matrices_are_cut_and_full_launches_are_not():
    assert ops.wide_parts(2048, 2560, 9728, 256)[0] > 1 and ops.wide_parts(640, 5120, 25600, 256)[0] > 1
    assert ops.wide_parts(2048, 2560, 4096, 256)[0] == 1 and ops.wide_parts(2048, 5120, 25600, 256)[0] == 1


# us of product and norm uncut, in two, three and four ranges, and by the route before there were any: 768 rows 37.1, 30.2, 30.9,
# 30.7 and 34.9; 435 rows 38.9, 28.7, 31.5, 31.4 and 33.6; 512 rows 39.7, 31.5, 33.8, 32.4 and 37.3; and a matrix that the
# second-level caches hold, 335 rows 17.1, 18.7, 20.1, 22.2 and 20.9
@pytest.mark.parametrize("rows, n, k, cut", [(768, 2560, 4096, True), (435, 4096, 4096, True), (512, 4096, 4096, True),
                                             (335, 4096, 2048, False), (1024, 2560, 9728, True), (440, 2048, 6144, True)])
def test_full_rounds_of_small_tiles_are_cut_where_memory_holds_the_matrix(rows, n, k, cut):
    assert (ops.wide_parts(rows, n, k, 256)[0] > 1) is cut


def launches(rows, n, k, gated):
    """(columns of the first of two launches or 0, its tile, the tile of the others)"""
    (ahead, first, rest), us = (ctypes.c_int() for _ in range(3)), ctypes.c_float()
    call = library.load().pylon_gemm_wide_launches
    assert call(rows, n, k, int(gated), 256, *map(ctypes.byref, (ahead, first, rest, us))) == 0
    return ahead.value, first.value, rest.value, us.value


# gate/up of 4B, 8B and 32B sizes, the sizes whose results are compared on the device, and some that stay one launch
@pytest.mark.parametrize("rows, n, k, gated, ahead", [
    (2048, 9728, 2560, True, 8192), (2096, 12288, 4096, True, 10880), (1000, 25600, 5120, True, 24576),
    (1000, 9732, 1280, True, 6144), (2048, 9732, 576, True, 8192), (1000, 16516, 832, False, 16384),
    (2040, 8368, 832, False, 8192), (512, 25600, 5120, True, 0), (2048, 12288, 4096, True, 0), (2040, 5124, 320, False, 0)])
def test_whole_rounds_in_a_launch_of_their_own(rows, n, k, gated, ahead):
    columns, first, rest, us = launches(rows, n, k, gated)
    assert columns == ahead and (first < 0) == (ahead == 0)
    tile, alone = ctypes.c_int(), ctypes.c_float()
    assert library.load().pylon_gemm_wide_plan(rows, n, k, int(gated), 256, ctypes.byref(tile), ctypes.byref(alone)) == 0
    assert us < 0.98 * alone.value if ahead else (us, rest) == (alone.value, tile.value)  # what one launch of one tile takes


def test_launches_are_asked_for_products_that_there_are():
    place = ctypes.byref(ctypes.c_int())
    time = ctypes.byref(ctypes.c_float())
    call = library.load().pylon_gemm_wide_launches
    assert call(100, 64, 64, 0, 256, place, place, place, time) == 0
    assert call(0, 64, 64, 0, 256, place, place, place, time) != 0 and call(100, 64, 32, 0, 256, place, place, place, time) != 0
    assert call(100, 64, 64, 0, 256, None, place, place, time) != 0


# either side of whole rounds of 256 x 256 tiles (216 of 256 are five sixths, 192 are not), of the depth and of the rows
@pytest.mark.parametrize("rows, n, k, own", [
    (2048, 6144, 4096, True), (2049, 6144, 4096, False), (2049, 6144, 5120, True), (2048, 8192, 4096, False),
    (513, 6144, 2560, True), (512, 6144, 2560, False), (1000, plan.TALL, 5120, False)])
def test_projections_of_long_portions(rows, n, k, own):
    assert plan.portion_beats_library(rows, n, k) is own


@pytest.fixture
def launched(monkeypatch):
    seen = []

    def call(name, *args):
        if name.endswith("_plan"):
            return real(name, *args)
        seen.append((name.removeprefix("pylon_"), args))

    real = ops._lib.call
    monkeypatch.setattr(ops, "_raw_device", lambda: 0)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_watched", lambda x, weight: False)
    monkeypatch.setattr(ops._lib, "compute_units", lambda: 256)
    monkeypatch.setattr(ops._lib, "call", call)
    plain = torch.nn.functional.linear
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: (seen.append(("library", ())), plain(x, w))[1])
    with FakeTensorMode(), warnings.catch_warnings():
        warnings.simplefilter("ignore")  # data pointers of tensors without data
        yield seen


def empty(rows, k, gap=0, dtype=torch.bfloat16):
    return torch.empty(rows, k + gap, dtype=dtype, device="cuda:0")[:, :k]


@pytest.mark.parametrize("gap", [0, 64])
def test_a_portions_residual_product_is_the_tiled_kernels(launched, gap):
    """Float parts, or one bfloat16 result; as many as the layers launched by one call expect.  Few rows, operands that
    the kernel does not take and products that something follows go where they went."""
    for rows in (129, 192, 300, 512, 700, 2048):
        for n, k in ((2560, 4096), (2560, 9728), (4096, 4096), (1024, 1024), (1024, 3072)):
            launched.clear()
            got = ops.linear_into_residual(empty(rows, k), empty(n, k, gap), out_dtype=torch.bfloat16)
            parts, tile = ops.wide_parts(rows, n, k, 256)
            (name, args), = launched
            if parts > 1:
                assert name == "gemm_wide_parts" and args[-3:-1] == (parts, tile)
                assert got.dtype == torch.float32 and got.shape == (parts, rows, n)
            else:
                assert name == "gemm_wide" and got.dtype == torch.bfloat16 and got.shape == (rows, n)
            assert layer_run._into_residual(rows, n, k, k + gap, 256) == ((parts, -1 - tile) if parts > 1 else (0, 0))
            whole = ops.linear_into_residual(empty(rows, k), empty(n, k, gap), out_dtype=torch.float32)
            assert whole.dtype == torch.float32 and whole.shape[-2:] == (rows, n) and (whole.dim() == 3) == (parts > 1)
    for rows, n, k in ((128, 2560, 4096), (300, 2560, 4104), (300, 2562, 4096)):
        asked = []
        for entry in (ops.linear_into_residual, ops.linear_for_residual):
            launched.clear()
            entry(empty(rows, k), empty(n, k, gap), out_dtype=torch.bfloat16)
            asked.append([name for name, _ in launched])
        assert asked[0] == asked[1] and "gemm_wide_parts" not in asked[0]
        assert layer_run._into_residual(rows, n, k, k + gap, 256) == layer_run._residual(rows, n, k, k + gap, 256)


def test_an_uncut_product_that_the_librarys_tiles_fill_is_the_librarys(launched):
    for rows, n, k, name in ((2048, 8192, 8192, "library"), (2049, 8192, 8192, "gemm_wide"), (3000, 5120, 8192, "library"),
                             (2048, 5120, 8192, "gemm_wide"), (1000, 8192, 8192, "gemm_wide"), (1792, 8192, 28672, "gemm_wide")):
        assert ops.wide_parts(rows, n, k, 256)[0] == 1
        launched.clear()
        got = ops.linear_into_residual(empty(rows, k), empty(n, k), out_dtype=torch.bfloat16)
        assert [seen for seen, _ in launched] == [name] and got.dtype == torch.bfloat16 and got.shape == (rows, n)
        launched.clear()
        ops.linear_into_residual(empty(rows, k), empty(n, k), out_dtype=torch.float32)  # whose sums are to stay unrounded
        assert [seen for seen, _ in launched] == ["gemm_wide_parts"]


def test_a_followed_product_stays_with_the_library(launched, monkeypatch):
    monkeypatch.setattr(ops, "_watched", lambda x, weight: True)
    ops.linear_into_residual(empty(2048, 9728), empty(2560, 9728), out_dtype=torch.bfloat16)
    ops.linear_of_portion(empty(2048, 2560), empty(6144, 2560), out_dtype=torch.bfloat16)
    assert [name for name, _ in launched] == ["library"] * 2


def test_a_long_portions_projection(launched):
    for rows, n, k, name in ((2048, 6144, 2560, "gemm_wide"), (2048, 8192, 4096, "library"), (2048, 6144, 2564, "library")):
        launched.clear()
        assert ops.linear_of_portion(empty(rows, k), empty(n, k), out_dtype=torch.bfloat16).shape == (rows, n)
        assert [seen for seen, _ in launched] == [name]


# rows of a multiple of 8 KB: either side of 1,024 rows, of tiles of 192 rows or columns that fit one round, of three quarters
# of one and five sixths of several, of 16 KB; of other rows what there was
@pytest.mark.parametrize("rows, n, k, own", [
    (1700, 8192, 4096, False), (1538, 8192, 4096, False), (1536, 8192, 4096, True), (1024, 16384, 4096, True),
    (1728, 7168, 4096, True), (1729, 7168, 4096, False), (1152, 10240, 4096, True), (1153, 10240, 4096, False),
    (1300, 9216, 8192, True), (1345, 9216, 8192, False), (2048, 12288, 4096, True), (2049, 12288, 4096, False),
    (4096, 10240, 4096, True), (2048, 8192, 8192, False), (2048, 8192, 12288, True), (1536, 10560, 2560, True),
    (2048, 14592, 2560, False), (2048, 10240, 5120, True)])
def test_the_rule_for_projections_decides_both_ways(launched, rows, n, k, own):
    ops.linear_of_portion(empty(rows, k), empty(n, k), out_dtype=torch.bfloat16)
    assert [seen for seen, _ in launched] == ["gemm_wide" if own else "library"]
    assert plan.portion_beats_library(rows, n, k) is own
    assert plan.portion_beats_library(rows, n, k, units=100000) is True  # a device whose rounds nothing fills
