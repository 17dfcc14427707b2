"""Which kernel multiplies a few rows of bfloat16 activations by a bfloat16 matrix.

Pure functions of the shape: they touch no tensor and run anywhere, so the choices can be
tested without a GPU.  Every figure below was measured on one MI355X, under a graph, over 36
different matrices in turn (so that none came from a cache).  Those of the rows kernel are from before its loads
of w were marked as read once: it takes 4 to 16 % less since (2560 x 9728 at 8 rows 11.2 -> 10.1 us, 2 x 9728 x 2560 20.5
-> 18.1, 6144 x 4096 12.9 -> 11.0; two halves of the rows 2 to 5 %).  No line was drawn again for that; where one was known
to lie too far on the other kernel's side already, the text beside it says so.

Three kernels take part.  ``rows`` (``gemm_rows``): both operands go through LDS in whole
256-byte row segments, the rows of x are shared by a workgroup, K may be cut over workgroups.
``skinny`` (``gemm_skinny``): the earlier one, whose waves split K and read x in the shape of
a matrix-instruction operand.  ``library``: the library's tiled product.  Up to 64 rows the
product is bound by moving the matrix once, and by what a compute unit can pull: the first
kernel wins almost everywhere; the exceptions are listed where they are decided.
"""
from __future__ import annotations

from dataclasses import dataclass
from functools import lru_cache

FEW_ROWS = 16      # one tile of rows of x
STREAM_ROWS = 64   # most rows of x a workgroup of a weight-streaming kernel takes
SPLIT_ROWS = 128   # most rows the rows kernel takes as two halves, each to workgroups of its own
TALL = 32768       # a matrix of at least this many rows (a vocabulary head) is "tall"
UNITS = 256        # compute units of an MI355X; callers on a device pass its own count


@dataclass(frozen=True)
class Product:
    """``kernel``: "rows", "skinny" or "library"; ``parts``: ranges K is cut into (each a float
    partial result for the consumer to add); ``col_tiles``: tiles of 16 columns per wave of
    the rows kernel."""
    kernel: str
    parts: int = 1
    col_tiles: int = 1


def aliased_rows(k: int) -> bool:
    """Rows of a power-of-two length of 8 KB or more: the 256-byte segments that a chunk is of
    many rows then meet in few memory channels, and the rows kernel streams 10 to 20 % slower
    (gate/up 2x12288 x 4096 at 8 rows: 42 us against the skinny kernel's 39)."""
    return k % 4096 == 0


def gated_row_padding(k: int, element_size: int) -> int:
    """Elements to leave unused behind every row of a fused gate/up matrix of 16-bit elements
    (of rows of at least 1,024 of them).
    A workgroup's gate rows and its up rows, half the matrix further, otherwise tend to meet in
    the same memory channels, most of all where a row is a power-of-two length of 8 KB or more:
    2x12288 x 4096: the rows kernel at 8 rows 42.4 -> 35.4 us (which then beats the skinny
    kernel's 38.7), at 64 rows 45.1 -> 37.9.  At other widths the streaming kernels gain little
    (2x9728 x 2560 at 8 rows 20.1 -> 19.5 us) and the library's product for prompt portions some
    (2,048 rows of 2x9728 x 2560: 212 -> 187 us alone, 0.2 ms of a 19.8 ms step): a whole step
    at the Qwen3-4B shape 2.526 -> 2.516 ms decoding and 19.81 -> 19.60 ms for 2,048 prompt tokens,
    old and new in turn on one device, three times.  The other products are within 1 % either
    way and stay as they are; 192 elements do no better than 64."""
    return 64 if element_size == 2 and k >= 1024 else 0  # not worth doubling a toy's matrix


def head_row_padding(k: int, element_size: int) -> int:
    """The same behind the rows of a vocabulary head of its own (one that is the embedding too is read row by row
    as it lies), where a row is a multiple of 8 KB, but no power of two beyond it.  ``linear``, us, close -> apart, the
    rows kernel with 64 and 128 columns a workgroup or, close and beyond 32 rows, the library:

    151936 x 4096 at 1, 8, 24, 33, 48 and 64 rows 226, 229, 252, 258, 261, 270 -> 206, 205, 212, 215, 221, 228;
    32000 x 4096 at 1, 32, 48, 64 rows 53, 57, 65, 60 -> 47, 49, 67, 50;
    128256 x 12288 at 1, 8, 32, 48, 64 rows 546, 555, 574, 586, 613 -> 533, 536, 543, 544, 562;
    65536 x 20480 at 1, 32, 64 rows 455, 477, 484 -> 451, 454, 472.
    But 65536 x 8192 at 1, 32, 33, 48, 64 rows 233, 237, 214, 205, 216 -> 229, 235, 240, 242, 245; 151936 x 8192 at
    33, 48 rows 494, 479 -> 512, 516; 128256 x 16384 at 33, 48 rows 755, 757 -> 787, 805: the library does well with
    those as they lie.  From 65 rows on (the library) at most 1.5 % slower and up to 30 % faster; heads of other
    widths are within 2 %."""
    return 64 if element_size == 2 and aliased_rows(k) and (k == 4096 or k & (k - 1)) else 0


def rows_split(n: int, k: int, rows: int = STREAM_ROWS, units: int = UNITS) -> tuple:
    """(parts, col_tiles) of the rows kernel for a product into the residual stream.
    Workgroups of 128 columns for deep matrices (beyond 16 rows, where the rows of x weigh
    more, from a depth of 8192) and for wide ones, else of 64; K cut into the largest power of
    two of parts (at most 16, of at least 256 elements each) that keeps the workgroups at one
    per compute unit or fewer: more of them only re-read the rows of x.  (The kernel then gives
    every workgroup the same share of the columns, so that the launch fills whole rounds of the
    units, where the share stays at least as many rows of w as there are rows of x.)"""
    col_tiles = 2 if (k >= 8192 and rows > FEW_ROWS) or k >= 16384 or n > 4096 else 1
    groups = -(-n // (64 * col_tiles))
    parts = 1
    while parts < 16 and 2 * parts * groups <= units and k // (2 * parts) >= 256:
        parts *= 2
    return parts, col_tiles


def skinny_parts(n: int, k: int, units: int = UNITS) -> int:
    """Ranges the skinny kernel cuts K into so that a matrix of few rows still fills the chip
    (at most 4: with 8 a whole decode step measured 7 % slower)."""
    tiles = (n + 15) // 16
    parts = 1
    while tiles * parts < 2 * units and parts < 4 and k // (parts * 2) >= 512:
        parts *= 2
    return parts


def deep_or_narrow(n: int, k: int) -> bool:
    """Matrices much deeper than wide (a down projection) and those of few rows (an out
    projection)."""
    return k >= 2 * n or n <= 4096


@lru_cache(maxsize=4096)  # asked for every product of a step
def plan_residual(rows: int, n: int, k: int, units: int = UNITS) -> Product:
    """A product about to be added to the float32 residual stream (out and down projections),
    ``rows`` <= 128: float32 sums, never rounded, from whichever kernel.

    Up to 16 rows the rows kernel beats the skinny one for deep, narrow and moderately wide
    matrices (2560x4096 at 8 rows: 5.8 against 8.5 us, 2560x9728 10.9 against 14.0, 5120x8192
    20.1 against 23.2, 5120x25600 48 against 65).  Of wider ones those whose rows are of a power-of-two
    length are the skinny kernel's (16384x4096 30 against 35); the others stay with it, too, since an earlier form of
    the rows kernel (10240x10240 59, where the rows kernel now takes 36).  From 17 to 64 rows the rows
    kernel with K cut into parts beats the library, which does not cut K (at 64 rows: 2560x4096 8.5 against
    14.3 us, 2560x9728 13.4 against 28.0, 4096x4096 9.5 against 15.1, 4096x12288 22.4 against
    36.6, 5120x5120 13.5 against 21.5, 5120x8192 21.4 against 28.8, 5120x17408 37 against 86,
    6144x6144 17.7 against 25.4, 10240x10240 42 against 57), except for wide matrices whose rows
    are of a power-of-two length (8192x8192 33.9 against 32.2, 16384x4096 36.0 against 32.6).
    From 65 to 128 rows the rows kernel takes the rows as two halves, each to workgroups of its
    own, two that stream the same rows of w side by side on one die: 2560x9728 at 65, 96 and 128
    rows 19.0, 19.9 and 22.4 us against the library's 25.3, 26.0 and 52.2 (bfloat16 result),
    2560x4096 12.1, 13.2 and 15.0 against 13.1, 13.0 and 23.8; the same choices as for 64 rows."""
    few = rows <= FEW_ROWS
    if few:
        if deep_or_narrow(n, k) or n <= 8192:
            return Product("rows", *rows_split(n, k, rows, units))
        return Product("skinny", skinny_parts(n, k, units))
    if aliased_rows(k) and n >= 8192:
        return Product("library")
    return Product("rows", *rows_split(n, k, rows, units))


@lru_cache(maxsize=4096)  # asked for every product of a step
def plan_projection(rows: int, n: int, k: int, row_stride: int = 0) -> Product:
    """Any other product (q/k/v; the vocabulary head) of up to 64 rows; what it leaves to the library and what has
    more rows may still go to a kernel (:func:`rows_match_library`, :func:`wide_beats_library`).  ``row_stride``: of the
    matrix in memory; it counts at the widths of :func:`head_row_padding`.

    A head (tall matrix): the rows kernel with 128 columns per workgroup (151936 x 2560: 137 us
    against the skinny kernel's 157 at 8 rows; 167 against the library's 184 at 64 rows, 147
    against 171 at 32; x 5120: 267 against 302 and 294 against 310).  With aliased rows (x 4096)
    64 columns per workgroup do better (221 against 224 us at 1 row, 229 against 231 at 8, 258
    against 276 at 32), and beyond 32 rows the library (270 against 291 and 287 at 64 rows); an
    engine's head of that width has its rows apart (:func:`head_row_padding`) and goes as the others.
    A projection up to 16 rows: the rows kernel (6144 x 2560 at 8 rows 9.4 against the skinny
    kernel's 12.1 us, 10240 x 5120 20 against 31, 6144 x 4096 11.7 against 16.2).  Beyond 16
    rows the library, beside which the rows kernel without K cut over workgroups was within 10 % either way when
    this line was drawn, with the rows of x of a workgroup that covers 64 of many columns weighing most (now 6144 x
    2560 11.7 against 13.1 us at 32 rows, 13.2 against 15.5 at 64; 6144 x 4096 14.3 against 15.1 and 19.0
    against 17.8); a consumer that adds partial sums gets them (:func:`plan_summed_later`)."""
    few = rows <= FEW_ROWS
    if rows > STREAM_ROWS:
        return Product("library")
    if n >= TALL:
        if aliased_rows(k) and not (head_row_padding(k, 2) and row_stride > k and not aliased_rows(row_stride)):
            return Product("rows", 1, 1) if rows <= 32 else Product("library")
        return Product("rows", 1, 2)
    return Product("rows") if few else Product("library")


@lru_cache(maxsize=4096)  # asked for every product of a step
def plan_summed_later(rows: int, n: int, k: int, units: int = UNITS) -> Product:
    """A projection whose consumer can add float partial sums itself (q/k/v in front of the
    decode attention that prepares its own operands): K is cut over workgroups where the uncut
    launch would leave compute units without one.

    Up to 16 rows: workgroups of 64 columns and 2 or 4 parts, as many as keep the workgroups
    within the units.  At 8 rows 6144 x 2560 takes 7.6 us (2 parts) against 9.4 uncut, 4096 x
    2048 5.0 (4) against 7.1, 7168 x 2560 8.6 against 9.3; 6144 x 4096 (12.1 against 11.7) and 7168 x 5120 (14.1
    either way) gain nothing since an uncut launch starts sooner; 10240 x 5120 stays uncut.  With what the
    attention kernel then pays for adding them, a whole step at the Qwen3-4B shape, batch 8, was 2.603 -> 2.531 ms.
    From 17 to 64 rows the rows kernel so cut beats the library, which does not cut K: 6144 x
    2560 at 17, 32, 48 and 64 rows 8.0, 8.3, 9.3 and 9.8 us (four parts of 128 columns) against
    12.6, 13.1, 15.5 and 15.5; 6144 x 4096 10.4 to 12.3 against 14.6 to 17.8; 10240 x 5120 (two
    parts) 19.7 to 23.1 against 23.8 to 31.8.  From 65 to 128 rows, as two halves: 6144 x 2560 13.1 to
    15.8 us against the library's 16.3 to 19.0.  Without a cut as :func:`plan_projection`."""
    if n < TALL and rows <= FEW_ROWS:
        groups, parts = -(-n // 64), 1
        while parts < 4 and 2 * parts * groups <= units and k // (2 * parts) >= 256:
            parts *= 2
        if parts > 1:
            return Product("rows", parts, 1)
    elif n < TALL and rows <= SPLIT_ROWS:
        parts, col_tiles = rows_split(n, k, rows, units)
        if parts > 1:
            return Product("rows", parts, col_tiles)
    return plan_projection(rows, n, k)


def rows_match_library(rows: int, n: int, k: int) -> bool:
    """Whether a bfloat16 product of 17 to 48 rows that :func:`plan_projection` leaves to the library takes the
    rows kernel after all: for matrices wide enough to fill the compute units uncut, whose rows are of no
    power-of-two length, the device takes no longer (at 17, 32 and 48 rows 6144 x 2560 10.8, 11.7, 11.6 us
    against 12.6, 13.1, 15.5; 7168 x 2560 9.4, 9.9, 11.9 against 11.3, 11.8, 15.8; 10240 x 5120 19, 21, 28
    against 24, 25, 31; rows of a power-of-two length were the slower ones when this was drawn, 6144 x 4096 is now 13.1,
    14.3, 16.1 against 14.6, 15.1, 17.2) and the host 10 us instead of 26, which is what a step of few prompt
    tokens waits for."""
    return rows <= 48 and 5120 <= n < TALL and not aliased_rows(k)


def wide_beats_library(rows: int, n: int, k: int, units: int = UNITS) -> bool:
    """Whether a product of more than 64 rows without an activation behind it goes to the engine's own
    tiled kernel (``gemm_wide``) or to the library's: a projection of up to :data:`PORTION_ROWS` rows, a longer portion's where
    :func:`portion_beats_library` has no line of its own, and whatever else :func:`ops.linear` is given.  (Out and down of more
    than 128 rows have :func:`ops.wide_parts` and come here no more; the lines of matrices at least as deep as wide were
    read off them, uncut and in the tiles of then, and hold for other products of such sizes.)  The own kernel's tile is chosen so
    that the launch fills whole rounds of the compute units; for many rows the library's 256 x 256 tile is the faster main loop where
    a matrix is wide enough for it.  A layer of a prompt step in us, library against own kernel (both with
    gate/up in the own kernel's epilogue):

    out and down: 4B sizes (2560 wide) at 160, 800, 1024, 1300, 2048 tokens 195, 328, 352, 404, 567 against
    175, 315, 364, 386, 570; 8B (4096) at 160, 600, 1300, 1600, 2048 270, 401, 628, 828, 794 against 237, 410,
    610, 692, 781; 32B (5120) at 160, 600, 1300, 1600, 1800, 2048 529, 868, 1456, 1927, 1707, 1829 against 422,
    814, 1333, 1681, 1691, 2164.
    q/k/v (6144 wide; 32B 10240): 4B at 100, 250, 1300, 1800, 2048 175, 195, 404, 516, 567 against 158, 187, 395,
    530, 569; 8B at 160, 1024, 1800, 2048 270, 502, 746, 794 against 265, 502, 759, 809; 32B at 2048 1829 against
    1902.
    A matrix at least as deep as wide has few tiles, and between one 64 x 64 tile a unit and a few of them the
    own kernel, uncut, leaves units waiting: out and down of 4B at 384, 450, 512, 700 tokens 211,
    231, 234, 280 against 206, 245, 270, 297; of 8B at 260, 384, 512, 640, 700 287, 310, 345, 408, 432 against 310,
    352, 365, 429, 438; of 32B at 260, 384, 450, 700 563, 609, 767, 927 against 584, 655, 693, 845.
    Full portions of a narrow matrix: one round of 128 x 192 tiles that leaves units idle, where the library has a
    tile that suits 2048 rows, and none for the few that decode beside them (us that a layer takes longer with the
    library, out and down of 4B at 1500, 1700, 1800, 1900, 2000, 2048, 2049, 2056, 2112 tokens 2, 6, 2, -8, -9, -15, 10,
    9, 7; of 8B, at 4096 columns, 6 to 20 from 1900 on).

    The lines are read off whole steps of those widths and of 1024, 2048 and 1024 by 12288; near them either side is
    the faster one by up to 2 % of a layer.  Whole steps, because up to about 350 tokens a step waits for the host,
    to which the library's call costs 26 us and this one 10: on the device alone the own kernel, which does not cut
    K, is the slower one for few rows of a deep matrix (160 rows of 2560 x 9728 58 us against 43, of 512 x 12288 62
    against 26), in a step it is not (1024 wide models at 129 to 700 tokens 25 to 29 us a layer less, 4B at 200 to 330
    10)."""
    tiles = -(-rows // 64) * -(-n // 64)
    if k >= n and units < tiles <= (704 if n <= 4096 else 480):
        return False
    if 1850 < rows <= 2048 and n < 3072:
        return False
    if n >= 40960 and not wide_gated_beats_library(rows, n // 2):  # a gate/up matrix on its way to the library
        return False
    return rows <= 1700 or n <= 4096


PORTION_ROWS = 512  # a long portion has more rows


def library_fills_rounds(rows: int, n: int, k: int, units: int = UNITS) -> bool:
    """Whether an uncut product without an activation is the library's because its 256 x 256 tiles are those that fill the
    rounds: of one round more than three quarters, and tiles of 192 rows or of 192 columns do not fit it, of several
    more than five sixths.  Where rows of w are of a multiple of 8 KB its main loop is then the quicker one, us here and there:
    8192 x 4096 at 1538, 1700, 2048 rows 92 and 82, 99 and 89, 103 and 94; 12288 x 4096 at 1100, 1280, 2049 99 and 92, 100 and
    93, 177 and 167; 16384 x 4096 at 1600, 2048 183 and 174, 208 and 187; 7168 x 4096 at 1792 91 and 81; 8192 x 8192 at 2033
    196 and 175; where smaller tiles fit, the own kernel is: 7168 x 4096 at 1700 (192 x 256) 77 and 79, 10240 x 4096 at 1134
    76 and 77, 12288 x 4096 at 2000 (three quarters of two rounds) 154 and 166.  Up to 1,024 rows it is the one or the other
    with no line between (16384 x 8192 at 972 187 and 244, 16384 x 4096 at 900 103 and 103, 20480 x 4096 at 668 102 and 94), as
    with rows of more than 16 KB (8192 x 28672 at 1792 638 and 815, at 1900 681 and 671)."""
    if rows <= 1024 or not aliased_rows(k) or k > 8192:
        return False
    tiles = -(-rows // 256) * -(-n // 256)
    rounds = -(-tiles // units)
    if rounds > 1:
        return 6 * tiles > 5 * units * rounds
    return 4 * tiles > 3 * units and min(-(-rows // 192) * -(-n // 256), -(-rows // 256) * -(-n // 192)) > units


def portion_beats_library(rows: int, n: int, k: int, units: int = UNITS) -> bool:
    """Whether a portion's projection (q/k/v and the like) of more than :data:`PORTION_ROWS` rows takes the tiled
    kernel, with its tiles of 160 and 192 columns and its whole rounds in a launch of their own; else the library has it.
    Where rows of w are of a multiple of 8 KB: unless :func:`library_fills_rounds`.  Else everywhere but where 256 x 256 tiles
    fill five sixths of their rounds and K is short: there what :func:`wide_beats_library` says.  us, here
    against the library: 6144 x 2560 at 1024, 1400 and 2048 rows 36 and 39, 45 and 55, 52 and 56, but at 2049 (216 tiles)
    61 and 59; 10560 x 2560 at 1400, 1536 (252) 65 and 71, 66 and 72; 14592 x 2560 at 900 and 2048 (228, 456) 64 and 66,
    127 and 123; 10240 x 5120 at 1024 and 2048 87 and 95, 170 and 185.  Over 934 sizes of 4,352 to 24,576 columns, K of 2,048 to
    8,192 and 513 to 4,096 rows it takes 0.6 % longer than the quicker of the two at each (1.2 with one line of five sixths
    for K below 5,120, and up to 1,700 rows none)."""
    if rows <= PORTION_ROWS or n >= TALL:
        return False
    if aliased_rows(k):
        return not library_fills_rounds(rows, n, k, units)
    tiles = -(-rows // 256) * -(-n // 256)
    full = 6 * tiles >= 5 * units * -(-tiles // units)
    return not (full and k < 5120) or wide_beats_library(rows, n, k, units)


def wide_gated_beats_library(rows: int, n_half: int) -> bool:
    """The same for gate/up, whose activation the own kernel has in its epilogue: everywhere
    but for very wide matrices where a third tile of 160 rows is begun and the library's two of 192 hold them
    (us that a layer of a prompt step takes longer with the library: 32B, 25600 wide, at 257, 289, 320, 321, 350,
    384 tokens 14, 17, 16, -18, -17, -21; 17408 wide at 289, 320, 321, 384 18, 17, 16, 15; 8B, 12288, at 330, 384 1, 3).
    Not asked by :func:`ops.linear_capped` and :func:`ops.linear_relu2`, which keep their float32 sums."""
    return not (n_half >= 20480 and 320 < rows <= 384)


@lru_cache(maxsize=4096)  # asked for every product of a step
def plan_gated(rows: int, n_half: int, k: int, row_stride: int) -> Product:
    """``silu(x gate^T) * (x up^T)`` over a fused matrix of ``2 * n_half`` rows; "library" means
    its product followed by the activation kernel (up to 64 rows its float32 result).

    Against the skinny kernel at 8 rows: 2x9728 x 2560 19.4 against 24.7 us, 2x25600 x 5120 91
    against 103, 2x17408 x 5120 63 against 73, 2x6144 x 2048 10.6 against 14.4; but 2x12288 x
    4096 42 against 39 (aliased rows; with the rows :func:`gated_row_padding` apart in memory
    35.4 against 38.7).  Small matrices stay with the skinny kernel since an earlier form of the other (2x3072 x
    1024 6.7, where the rows kernel now takes 6.0).
    Against the library and the activation kernel from 17 to 64 rows: 2x9728 x 2560 19 to 23
    against 25 to 30, 2x12288 x 4096 43 to 45 against 48 to 50 (apart 36 to 38 against 40 to 44), 2x17408 x
    5120 66 to 76 against 82 to 89, 2x25600 x 5120 92 to 94 against 94 to 106, 2x6144 x 2048 11.4 to 15.0
    against 17.2 to 18.6, 2x3072 x 1024 6.4 to 8.9 against 14.0 to 14.5.  Matrices whose up rows lie 2 GB and
    more behind their gate rows are not the rows kernel's: one view once spanned both (each half now has its own), and
    nothing of that size has been measured."""
    if rows > STREAM_ROWS:  # 2x9728 x 2560 at 65 to 128 rows: 41 to 48 us against the library's 36 to 38
        return Product("library")
    few = rows <= FEW_ROWS
    fits = (n_half + 64) * row_stride * 2 < 2 ** 31
    if fits and (not few or (not aliased_rows(row_stride) and n_half >= 4096)):
        return Product("rows", 1, 2)
    return Product("skinny") if few else Product("library")
