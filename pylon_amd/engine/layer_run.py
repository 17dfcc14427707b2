"""The layers of a step of few prompt tokens, launched a few at a time by one call.

A step of up to a few hundred prompt tokens waits for the host, which spends 12 us on every launch that the parts make
one by one.  Where all layers of a model are alike, plain (pre-normed attention with norms and rotation head by head,
gated feed-forward) and every one of their products runs on the engine's own kernels (at 4B sizes 2 to 48 and 65 to 512
tokens, 8B 2 to 16 and 65 to 512, 32B 2 to 48, 65 to 320 and 385 to 512), :func:`run_layers` gathers the
addresses of what a layer reads and has four layers at a time launched in a loop of native code
(``csrc/layer_run.hip``): the same kernels with the same arguments in the same order, so the same bits.  The device works
on them while the next four are gathered.  Anything else, a part of another type, a product that is the library's,
decoding requests in the step, a tensor that something follows, is left to the parts, from the layer on where it shows."""
from __future__ import annotations

from array import array
from functools import lru_cache
from typing import Optional, Tuple

import torch

from ..kernels import ops, plan
from ..kernels import library
from ..parts.attention import Attention
from ..parts.block import PreNormBlock
from ..parts.feed_forward import GatedFeedForward
from ..parts.norm import RMSNorm
from ..parts.position import NoPosition, RotaryPosition

# Beyond, the device takes longer than the host either way: lone steps of 28 layers at a width of 1,024, by the parts and by
# one call, 100 tokens 2,702 and 1,373 us, 300 2,762 and 2,179, 512 2,785 and 2,485, 700 2,809 and 2,677, 1,000 2,909 and 2,952; of
# 36 at 4B sizes 21 tokens 3,346 and 2,418, from 100 on (3,927 and 3,951) no difference.
MOST_TOKENS = 512
TOGETHER = 4  # layers of one call: the device waits for the first of them only, the others are gathered while it works


def alike(spec) -> bool:
    """Whether the layers that the schedule runs are plain, all the same, and run once each in order."""
    if not spec.layers or spec.streams != 1 or spec.stream_parts:
        return False
    first = layer = spec.layers[0]
    if (layer.arrangement != "pre_norm" or layer.input_conv is not None or layer.sublayer_scale or layer.depth_mix is not None
            or layer.residual_factor != 1.0 or layer.mixer.kind != "attention" or layer.feed_forward is None
            or layer.feed_forward.kind != "gated_mlp" or layer.feed_forward.bias):
        return False
    return (all(other == first for other in spec.layers[1:]) and not any(spec.embedding_again())
            and all(e.begins_pass is None for e in spec.schedule)
            and spec.resolved_schedule() == tuple((i, i, True) for i in range(len(spec.layers))))


def _projection(rows: int, n: int, k: int, stride: int, units: int) -> Optional[Tuple[int, int]]:
    """(parts, col_tiles) of :func:`ops.linear` with a bfloat16 result, for a matrix of n rows of k elements ``stride``
    apart; (0, 0) for :func:`ops.gemm_wide`; None where it takes neither."""
    if rows > plan.STREAM_ROWS:
        return (0, 0) if ops.wide_sizes_ok(rows, n, k, k, stride) and plan.wide_beats_library(rows, n, k, units=units) else None
    if k % 8 or stride % 8 or n >= plan.TALL:
        return None
    choice = plan.plan_projection(rows, n, k, stride)
    if choice.kernel == "rows":
        return 1, choice.col_tiles
    return (1, 1) if choice.kernel == "library" and plan.rows_match_library(rows, n, k) else None


def _residual(rows: int, n: int, k: int, stride: int, units: int) -> Optional[Tuple[int, int]]:
    """The same of :func:`ops.linear_for_residual`."""
    if rows <= plan.SPLIT_ROWS and k % 8 == 0 and stride % 8 == 0:
        choice = plan.plan_residual(rows, n, k, units=units)
        return (choice.parts, choice.col_tiles) if choice.kernel == "rows" else None
    return _projection(rows, n, k, stride, units) if rows > plan.STREAM_ROWS else None


def _into_residual(rows: int, n: int, k: int, stride: int, units: int) -> Optional[Tuple[int, int]]:
    """The same of :func:`ops.linear_into_residual`; (parts, -1 - tile) for :func:`ops.gemm_wide_parts`."""
    if rows > plan.SPLIT_ROWS and ops.wide_sizes_ok(rows, n, k, k, stride):
        parts, tile = ops.wide_parts(rows, n, k, units)
        if parts > 1:
            return parts, -1 - tile
        return None if plan.library_fills_rounds(rows, n, k, units=units) else (0, 0)
    return _residual(rows, n, k, stride, units)


def _gated(rows: int, n: int, k: int, stride: int) -> Optional[Tuple[int, int]]:
    """The same of :func:`ops.linear_glu`."""
    if rows > plan.STREAM_ROWS:
        return (0, 0) if ops.wide_sizes_ok(rows, n, k, k, stride, gated=True) and plan.wide_gated_beats_library(rows, n // 2) else None
    if k % 8 or stride % 8 or plan.plan_gated(rows, n // 2, k, stride).kernel != "rows":
        return None
    return 1, 1


@lru_cache(maxsize=1024)  # asked for every step of few prompt tokens
def _products(rows: int, units: int, qkv, out, gate_up, down) -> Optional[tuple]:
    """What the four products of a layer are, each matrix given as (rows, columns, row stride); None where one of them is
    not the engine's own."""
    found = (_projection(rows, *qkv, units), _into_residual(rows, *out, units), _gated(rows, *gate_up),
             _into_residual(rows, *down, units))
    return None if None in found else tuple(number for product in found for number in product)


# What the parts of a plain layer do when they are asked themselves, and what they were written to do.
_STEPS = ((PreNormBlock, "forward"), (Attention, "forward"), (GatedFeedForward, "forward"), (RMSNorm, "add_forward"),
          (RMSNorm, "weight"), (RotaryPosition, "rotary"), (NoPosition, "rotary"))
_AS_WRITTEN = tuple(getattr(kind, name) for kind, name in _STEPS)


def _as_written() -> bool:
    """Whether no class of a plain layer's parts was given another method from outside."""
    return all(getattr(kind, name) is method for (kind, name), method in zip(_STEPS, _AS_WRITTEN))


def _plain(block) -> bool:
    if type(block) is not PreNormBlock:
        return False
    mixer, ff, norm1, norm2 = block.mixer, block.feed_forward, block.mixer_norm, block.feed_forward_norm
    if not (type(mixer) is Attention and type(ff) is GatedFeedForward and type(norm1) is RMSNorm and type(norm2) is RMSNorm
            and type(mixer.position) in (RotaryPosition, NoPosition) and mixer.plain and not mixer.special):
        return False
    # a part of its own type whose step was replaced (a wrapper that watches it, say) has the step in its own attributes
    return not ("forward" in block.__dict__ or "forward" in mixer.__dict__ or "forward" in ff.__dict__
                or "add_forward" in norm1.__dict__ or "weight" in norm1.__dict__ or "add_forward" in norm2.__dict__
                or "weight" in norm2.__dict__ or "rotary" in mixer.position.__dict__)


def run_layers(model, ctx, resid: torch.Tensor) -> Optional[Tuple[torch.Tensor, torch.Tensor]]:
    """``(resid, delta)`` behind the last layer, as the blocks hand them on, or None: then nothing was launched."""
    tokens, blocks = ctx.tokens, model.blocks
    if tokens > MOST_TOKENS or ctx.decode_only or ctx.fixed_shapes or ctx.leading_singles or not resid.is_cuda:
        return None
    block = blocks[0]
    if not (_as_written() and _plain(block)):
        return None
    # the choice of the products first: it is what a step is left to the parts for, and costs least
    spec, ff = block.mixer.spec, block.feed_forward.spec
    width, ff_size, heads, kv_heads, dim = spec.hidden_size, ff.intermediate_size, spec.n_heads, spec.n_kv_heads, spec.head_dim
    qkv_size = (heads + 2 * kv_heads) * dim
    mine, theirs, units = block.mixer.params, block.feed_forward.params, ops.compute_units()
    shapes = ((qkv_size, width), (width, spec.q_size), (2 * ff_size, width), (width, ff_size))
    matrices = (mine["qkv"], mine["out"], theirs["gate_up"], theirs["down"])
    if any(m.shape != shape or m.stride(1) != 1 or m.stride(0) < shape[1] for m, shape in zip(matrices, shapes)):
        return None
    products = _products(tokens, units, *((*m.shape, m.stride(0)) for m in matrices))
    first = ctx.cache(0)
    if products is None or first.k is None or not ops.prefill_sizes_ok(heads, kv_heads, dim, first.block_table.shape[1]):
        return None
    place, bf16, f32, grad = resid.get_device(), torch.bfloat16, torch.float32, torch.is_grad_enabled()
    if (place != torch.cuda.current_device() or resid.dtype != f32 or resid.shape != (tokens, width) or not resid.is_contiguous()
            or ops._watched(resid, resid) or ff.activation not in ops.GATE_ACTS):
        return None
    page, rotary = first.page_size, block.mixer.position.rotary()
    slots, table = (first.k.shape[0], page, kv_heads, dim), first.block_table.shape
    rot_dim = rotary[1] if rotary else 0
    if slots[0] * page >= 2 ** 31 or len(table) != 2 or table[0] < ctx.rows:
        return None

    def row(*shape):  # type, shape and strides of a tensor without gaps
        strides = [1]
        for size in shape[:0:-1]:
            strides.insert(0, strides[0] * size)
        return shape, tuple(strides)

    wanted = [(bf16, shape, (m.stride(0), 1)) for m, shape in zip(matrices, shapes)]
    as_qkv, as_out, as_gate_up, as_down = wanted
    as_gain, as_head, as_turn, as_cache = (f32, *row(width)), (f32, *row(dim)), (f32, *row(rot_dim // 2)), (bf16, *row(*slots))
    as_map, as_table = (torch.int32, *row(tokens)), (torch.int32, *row(*table))
    refused = False

    def at(t, like) -> int:
        """The address of an operand, which is refused where the parts would do something else with it."""
        nonlocal refused
        if not (type(t) in ops._PLAIN_TENSORS and t.dtype == like[0] and t.shape == like[1] and t.stride() == like[2]
                and t.get_device() == place and not (grad and t.requires_grad)):
            refused = True
            return 0
        address = t.data_ptr()
        if address & 15:
            refused = True
        return address

    maps = (first.slot_map, first.block_table)  # the views of one group of pages hold the same two
    slot_map, pages, positions = at(maps[0], as_map), at(maps[1], as_table), at(ctx.positions, as_map)
    if refused:
        return None

    def operands(index: int) -> Optional[tuple]:
        """What layer ``index`` reads, in the order of csrc/layer_run.hip; None where it is none of the plain ones."""
        block, cache = blocks[index], ctx.cache(index)
        if not _plain(block) or cache.page_size != page:
            return None
        a, f, turn = block.mixer.params, block.feed_forward.params, block.mixer.position.rotary()
        if (turn is None) != (rotary is None) or turn is not None and turn[1] != rot_dim:
            return None
        if cache.slot_map is maps[0] and cache.block_table is maps[1]:
            here = slot_map, pages
        else:
            here = at(cache.slot_map, as_map), at(cache.block_table, as_table)
        found = (at(block.mixer_norm.weight(), as_gain), at(a["qkv"], as_qkv), as_qkv[2][0],
                 at(a["q_norm"], as_head) if spec.qk_norm else 0, at(a["k_norm"], as_head) if spec.qk_norm else 0,
                 0 if turn is None else at(turn[0], as_turn), at(cache.k, as_cache), at(cache.v, as_cache), *here, table[1],
                 at(a["out"], as_out), as_out[2][0], at(block.feed_forward_norm.weight(), as_gain),
                 at(f["gate_up"], as_gate_up), as_gate_up[2][0], at(f["down"], as_down), as_down[2][0])
        return None if refused else found

    step = reals = delta = None
    for start in range(0, len(blocks), TOGETHER):
        fields, count = array("q"), 0
        for index in range(start, min(start + TOGETHER, len(blocks))):
            found = operands(index)
            if found is None:
                break
            fields.extend(found)
            count += 1
        whole = start + count == min(start + TOGETHER, len(blocks))
        if not whole and start == 0:
            return None
        if step is None:
            device = resid.device
            group = heads // kv_heads
            tile_rows = ops.prefill_rows(tokens, heads, group)
            tiles = ctx.token_tiles(tile_rows // group, skip_rows=0, fold=ops.prefill_fold(kv_heads))
            # one set of intermediate results, which every layer uses again
            narrow = [torch.empty((tokens, size), dtype=bf16, device=device)
                      for size in (width, qkv_size, spec.q_size, spec.q_size, ff_size)]
            sums = [torch.empty((parts, tokens, width) if parts > 1 else (tokens, width), dtype=f32 if parts else bf16, device=device)
                    for parts in (products[2], products[6])]
            normed, projected, q, context, hidden = (t.data_ptr() for t in narrow)
            delta = sums[1]
            step = array("q", (
                tokens, width, heads, kv_heads, dim, rot_dim, page, ff_size, ops.GATE_ACTS[ff.activation],
                ops.mask_code(spec.window, spec.chunk), positions, tiles.data_ptr(), tiles.shape[0], tile_rows, resid.data_ptr(),
                normed, projected, q, context, sums[0].data_ptr(), hidden, delta.data_ptr(), *products))
            reals = array("d", (block.mixer_norm.spec.eps, block.feed_forward_norm.spec.eps, spec.qk_norm_eps, spec.scale))
        if count:
            library.call("pylon_layer_run", fields.buffer_info()[0], count, int(start > 0), step.buffer_info()[0],
                         reals.buffer_info()[0], ops._stream())
        if not whole:  # from here on the parts
            for index in range(start + count, len(blocks)):
                resid, delta = blocks[index].forward(resid, delta, ctx, ctx.cache(index), True)
            break
    return resid, delta
