"""The layers of a step of few prompt tokens, launched by one call.

A step of up to a few hundred prompt tokens waits for the host, which spends 12 us on every launch that the parts make
one by one.  Where all layers of a model are alike, plain (pre-normed attention with norms and rotation head by head,
gated feed-forward) and every one of their products runs on the engine's own kernels, :func:`run_layers` gathers the
addresses of what a layer reads and has them launched in a loop of native code (``csrc/layer_run.hip``): the same
kernels with the same arguments in the same order, so the same bits.  Anything else, a part of another type, a product
that is the library's, decoding requests in the step, a tensor that something follows, is left to the parts."""
from __future__ import annotations

import ctypes
from array import array
from typing import Optional, Tuple

import torch

from ..kernels import ops, plan
from ..kernels import library
from ..parts.attention import Attention
from ..parts.block import PreNormBlock
from ..parts.feed_forward import GatedFeedForward
from ..parts.norm import RMSNorm
from ..parts.position import NoPosition, RotaryPosition

MOST_TOKENS = 512  # beyond, the device takes longer than the host either way


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


def _streams(weight: torch.Tensor) -> bool:
    """What :func:`ops.gemm_rows` asks of a matrix (``x`` is made here: close rows, aligned)."""
    return weight.shape[1] % 8 == 0 and weight.stride(0) % 8 == 0 and weight.data_ptr() % 16 == 0 and weight.stride(1) == 1


def _wide(x: torch.Tensor, weight: torch.Tensor, gated: bool = False) -> Optional[Tuple[int, int]]:
    return (0, 0) if ops._wide_ok(x, weight, gated=gated) else None


def _projection(x, weight, units) -> Optional[Tuple[int, int]]:
    """(parts, col_tiles) of :func:`ops.linear` with a bfloat16 result, (0, 0) for :func:`ops.gemm_wide`; None where it
    takes neither."""
    rows, (n, k) = x.shape[0], weight.shape
    if rows <= plan.STREAM_ROWS:
        if not _streams(weight) or n >= plan.TALL:
            return None
        choice = plan.plan_projection(rows, n, k, weight.stride(0))
        if choice.kernel == "rows":
            return 1, choice.col_tiles
        return (1, 1) if choice.kernel == "library" and plan.rows_match_library(rows, n, k) else None
    return _wide(x, weight) if plan.wide_beats_library(rows, n, k, units=units) else None


def _residual(x, weight, units) -> Optional[Tuple[int, int]]:
    """The same of :func:`ops.linear_for_residual`."""
    rows, (n, k) = x.shape[0], weight.shape
    if rows <= plan.SPLIT_ROWS and _streams(weight):
        choice = plan.plan_residual(rows, n, k, units=units)
        return (choice.parts, choice.col_tiles) if choice.kernel == "rows" else None
    return _projection(x, weight, units) if rows > plan.STREAM_ROWS else None


def _gated(x, weight) -> Optional[Tuple[int, int]]:
    """The same of :func:`ops.linear_glu`."""
    rows, n_half = x.shape[0], weight.shape[0] // 2
    if rows > plan.STREAM_ROWS:
        return _wide(x, weight, gated=True) if plan.wide_gated_beats_library(rows, n_half) else None
    if not _streams(weight) or plan.plan_gated(rows, n_half, weight.shape[1], weight.stride(0)).kernel != "rows":
        return None
    return 1, 1


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
    tokens = ctx.tokens
    if tokens > MOST_TOKENS or ctx.decode_only or ctx.fixed_shapes or ctx.leading_singles or not resid.is_cuda:
        return None
    if resid.dtype != torch.float32 or resid.dim() != 2 or not resid.is_contiguous():
        return None
    block = model.blocks[0]
    if not (_as_written() and all(map(_plain, model.blocks))):
        return None
    spec, ff = block.mixer.spec, block.feed_forward.spec
    width, qkv_size = spec.hidden_size, (spec.n_heads + 2 * spec.n_kv_heads) * spec.head_dim
    first = ctx.cache(0)
    rotary = block.mixer.position.rotary()
    if first.k is None or first.k.dim() != 4 or ops._watched(resid, resid):
        return None
    device, bf16, f32 = resid.device, torch.bfloat16, torch.float32
    place = resid.get_device()
    if place != torch.cuda.current_device():
        return None

    def scratch(*shape, dtype=bf16):
        return torch.empty(shape, dtype=dtype, device=device)

    normed, projected = scratch(tokens, width), scratch(tokens, qkv_size)
    q, context = scratch(tokens, spec.n_heads, spec.head_dim), scratch(tokens, spec.n_heads, spec.head_dim)
    hidden = scratch(tokens, ff.intermediate_size)
    if not ops.prefill_attention_ok(q, first.k, first.block_table) or ff.activation not in ops.GATE_ACTS:
        return None
    units = ops.compute_units()
    mine, theirs = block.mixer.params, block.feed_forward.params
    products = (_projection(normed, mine["qkv"], units), _residual(context.view(tokens, spec.q_size), mine["out"], units),
                _gated(normed, theirs["gate_up"]), _residual(hidden, theirs["down"], units))
    if None in products:
        return None

    def good(t, dtype, shape) -> bool:
        return (t.dtype == dtype and t.shape == shape and t.get_device() == place and t.is_contiguous()
                and not ops._watched(t, t))

    def matrix(t, like) -> bool:
        return (t.dtype == bf16 and t.shape == like.shape and t.stride() == like.stride() and t.stride(1) == 1
                and t.get_device() == place and t.data_ptr() % 16 == 0 and not ops._watched(t, t))

    def ints(t, numel) -> bool:
        return t is not None and t.dtype == torch.int32 and t.get_device() == place and t.is_contiguous() and t.numel() == numel

    views = [ctx.cache(index) for index in range(len(model.blocks))]
    maps, tables = ({id(t): t for t in found}.values() for found in ([v.slot_map for v in views], [v.block_table for v in views]))
    if not (resid.shape == (tokens, width) and ints(ctx.positions, tokens) and all(ints(m, tokens) for m in maps)
            and all(t is not None and t.dim() == 2 and t.shape[0] >= ctx.rows and ints(t, t.numel()) for t in tables)):
        return None  # what the parts refuse (the views of one group of pages hold the same map and table)
    shapes = dict(qkv=(qkv_size, width), out=(width, spec.q_size), gate_up=(2 * ff.intermediate_size, width),
                  down=(width, ff.intermediate_size))
    if any(tuple(p[name].shape) != shapes[name] for p, name in ((mine, "qkv"), (mine, "out"), (theirs, "gate_up"), (theirs, "down"))):
        return None
    fields = array("q")
    for index, block in enumerate(model.blocks):
        a, f, cache = block.mixer.params, block.feed_forward.params, ctx.cache(index)
        gain1, gain2, q_norm, k_norm = block.mixer_norm.weight(), block.feed_forward_norm.weight(), a.get("q_norm"), a.get("k_norm")
        turn = block.mixer.position.rotary()
        if not (matrix(a["qkv"], mine["qkv"]) and matrix(a["out"], mine["out"]) and matrix(f["gate_up"], theirs["gate_up"])
                and matrix(f["down"], theirs["down"]) and good(gain1, f32, (width,)) and good(gain2, f32, (width,))
                and good(cache.k, bf16, first.k.shape) and good(cache.v, bf16, first.k.shape)
                and cache.page_size == cache.k.shape[1] == first.page_size and cache.block_table.shape == first.block_table.shape
                and (turn is None) == (rotary is None) and (turn is None or turn[1] == rotary[1] and good(turn[0], f32, (turn[1] // 2,)))):
            return None
        if spec.qk_norm and not (good(q_norm, f32, (spec.head_dim,)) and good(k_norm, f32, (spec.head_dim,))):
            return None
        fields.extend((gain1.data_ptr(), a["qkv"].data_ptr(), a["qkv"].stride(0),
                       q_norm.data_ptr() if spec.qk_norm else 0, k_norm.data_ptr() if spec.qk_norm else 0,
                       0 if turn is None else turn[0].data_ptr(), cache.k.data_ptr(), cache.v.data_ptr(),
                       cache.slot_map.data_ptr(), cache.block_table.data_ptr(), cache.block_table.shape[1],
                       a["out"].data_ptr(), a["out"].stride(0), gain2.data_ptr(), f["gate_up"].data_ptr(),
                       f["gate_up"].stride(0), f["down"].data_ptr(), f["down"].stride(0)))
    if first.k.shape[0] * first.page_size >= 2 ** 31 or first.k.shape[2:] != (spec.n_kv_heads, spec.head_dim):
        return None
    group = spec.n_heads // spec.n_kv_heads
    tile_rows = ops.prefill_rows(tokens, spec.n_heads, group)
    tiles = ctx.token_tiles(tile_rows // group, skip_rows=0, fold=ops.prefill_fold(spec.n_kv_heads))

    def sums(parts):
        return scratch(parts, tokens, width, dtype=f32) if parts > 1 else scratch(tokens, width, dtype=f32 if parts else bf16)

    out_sum, down_sum = sums(products[1][0]), sums(products[3][0])
    step = array("q", (
        tokens, width, spec.n_heads, spec.n_kv_heads, spec.head_dim, rotary[1] if rotary else 0, first.page_size,
        ff.intermediate_size, ops.GATE_ACTS[ff.activation], ops.mask_code(spec.window, spec.chunk), ctx.positions.data_ptr(),
        tiles.data_ptr(), tiles.shape[0], tile_rows, resid.data_ptr(), normed.data_ptr(), projected.data_ptr(), q.data_ptr(),
        context.data_ptr(), out_sum.data_ptr(), hidden.data_ptr(), down_sum.data_ptr(),
        *(number for product in products for number in product)))
    reals = array("d", (block.mixer_norm.spec.eps, block.feed_forward_norm.spec.eps, spec.qk_norm_eps, spec.scale))
    library.call("pylon_layer_run", fields.buffer_info()[0], len(model.blocks), step.buffer_info()[0], reals.buffer_info()[0],
                 ops._stream())
    return resid, down_sum
