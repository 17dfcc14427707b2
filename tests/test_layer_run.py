"""Which models have layers that one call may launch, and that their products are those the parts launch."""
import warnings
from dataclasses import replace

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from pylon_amd.config.registry import resolve
from pylon_amd.engine import layer_run
from pylon_amd.engine.layer_run import alike
from pylon_amd.kernels import ops, plan

CONFIG = {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_act": "silu", "num_hidden_layers": 3,
          "hidden_size": 128, "num_attention_heads": 2, "num_key_value_heads": 1, "head_dim": 64, "intermediate_size": 256,
          "vocab_size": 100, "rope_theta": 1e6, "rms_norm_eps": 1e-6, "tie_word_embeddings": True, "max_position_embeddings": 512}


def spec():
    arch = resolve(CONFIG)
    return arch.model_spec(arch.parse_config(CONFIG))


def with_layer(plain, index, **more):
    layers = list(plain.layers)
    layers[index] = replace(layers[index], **more)
    return replace(plain, layers=tuple(layers))


def test_plain_layers_that_are_all_the_same_are():
    assert alike(spec()) and alike(replace(spec(), layers=spec().layers[:1], schedule=spec().schedule[:1]))


@pytest.mark.parametrize("change", [
    lambda s: with_layer(s, 1, mixer=replace(s.layers[1].mixer, window=40)),
    lambda s: with_layer(s, 2, feed_forward=replace(s.layers[2].feed_forward, activation="gelu_tanh")),
    lambda s: with_layer(s, 2, mixer_norm=replace(s.layers[2].mixer_norm, eps=1e-5)),
    lambda s: replace(s, layers=tuple(replace(layer, residual_factor=0.5) for layer in s.layers)),
    lambda s: replace(s, layers=tuple(replace(layer, sublayer_scale=True) for layer in s.layers)),
    lambda s: replace(s, schedule=s.schedule + s.schedule[:1]),
    lambda s: replace(s, schedule=s.schedule[::-1]),
    lambda s: replace(s, schedule=s.schedule[:2]),
    lambda s: replace(s, streams=2)])
def test_others_are_not(change):
    assert not alike(change(spec()))


def test_a_layer_that_borrows_a_cache_is_not():
    plain = spec()
    assert not alike(replace(plain, schedule=(*plain.schedule[:2], replace(plain.schedule[2], cache=1))))


def test_portions_by_other_rules_are_left_to_the_parts():
    assert layer_run.MOST_TOKENS <= plan.PORTION_ROWS  # beyond, projections have a rule of their own
    assert layer_run._into_residual(2048, 8192, 8192, 8192, 256) is None  # the library's
    assert layer_run._into_residual(2049, 8192, 8192, 8192, 256) == (0, 0)


# (q/k/v, context, width, feed-forward): 4B, 8B and 32B sizes, narrow layers, a narrow and deep one, one whose rows are of no
# multiple of 64; with the matrices' rows apart as well
@pytest.mark.parametrize("qkv, context, width, ff", [
    (6144, 4096, 2560, 9728), (6144, 4096, 4096, 12288), (10240, 8192, 5120, 25600), (3072, 1024, 1024, 3072),
    (1920, 1536, 512, 5120), (5120, 2048, 2056, 4104)])
@pytest.mark.parametrize("apart", [0, 64])
def test_the_products_are_those_of_their_entry_points(monkeypatch, qkv, context, width, ff, apart):
    """Where a step's layers are launched by one call, (ranges of K, column tiles) of every product, (ranges, -1 less the
    tile) for ranges of the tiled kernel, (0, 0) for it uncut, are what the entry point that the part calls launches."""
    launched, bf16 = [], torch.bfloat16
    monkeypatch.setattr(ops, "_raw_device", lambda: 0)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_watched", lambda x, weight: False)
    monkeypatch.setattr(ops, "_dev", lambda t, name, dtype=None: 0)
    monkeypatch.setattr(ops._lib, "compute_units", lambda: 256)
    plan_of = ops._lib.call

    def call(name, *args):
        if name == "pylon_gemm_wide_parts_plan":  # on the host
            return plan_of(name, *args)
        launched.append((args[10], args[12]) if name == "pylon_gemm_rows" else (0, 0) if name == "pylon_gemm_wide"
                        else (args[8], -1 - args[9]) if name == "pylon_gemm_wide_parts" else None)

    monkeypatch.setattr(ops._lib, "call", call)
    monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w: launched.append(None) or x.new_empty(x.shape[0], w.shape[0]))
    monkeypatch.setattr(ops, "_library_float", lambda x, w, out=None: launched.append(None) or x.new_empty(
        x.shape[0], w.shape[0], dtype=torch.float32))
    taken = set()
    with FakeTensorMode(), warnings.catch_warnings():
        warnings.simplefilter("ignore")  # data pointers of tensors without data

        def choice(entry, rows, n, k, **more):
            x = torch.empty(rows, k, dtype=bf16, device="cuda:0")
            launched.clear()
            entry(x, torch.empty(n, k + apart, dtype=bf16, device="cuda:0")[:, :k], **more)
            return launched[0]

        for rows in (1, 2, 16, 17, 31, 32, 33, 48, 49, 64, 65, 100, 128, 129, 192, 193, 256, 300, 384, 385, 511, 512):
            asked = (layer_run._projection(rows, qkv, width, width + apart, 256),
                     layer_run._into_residual(rows, width, context, context + apart, 256),
                     layer_run._gated(rows, 2 * ff, width, width + apart),
                     layer_run._into_residual(rows, width, ff, ff + apart, 256))
            made = (choice(ops.linear_of_portion, rows, qkv, width, out_dtype=bf16),
                    choice(ops.linear_into_residual, rows, width, context, out_dtype=bf16),
                    choice(ops.linear_glu, rows, 2 * ff, width, out_dtype=bf16),
                    choice(ops.linear_into_residual, rows, width, ff, out_dtype=bf16))
            for name, mine, theirs in zip(("qkv", "out", "gate/up", "down"), asked, made):
                assert mine == theirs, (rows, name)  # None: the library's, or the skinny kernel's
                taken.add(None if mine is None else (mine[0] > 0) + (mine[1] < 0))
    assert taken >= {1, 2}  # ranges of the rows kernel and of the tiled one
