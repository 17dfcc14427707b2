"""Which models have layers that one call may launch."""
from dataclasses import replace

import pytest

from pylon_amd.config.registry import resolve
from pylon_amd.engine.layer_run import alike

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
