"""The layers of a step of few prompt tokens, launched by one call: the bits of the parts' own launches, which steps it
takes, and that what it does not take is left to the parts."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def config(**more):
    return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_act": "silu", "num_hidden_layers": 3,
            "hidden_size": 1024, "num_attention_heads": 32, "num_key_value_heads": 8, "head_dim": 128,
            "intermediate_size": 4096, "vocab_size": 1500, "rope_theta": 1e6, "rms_norm_eps": 1e-6,
            "tie_word_embeddings": True, "max_position_embeddings": 4096, **more}


def runner_of(cfg, **options):
    from pylon_amd.config import PylonConfig
    from pylon_amd.engine import Runner

    options = {"dtype": "bfloat16", "max_batch_size": 4, "page_size": 64, "num_pages": 40, "cuda_graphs": False, **options}
    return Runner.from_random(cfg, 7, PylonConfig(**options), std=0.02, norm_jitter=0.1)


@pytest.fixture(scope="module")
def runner():
    return runner_of(config())


@pytest.fixture
def taken(monkeypatch):
    """For every step, whether one call launched its layers."""
    from pylon_amd.engine import layer_run

    seen, real = [], layer_run.run_layers

    def watch(*args):
        got = real(*args)
        seen.append(got is not None)
        return got

    monkeypatch.setattr(layer_run, "run_layers", watch)
    return seen


def serve(runner, portions):
    """Logits of steps whose entries are (request, tokens), every token's wanted, then of one token for each request."""
    from pylon_amd.engine import StepEntry

    ids = torch.arange(4096).mul(7919).remainder(1499).tolist()
    seqs, out = {}, []
    for portion in [*portions, [(r, 1) for r in sorted({r for p in portions for r, _ in p})]]:
        entries = []
        for r, count in portion:
            seq = seqs.setdefault(r, None) or runner.open(r)
            seqs[r] = seq
            entries.append(StepEntry(seq, [ids[(seq.length + i) * 3 + r] for i in range(count)], list(range(count))))
        out.append(runner.step(entries).clone())
    for seq in seqs.values():
        runner.close(seq)
    return out


# up to 16 rows, 17 to 48 and beyond 64 (the tiled kernel: bfloat16 results between the layers; up to 128 float sums),
# several requests, a second portion behind cached tokens, and the most tokens that one call takes
@pytest.mark.parametrize("portions, one_call", [
    ([[(0, 2)]], [True]), ([[(0, 16)]], [True]), ([[(0, 17)]], [True]), ([[(0, 48)]], [True]), ([[(0, 20), (1, 21)]], [True]),
    ([[(0, 65)]], [True]), ([[(0, 128)]], [True]), ([[(0, 129)], [(0, 40)]], [True, True]), ([[(0, 300), (1, 212)]], [True]),
    ([[(0, 49)]], [False]), ([[(0, 513)]], [False]), ([[(0, 1)]], [False]), ([[(0, 30)], [(0, 1), (1, 20)]], [True, False])])
def test_the_bits_of_the_parts_launches(runner, taken, portions, one_call):
    got = serve(runner, portions)
    assert taken == one_call + [False]  # and the decode step behind
    runner.model.alike, kept = False, runner.model.alike
    try:
        want = serve(runner, portions)
    finally:
        runner.model.alike = kept
    assert kept and len(got) == len(want)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_what_is_followed_or_of_another_kind_is_left_to_the_parts(runner, taken):
    from pylon_amd.parts.norm import RMSNorm

    weight = runner.model.blocks[1].mixer.params["out"]
    weight.requires_grad_(True)
    try:
        serve(runner, [[(0, 20)]])
    finally:
        weight.requires_grad_(False)

    class Other(RMSNorm):
        pass

    norm = runner.model.blocks[2].feed_forward_norm
    norm.__class__ = Other
    try:
        serve(runner, [[(0, 20)]])
    finally:
        norm.__class__ = RMSNorm
    apart = torch.empty((1024, 4096 + 64), dtype=torch.bfloat16, device="cuda:0")[:, :4096]
    old = runner.model.blocks[1].feed_forward.params["down"]
    apart.copy_(old)
    runner.model.blocks[1].feed_forward.params["down"] = apart
    try:
        serve(runner, [[(0, 20)]])
    finally:
        runner.model.blocks[1].feed_forward.params["down"] = old
    assert not any(taken)


def test_models_of_unlike_layers_and_of_32_bits_are_not_asked():
    assert not runner_of(config(), dtype="float32").model.alike
    assert runner_of(config(num_hidden_layers=1)).model.alike


def test_the_fields_that_both_sides_count():
    import ctypes

    from pylon_amd.kernels import library

    fields = (ctypes.c_int * 3)()
    library.call("pylon_layer_run_fields", ctypes.addressof(fields))
    assert tuple(fields) == (18, 30, 4)


@pytest.mark.parametrize("part, step", [("", "forward"), ("mixer", "forward"), ("feed_forward", "forward"),
                                        ("mixer_norm", "add_forward"), ("feed_forward_norm", "weight"),
                                        ("mixer.position", "rotary")])
@pytest.mark.parametrize("of_its_type", [False, True])
def test_a_replaced_step_of_a_part_is_taken(runner, taken, monkeypatch, part, step, of_its_type):
    thing = runner.model.blocks[1]
    for name in filter(None, part.split(".")):
        thing = getattr(thing, name)
    calls, real = [], getattr(thing, step)
    if of_its_type:
        method = getattr(type(thing), step)
        monkeypatch.setattr(type(thing), step, lambda self, *args, **more: (calls.append(1), method(self, *args, **more))[1])
    else:
        monkeypatch.setattr(thing, step, lambda *args, **more: (calls.append(1), real(*args, **more))[1], raising=False)
    serve(runner, [[(0, 20)]])
    assert not any(taken) and len(calls) >= 2  # in the prompt's step and the one behind it


def test_maps_and_tables_that_the_parts_refuse_are_not_launched_on(runner, monkeypatch):
    from dataclasses import replace

    from pylon_amd.engine import layer_run

    answers, real = [], layer_run.run_layers

    def watch(model, ctx, resid):
        def of_layer(i, **other):
            return replace(ctx, views={**ctx.views, i: replace(ctx.views[i], **other)})

        view = ctx.views[2]
        if not ctx.decode_only:
            for broken in (replace(ctx, positions=ctx.positions.long()), replace(ctx, positions=ctx.positions[:-1]),
                           of_layer(2, slot_map=view.slot_map.long()), of_layer(2, slot_map=view.slot_map[:-1]),
                           of_layer(2, slot_map=view.slot_map.repeat_interleave(2)[::2]), of_layer(2, slot_map=None),
                           of_layer(2, block_table=view.block_table.long()), of_layer(2, block_table=view.block_table[:0]),
                           of_layer(2, block_table=view.block_table.cpu())):
                answers.append(real(model, broken, resid))
        return real(model, ctx, resid)

    monkeypatch.setattr(layer_run, "run_layers", watch)
    serve(runner, [[(0, 20)]])
    assert answers == [None] * 9


def runner_of_layers(monkeypatch, cfg, change, **options):
    """A runner whose layers are ``change(layer)`` of the plain ones."""
    from dataclasses import replace

    from pylon_amd.engine import runner as engine

    def resolve(config, real=engine.resolve):
        arch = real(config)

        def spec(parsed):
            plain = arch.model_spec(parsed)
            return replace(plain, layers=tuple(map(change, plain.layers)))

        return replace(arch, model_spec=spec)

    monkeypatch.setattr(engine, "resolve", resolve)
    return runner_of(cfg, **options)


# other layers than those above: a window, the other gate, no rotation, other widths and heads, a deep product over gemm_wide
@pytest.mark.parametrize("mixer, ff, sizes", [
    (dict(window=24), {}, {}), ({}, dict(activation="gelu_tanh"), {}), (dict(position="none"), {}, {}),
    (dict(window=100), dict(activation="gelu_tanh"), dict(hidden_size=2560, intermediate_size=1536)),
    ({}, {}, dict(hidden_size=512, num_attention_heads=24, num_key_value_heads=3, head_dim=64, intermediate_size=5120))])
def test_the_bits_of_other_layers(monkeypatch, taken, mixer, ff, sizes):
    from dataclasses import replace

    def change(layer):
        more = dict(mixer)
        if "position" in more:
            more["position"] = replace(layer.mixer.position, kind="none")
        return replace(layer, mixer=replace(layer.mixer, **more), feed_forward=replace(layer.feed_forward, **ff))

    runner = runner_of_layers(monkeypatch, config(**sizes), change)
    portions = [[(0, 12)], [(0, 70)], [(0, 30), (1, 40)], [(2, 200), (1, 111)]]
    got = serve(runner, portions)
    steps = list(taken)
    runner.model.alike = False
    assert any(steps) and all(torch.equal(a, b) for a, b in zip(got, serve(runner, portions), strict=True))


def test_the_first_layers_are_launched_before_the_last_are_looked_at(monkeypatch):
    from pylon_amd.engine import layer_run

    runner = runner_of(config(num_hidden_layers=9))
    events, plain, call = [], layer_run._plain, layer_run.library.call
    monkeypatch.setattr(layer_run, "_plain", lambda block: (events.append("layer"), plain(block))[1])
    monkeypatch.setattr(layer_run.library, "call", lambda name, *args: (
        name == "pylon_layer_run" and events.append(args[1]), call(name, *args))[1])
    serve(runner, [[(0, 20)]])
    assert events == ["layer"] * 5 + [4] + ["layer"] * 4 + [4, "layer", 1]


# a layer that only the parts run, where none was launched yet, inside a call's layers and as the first of a call's; sums in
# float parts and a bfloat16 result on their way between the two
@pytest.mark.parametrize("at", [3, 4, 6, 8])
@pytest.mark.parametrize("tokens", [20, 140])
def test_the_parts_go_on_where_a_layer_is_theirs(monkeypatch, taken, at, tokens):
    runner = runner_of(config(num_hidden_layers=9))
    want = serve(runner, [[(0, tokens)]])
    block, calls = runner.model.blocks[at], []
    monkeypatch.setattr(block, "forward", lambda *args, real=block.forward: (calls.append(1), real(*args))[1], raising=False)
    got = serve(runner, [[(0, tokens)]])
    assert taken == [True, False, at > 3, False] and len(calls) == 2
    assert all(torch.equal(a, b) for a, b in zip(got, want, strict=True))


def test_a_step_that_is_left_to_the_parts_allocates_nothing_for_the_question(runner, monkeypatch):
    from pylon_amd.engine import layer_run

    count, real, asked = (lambda: torch.cuda.memory_stats()["allocation.all.allocated"]), layer_run.run_layers, []

    def watch(*args):
        before = count()
        asked.append((real(*args) is None, count() - before))
        return None

    monkeypatch.setattr(layer_run, "run_layers", watch)
    serve(runner, [[(0, 49)], [(1, 600)]])
    assert asked == [(True, 0)] * 3
