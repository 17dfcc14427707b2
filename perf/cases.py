"""What this engine is timed on: requests served through ``Runner.step``, from their prompts to their
last token.

A case is a model (design, layer sizes, number of layers, element type, weights drawn from the seed) and a
batch of requests: ``requests`` prompts of up to ``prompt`` tokens (all of that length, or, ``ragged``,
spread between half of it and all of it), each followed by ``new`` tokens.  One pass serves them as the
engine's scheduler does: every step brings up to 2,048 prompt tokens, beside one token for each request
whose prompt is through; once all prompts are through, a step is one token for every request, replayed
from a graph.  The tokens that follow a prompt are given with the prompts, so that a tie between two
logits cannot send two correct implementations down different texts.  The outputs are the float32 logits
after every prompt and after every further token.

The designs are the dense ones of this repository.  Models with a mixture of experts are left out for one
reason: with weights that nobody trained, the choice of a token's experts hangs on near ties that rounding
decides, and two correct implementations then differ by a whole expert.

Sizes are the layer sizes of ``bench.py`` (Qwen3 4B, 8B and 32B; the other designs at the 4B and 8B
sizes).  A whole model repeats the same layers, and the rounding of 36 of them adds up to what another order
of sums could no longer be told from (2.9e-2 of the logits), so there are 12 layers at most; of Ranudra,
whose copies of the stream untrained coefficients take differences of, 4 (0.6e-2; 8 layers: 5e-2 and more).
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from pylon_amd.config import PylonConfig
from pylon_amd.config.registry import resolve
from pylon_amd.engine import Runner, StepEntry

PORTION = 2048  # prompt tokens of one step
PAGE = 256
VOCAB = 151936

SHAPES = {  # width, heads, key/value heads, head size, feed-forward, layers, head tied to the embedding, rotary base
    "4b": (2560, 32, 8, 128, 9728, 36, True, 5000000.0),
    "8b": (4096, 32, 8, 128, 12288, 36, False, 1000000.0),
    "32b": (5120, 64, 8, 128, 25600, 64, False, 1000000.0),
}
MOST_TOKENS = 8192  # tokens of one drawn case


def listed():
    def case(name, design, shape, layers, requests, prompt, new, ragged=False, dtype="bfloat16"):
        return {"name": name, "design": design, "shape": shape, "layers": layers, "dtype": dtype,
                "requests": requests, "prompt": prompt, "new": new, "ragged": ragged}

    return [
        # the smallest call: the first token of a one-line question
        case("first-token", "qwen3", "4b", 12, 1, 21, 0),
        # one user's chat: a short prompt and an answer at batch 1
        case("chat-1", "qwen3", "4b", 12, 1, 64, 64),
        # the headline workload of bench.py: eight requests of 128 tokens and their answers
        case("chat-8", "qwen3", "4b", 12, 8, 128, 64),
        # a full server: 48 requests of uneven prompts, a step of 48 tokens each time
        case("chat-48-ragged", "qwen3", "8b", 8, 48, 150, 24, ragged=True),
        # a prompt of exactly one portion: time to the first token
        case("prompt-2048", "qwen3", "4b", 8, 1, 2048, 0),
        # a few uneven prompts that meet in one step, larger layers: mid-sized products
        case("prompts-ragged-32b", "qwen3", "32b", 4, 5, 170, 4, ragged=True),
        # a document near the context's end: prompt in portions over a growing cache, then an answer
        case("document-8000", "qwen3", "4b", 12, 1, 8000, 32),
        # several long prompts: decoding requests beside portions, then decoding over long caches
        case("long-4", "qwen3", "8b", 8, 4, 3000, 16, ragged=True),
        # the true 32-bit path, as the replay of traces uses it
        case("float32", "qwen3", "4b", 6, 3, 120, 6, ragged=True, dtype="float32"),
        # retention beside attention with a sink and a bias by distance, short convolutions
        case("vupuzen", "vupuzen", "4b", 8, 4, 1500, 24, ragged=True),
        # gated linear attention beside latent attention, two copies of the stream
        case("ranudra", "ranudra", "4b", 4, 6, 900, 24, ragged=True),
        # lightning attention beside windowed attention with a sink, layers run twice
        case("farorax", "farorax", "8b", 8, 2, 2500, 24, ragged=True),
    ]


def draw(rng: random.Random):
    def spread(low, high):  # over the logarithm
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    design = rng.choice(["qwen3"] * 5 + ["vupuzen", "ranudra", "farorax"])
    dtype = "float32" if design == "qwen3" and rng.random() < 0.15 else "bfloat16"
    shape = rng.choice(["4b", "8b"] if design != "qwen3" or dtype == "float32" else ["4b", "4b", "8b", "32b"])
    few = shape == "32b" or dtype == "float32" or design == "ranudra"
    layers = rng.randint(2, 4) if few else rng.randint(3, 8)
    if dtype == "float32":
        requests, prompt, new = spread(1, 6), spread(3, 300), rng.randint(0, 8)
    else:
        requests = spread(1, 64)
        prompt = spread(5, max(5, min(8000, MOST_TOKENS // requests)))
        new = rng.choice([0, rng.randint(1, 32)])
    return {"design": design, "shape": shape, "layers": layers, "dtype": dtype, "requests": requests,
            "prompt": prompt, "new": new, "ragged": rng.random() < 0.7}


# ---- the models' configurations ---------------------------------------------------------------


def config_of(case):
    width, heads, kv_heads, dim, ff, _, tied, theta = SHAPES[case["shape"]]
    layers = case["layers"]
    attention = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": dim}
    again = layers // 4  # this many layers run twice, where a design has loops
    own = layers - again
    start = (own - again) // 2
    loop = {"start": start, "stop": start + again, "times": 2} if again else None
    state_heads = max(1, width // (2 * dim))  # heads of the mixers that keep a state
    if case["design"] == "qwen3":
        return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_act": "silu",
                "num_hidden_layers": layers, "hidden_size": width, "num_attention_heads": heads,
                "num_key_value_heads": kv_heads, "head_dim": dim, "intermediate_size": ff, "vocab_size": VOCAB,
                "rope_theta": theta, "rms_norm_eps": 1e-6, "tie_word_embeddings": tied, "max_position_embeddings": 8192}
    if case["design"] == "vupuzen":
        mlp = {"kind": "dense", "ff": ff, "limit": 7.0}
        softmax = {"type": "attention", "mlp": mlp, "mixer": {**attention, "scale": dim ** -0.5, "bias_max": 2048}}
        decay = [1.0 - 2.0 ** (-5 - 3 * h / max(1, state_heads - 1)) for h in range(state_heads)]
        retention = {"type": "retention", "mlp": mlp, "mixer": {
            "heads": state_heads, "dim": dim, "vdim": dim, "decay": decay, "rot": {"dims": dim, "base": 1000000.0}}}
        return {"architecture": "Vupuzen", "vocab": VOCAB, "width": width, "canon": {"taps": 4}, "norm": {"eps": 1e-6},
                "logit_scale": 1.0, "layers": [retention if i % 4 == 0 else softmax for i in range(layers)]}
    if case["design"] == "ranudra":
        mlp = {"kind": "dense", "ff": ff * 3 // 2}
        sizes = {"heads": heads, "dim": dim, "rot_dim": 64, "vdim": dim, "kv_rank": 256, "scale": (dim + 64) ** -0.5,
                 "mask": {"size": 1024}}
        kinds = [{"type": "gla", "mlp": mlp, "mixer": {"heads": state_heads, "dim": dim, "vdim": dim, "tau": 12.0}},
                 {"type": "latent_attention", "mlp": mlp, "mixer": {**sizes, "rot": {
                     "base": 500000.0, "dims": 64,
                     "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}},
                 {"type": "latent_attention_2", "mlp": mlp,
                  "mixer": {**sizes, "rot": {"base": 100000.0, "dims": 64}}}]
        return {"architecture": "Ranudra", "vocab": VOCAB, "width": width, "streams": 2, "embedding": {"scale": 12.0},
                "norm": {"eps": 1e-6}, "loop": loop, "layers": [kinds[i % 3] for i in range(own)]}
    if case["design"] == "farorax":
        mlp = {"kind": "dense", "ff": ff}
        decay = [1.0 - 2.0 ** (-1 - 8 * h / max(1, state_heads - 1)) for h in range(state_heads)]
        kinds = [{"type": "lightning", "mlp": mlp,
                  "mixer": {"heads": state_heads, "dim": dim, "vdim": dim, "decay": decay}},
                 {"type": "attention", "mlp": mlp, "mixer": {
                     **attention, "scale": dim ** -0.5, "mask": {"size": 1024},
                     "rot": {"base": 500000.0, "dims": dim,
                             "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}}]
        return {"architecture": "Farorax", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-6}, "residual_mult": 0.25,
                "logit_softcap": 40.0, "loop": loop, "layers": [kinds[i % 2] for i in range(own)]}
    raise ValueError(case["design"])


def runs_of(config):
    """(layer, number of the pass that begins right before it, or None) in running order."""
    count, loop = len(config["layers"]), config.get("loop")
    if not loop:
        return [(i, None) for i in range(count)]
    runs = [(i, None) for i in range(loop["start"])]
    for t in range(loop["times"]):
        runs += [(i, t if i == loop["start"] else None) for i in range(loop["start"], loop["stop"])]
    return runs + [(i, None) for i in range(loop["stop"], count)]


# ---- the requests -----------------------------------------------------------------------------


def lengths_of(case):
    """Tokens of every request's prompt."""
    n, most = case["requests"], case["prompt"]
    if not case["ragged"] or n == 1:
        return [most] * n
    least = (most + 1) // 2
    return [least + (most - least) * ((7 * i + 3) % n) // (n - 1) for i in range(n)]


def steps_of(case):
    """The steps of a pass: each a list of (request, first token, tokens, whether its logits are wanted)."""
    prompts, new = lengths_of(case), case["new"]
    done, fed, steps = [0] * len(prompts), [0] * len(prompts), []
    while True:
        through = [d == p for d, p in zip(done, prompts)]
        if all(through) and min(fed) >= new:
            return steps
        step, room = [], PORTION
        for r, ready in enumerate(through):
            # a request that was through early goes on until the last one has its tokens
            if ready and new:
                step.append((r, prompts[r] + fed[r], 1, True))
        for r, ready in enumerate(through):
            count = min(room, prompts[r] - done[r])
            if count:
                step.append((r, done[r], count, done[r] + count == prompts[r]))
                done[r] += count
                room -= count
        for r, first, _, _ in step:
            if first >= prompts[r]:
                fed[r] += 1
        steps.append(step)


def texts_of(case, seed):
    """Token ids of every request: its prompt and what follows it."""
    rng = np.random.default_rng(seed)
    ends = [0] * case["requests"]
    for step in steps_of(case):
        for r, first, count, _ in step:
            ends[r] = max(ends[r], first + count)
    return [rng.integers(0, VOCAB, n) for n in ends]


def prepare(case, seed):
    steps, texts = steps_of(case), texts_of(case, seed)
    pages = sum(len(t) // PAGE + 1 for t in texts) + 1
    options = PylonConfig(dtype=case["dtype"], max_batch_size=case["requests"], max_queue_size=case["requests"],
                          page_size=PAGE, prefill_chunk_size=PORTION, num_pages=pages, cuda_graphs=False)
    runner = Runner.from_random(config_of(case), seed, options, std=0.02, norm_jitter=0.1)
    if case["new"]:
        # as start-up does: the largest decode step once kernel by kernel, then its graph
        seqs = [runner.open(r) for r in range(case["requests"])]
        runner.step([StepEntry(seq, [0], [0]) for seq in seqs])
        for seq in seqs:
            runner.close(seq)
        runner.enable_graphs(case["requests"], max(len(t) for t in texts))
        runner.capture_graphs([case["requests"]])
    logits = torch.empty((sum(want for step in steps for *_, want in step), VOCAB), dtype=torch.float32, device="cuda:0")
    feeds = [[(r, texts[r][first: first + count].tolist(), [count - 1] if want else [])
              for r, first, count, want in step] for step in steps]
    return {"runner": runner, "feeds": feeds, "requests": case["requests"], "logits": logits}


def run(state):
    runner, logits, row = state["runner"], state["logits"], 0
    seqs = [runner.open(r) for r in range(state["requests"])]
    for feed in state["feeds"]:
        got = runner.step([StepEntry(seqs[r], tokens, want) for r, tokens, want in feed])
        if got is not None:
            logits[row: row + len(got)].copy_(got)
            row += len(got)
    for seq in seqs:
        runner.close(seq)
    return logits


# ---- what a pass cannot do without -------------------------------------------------------------


def work(case):
    width, heads, kv_heads, dim, ff, _, tied, _ = SHAPES[case["shape"]]
    config, size = config_of(case), 4 if case["dtype"] == "float32" else 2
    state_heads = max(1, width // (2 * dim))
    cached = heads * dim, 2 * kv_heads * dim  # what a query and a key cost: elements of q, elements kept a token
    matrices, attend = 0, []  # elements of all layers' matrices (of a layer run once); (window, cost) of each attention
    seen = set()
    linear = 0  # elements of the matrices over all runs: what a token multiplies with
    state = 0   # elements of all states
    for index, begins in runs_of(config) if case["design"] != "qwen3" else [(i, None) for i in range(case["layers"])]:
        layer = {"type": "attention"} if case["design"] == "qwen3" else config["layers"][index]
        kind = layer["type"]
        window = layer.get("mixer", {}).get("mask", {}).get("size")
        if kind in ("retention", "lightning", "gla"):
            inner = state_heads * dim
            own = 5 * width * inner
            state += inner * dim
            attend.append((None, 0, 0, 4 * inner * dim))
        elif kind.startswith("latent"):
            own = width * heads * (dim + 64) + width * (256 + 64) + 2 * heads * dim * 256 + width * heads * dim
            own += width * (heads if kind == "latent_attention" else heads * dim)
            attend.append((window, 2 * heads * (256 + 64 + 256), 256 + 64, 0))
        else:
            own = width * (heads + 2 * kv_heads) * dim + heads * dim * width
            attend.append((window, 4 * cached[0], cached[1], 0))
        own += (2 * (ff * 3 // 2) if case["design"] == "ranudra" else 3 * ff) * width
        if begins is not None and case["design"] == "farorax":
            own += 2 * width * width
        linear += own
        if index not in seen:
            matrices += own
            seen.add(index)
    bytes_, flops = 0.0, 0.0
    for step in steps_of(case):
        wanted = sum(want for *_, want in step)
        tokens = sum(count for _, _, count, _ in step)
        bytes_ += size * matrices + (size * VOCAB * width + 4 * wanted * VOCAB if wanted else 0) + size * tokens * width
        bytes_ += 8 * state * len(step)
        flops += 2.0 * tokens * linear + 2.0 * wanted * VOCAB * width
        for _, first, count, _ in step:
            for window, per_pair, kept, per_token in attend:
                reach = first + count if window is None else min(first + count, window + count - 1)
                last = np.arange(first + 1, first + count + 1, dtype=np.float64)
                flops += per_pair * float((last if window is None else np.minimum(last, window)).sum()) + per_token * count
                bytes_ += size * kept * (reach + count)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # against 64 bits the 32-bit path is 3e-6 to 7e-6 off, the bfloat16 one 0.6e-2 to 1.8e-2
    if case["dtype"] == "float32":
        return {"rel": 3e-5, "max": 3e-4}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------------------

F = torch.float64


class Weights:
    """The model's tensors by the names they have in a checkpoint, in 64 bits, one at a time."""

    def __init__(self, case, seed):
        options = PylonConfig(dtype=case["dtype"], max_batch_size=1, page_size=PAGE, num_pages=1, cuda_graphs=False)
        raw = config_of(case)
        runner = Runner.from_random(raw, seed, options, std=0.02, norm_jitter=0.1)
        arch = resolve(raw)
        self.targets = arch.weight_targets(arch.parse_config(raw))
        self.params = {path: owner.params[name] for path, owner, name in runner.model.named_params()}

    def __contains__(self, name):
        return name in self.targets

    def raw(self, name):
        target = self.targets[name]
        value = self.params[target.param]
        if tuple(value.shape) != tuple(target.shape):
            value = value[target.row_start: target.row_start + target.shape[0]]
        return value

    def __getitem__(self, name):
        return self.raw(name).to(F)


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(x):
    return x * torch.sigmoid(x)


def ranges(lengths):
    at = 0
    for n in lengths:
        yield slice(at, at + n)
        at += n


def angles(lengths, freq):
    """Angles [tokens, pairs] of all requests' tokens; formed in float32 where ``freq`` is."""
    pos = torch.cat([torch.arange(n, device=freq.device) for n in lengths]).to(freq.dtype)
    return (pos[:, None] * freq[None, :]).to(F)


def rotate(x, angle, halves, mult=1.0):
    """x [tokens, heads, dim]: pairs (i, i + n) with ``halves``, else neighbours, of the first 2n elements."""
    n = angle.shape[1]
    c, s = (angle.cos() * mult)[:, None], (angle.sin() * mult)[:, None]
    out = x.clone()
    first, second = (slice(0, n), slice(n, 2 * n)) if halves else (slice(0, 2 * n, 2), slice(1, 2 * n, 2))
    u, v = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * c - v * s, v * c + u * s
    return out


def attend(q, k, v, scale, lengths, window=None, sink=None, bias=None):
    """Softmax attention of every request's tokens: q [tokens, heads, dim], k and v [tokens, groups, ...].
    ``sink`` [heads]: exp(sink) joins the denominator.  ``bias(head, distances)`` is added to the scores."""
    heads, group = q.shape[1], q.shape[1] // k.shape[1]
    out = torch.empty((q.shape[0], heads, v.shape[2]), dtype=F, device=q.device)
    for at in ranges(lengths):
        n = at.stop - at.start
        far = torch.arange(n, device=q.device)[:, None] - torch.arange(n, device=q.device)[None]
        hidden = (far < 0) if window is None else (far < 0) | (far >= window)
        for h in range(heads):
            s = (q[at, h] @ k[at, h // group].T) * scale
            if bias is not None:
                s += bias(h, far.clamp(min=0))
            s.masked_fill_(hidden, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(n, 1)], 1)
            out[at, h] = torch.softmax(s, -1)[:, :n] @ v[at, h // group]
    return out


def fading(q, k, v, decay, lengths):
    """o_t = S_t^T q_t, S_t = decay S_(t-1) + k_t v_t^T, one decay a head; [tokens, heads, ...]."""
    out = torch.empty_like(v)
    for at in ranges(lengths):
        n = at.stop - at.start
        far = torch.arange(n, device=q.device)[:, None] - torch.arange(n, device=q.device)[None]
        for h in range(q.shape[1]):
            fade = torch.where(far >= 0, float(decay[h]) ** far.clamp(min=0).to(F), 0.0)
            out[at, h] = ((q[at, h] @ k[at, h].T) * fade) @ v[at, h]
    return out


def fading_channels(q, k, v, log_decay, lengths):
    """The same with a decay of its own for every token and channel, 64 tokens at a time."""
    out = torch.empty_like(v)
    for at in ranges(lengths):
        state = torch.zeros((q.shape[1], q.shape[2], v.shape[2]), dtype=F, device=q.device)
        for first in range(at.start, at.stop, 64):
            c = slice(first, min(first + 64, at.stop))
            run = log_decay[c].cumsum(0).transpose(0, 1)  # [heads, tokens, dim]
            qs, ks = q[c].transpose(0, 1) * run.exp(), k[c].transpose(0, 1) * (-run).exp()
            vs = v[c].transpose(0, 1)
            out[c] = ((qs @ ks.transpose(1, 2)).tril() @ vs + qs @ state).transpose(0, 1)
            state = run[:, -1, :, None].exp() * (state + ks.transpose(1, 2) @ vs)
    return out


def exact(case, seed):
    texts = texts_of(case, seed)
    lengths = [len(t) for t in texts]
    starts = np.concatenate([[0], np.cumsum(lengths)])
    order = [int(starts[r]) + first + count - 1 for step in steps_of(case) for r, first, count, want in step if want]
    ids = torch.from_numpy(np.concatenate(texts)).to("cuda:0")
    last = torch.tensor(order, device="cuda:0")
    forward = {"qwen3": exact_qwen3, "vupuzen": exact_vupuzen, "ranudra": exact_ranudra, "farorax": exact_farorax}
    return forward[case["design"]](config_of(case), Weights(case, seed), ids, lengths, last)


def exact_qwen3(c, w, ids, lengths, last):
    heads, groups, dim, eps = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["rms_norm_eps"]
    n = len(ids)
    x = w.raw("model.embed_tokens.weight")[ids].to(F)
    exponent = torch.arange(0, dim, 2, dtype=torch.float32, device=ids.device) / dim
    turn = angles(lengths, 1.0 / torch.pow(torch.tensor(c["rope_theta"], dtype=torch.float32, device=ids.device), exponent))
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = rms(x, eps) * w[p + "input_layernorm.weight"]
        a = p + "self_attn."
        q = rms((h @ w[a + "q_proj.weight"].T).view(n, heads, dim), eps) * w[a + "q_norm.weight"]
        k = rms((h @ w[a + "k_proj.weight"].T).view(n, groups, dim), eps) * w[a + "k_norm.weight"]
        v = (h @ w[a + "v_proj.weight"].T).view(n, groups, dim)
        o = attend(rotate(q, turn, True), rotate(k, turn, True), v, dim ** -0.5, lengths)
        x = x + o.reshape(n, -1) @ w[a + "o_proj.weight"].T
        h = rms(x, eps) * w[p + "post_attention_layernorm.weight"]
        f = silu(h @ w[p + "mlp.gate_proj.weight"].T) * (h @ w[p + "mlp.up_proj.weight"].T)
        x = x + f @ w[p + "mlp.down_proj.weight"].T
    head = "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"
    return (rms(x[last], eps) * w["model.norm.weight"]) @ w[head].T


def exact_vupuzen(c, w, ids, lengths, last):
    eps, n, taps = c["norm"]["eps"], len(ids), c["canon"]["taps"]
    x = w.raw("embed")[ids].to(F)
    for i, layer in enumerate(c["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        h = rms(x, eps) * w[p + "norm1"]
        taken, mixed = w[p + "canon1"], h.clone()
        for at in ranges(lengths):
            for j in range(taps):  # the last tap weighs the token itself
                back = taps - 1 - j
                if back < at.stop - at.start:
                    mixed[at.start + back: at.stop] += taken[:, j] * h[at.start: at.stop - back]
        h, p = mixed, p + "mix."
        heads, dim = m["heads"], m["dim"]
        if layer["type"] == "attention":
            q, k, v = ((h @ w[p + s].T).view(n, g, dim) for s, g in (("q", heads), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
            rel, far = w[p + "rel"], float(m["bias_max"])
            rows = rel.shape[0]
            half = rows // 2
            bucket = torch.tensor([d if d < half else min(rows - 1, half + math.floor(
                math.log(d / half) / math.log(far / half) * (rows - half))) for d in range(max(lengths))], device=ids.device)
            o = attend(q, k, v, float(m["scale"]), lengths, sink=torch.zeros(heads, dtype=F, device=ids.device),
                       bias=lambda head, d: rel[bucket[d], head]).reshape(n, -1)
        else:
            q, k, v = ((h @ w[p + s].T).view(n, heads, dim) for s in "qkv")
            dims = m["rot"]["dims"]
            index = torch.arange(dims // 2, dtype=torch.float32, device=ids.device)
            base = torch.tensor(m["rot"]["base"], dtype=torch.float32, device=ids.device)
            turn = angles(lengths, torch.pow(base, -(2.0 * index / dims)))
            o = fading(rotate(q, turn, True), rotate(k, turn, True) * dim ** -0.5, v, m["decay"], lengths)
            o = rms(o, eps).reshape(n, -1) * silu(h @ w[p + "g"].T)
        p = f"l{i}."
        x = x + rms(o @ w[p + "mix.o"].T, eps) * w[p + "norm1b"]
        h, limit = rms(x, eps) * w[p + "norm2"], float(layer["mlp"]["limit"])
        g = (h @ w[p + "mlp.gate"].T).clamp(max=limit)
        u = (h @ w[p + "mlp.up"].T).clamp(-limit, limit)
        x = x + rms((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[p + "mlp.down"].T, eps) * w[p + "norm2b"]
    return ((rms(x[last], eps) * w["final.norm"]) @ w["head"].T) * c["logit_scale"]


def exact_ranudra(c, w, ids, lengths, last):
    eps, n = c["norm"]["eps"], len(ids)

    def centred(x, weight):
        return rms(x - x.mean(-1, keepdim=True), eps) * weight

    def turns(rot):
        dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
        i = torch.arange(dims // 2, dtype=F, device=ids.device)
        f = base ** (-2.0 * i / dims)
        if sc is None:
            return angles(lengths, f), 1.0

        def where(times):
            return dims * math.log(sc["original"] / (2.0 * math.pi * times)) / (2.0 * math.log(base))

        lo, hi = max(math.floor(where(sc["fast"])), 0), min(math.ceil(where(sc["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        return angles(lengths, f / sc["factor"] * ramp + f * (1.0 - ramp)), 0.1 * math.log(sc["factor"]) + 1.0

    def latent(h, m, p, by_head):
        heads, dim, rank = m["heads"], m["dim"], m["kv_rank"]
        turn, mult = turns(m["rot"])
        q = (h @ w[p + "q"].T).view(n, heads, -1)
        q = torch.cat([q[..., :dim], rotate(q[..., dim:], turn, False, mult)], -1)
        both = h @ w[p + "dkv"].T
        kept = rms(both[:, :rank], eps) * w[p + "dkv.norm"]
        shared = rotate(both[:, None, rank:], turn, False, mult)
        k = torch.cat([(kept @ w[p + "uk"].T).view(n, heads, dim), shared.expand(-1, heads, -1)], -1)
        v = (kept @ w[p + "uv"].T).view(n, heads, -1)
        o = attend(q, k, v, m["scale"], lengths, m["mask"]["size"], w[p + "sink"] if p + "sink" in w else None)
        g = torch.sigmoid(h @ w[p + "g"].T)
        return (o * (g[:, :, None] if by_head else g.view(o.shape))).reshape(n, -1) @ w[p + "o"].T

    def gated(h, m, p):
        heads, dim = m["heads"], m["dim"]
        q, k, v = ((h @ w[p + s].T).view(n, heads, dim) for s in "qkv")
        z = (h @ w[p + "a1"].T) @ w[p + "a2"].T + w[p + "a2.b"]
        fade = (torch.nn.functional.logsigmoid(z) / m["tau"]).view(n, heads, dim)
        o = rms(fading_channels(q * dim ** -0.5, k, v, fade, lengths), eps) * w[p + "norm"]
        return (o.reshape(n, -1) * silu(h @ w[p + "g"].T)) @ w[p + "o"].T

    def joined(xs, sublayer, p):
        y = sublayer(torch.einsum("s,snd->nd", w[p + "in"], xs))
        return torch.einsum("st,snd->tnd", w[p + "mix"], xs) + w[p + "out"][:, None, None] * y

    x = w.raw("embed")[ids].to(F) * c["embedding"]["scale"]
    xs = x[None].repeat(c["streams"], 1, 1)
    for i, _ in runs_of(c):
        layer, p = c["layers"][i], f"l{i}."
        m, kind = layer["mixer"], layer["type"]
        xs = joined(xs, lambda u: gated(centred(u, w[p + "norm1"]), m, p + "mix.") if kind == "gla" else
                    latent(centred(u, w[p + "norm1"]), m, p + "mix.", kind == "latent_attention"), p + "hc1.")
        xs = joined(xs, lambda u: (centred(u, w[p + "norm2"]) @ w[p + "mlp.up"].T).relu().square() @ w[p + "mlp.down"].T,
                    p + "hc2.")
    return centred(xs.sum(0)[last], w["final.norm"]) @ w["embed"].T


def exact_farorax(c, w, ids, lengths, last):
    eps, n, mult = c["norm"]["eps"], len(ids), c["residual_mult"]
    x = embedded = w.raw("embed")[ids].to(F)
    for i, begins in runs_of(c):
        layer, p = c["layers"][i], f"l{i}."
        m, heads, dim = layer["mixer"], layer["mixer"]["heads"], layer["mixer"]["dim"]
        if begins is not None:
            x = torch.cat([x, embedded], -1) @ w["loop.in"].T + w["loop.step"][begins]
        h, p = rms(x, eps) * w[p + "norm1"], p + "mix."
        if layer["type"] == "lightning":
            q, k, v = (silu(h @ w[p + s].T).view(n, heads, dim) for s in "qkv")
            o = fading(q, k, v, m["decay"], lengths).reshape(n, -1)
            o = rms(o, eps) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].T)
        else:
            rot, sc = m["rot"], m["rot"]["scaling"]
            f = rot["base"] ** (-2.0 * torch.arange(rot["dims"] // 2, dtype=F, device=ids.device) / rot["dims"])
            wave = 2.0 * math.pi / f
            part = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
            blend = (1.0 - part) * f / sc["factor"] + part * f
            f = torch.where(wave < sc["original"] / sc["high"], f,
                            torch.where(wave > sc["original"] / sc["low"], f / sc["factor"], blend))
            turn = angles(lengths, f)
            q = rotate((h @ w[p + "q"].T).view(n, heads, dim), turn, False)
            k = rotate((h @ w[p + "k"].T).view(n, m["kv_heads"], dim), turn, False)
            v = (h @ w[p + "v"].T).view(n, m["kv_heads"], dim)
            o = attend(q, k, v, m["scale"], lengths, m["mask"]["size"], w[p + "sink"]).reshape(n, -1)
        x = x + mult * (o @ w[p + "o"].T)
        p = f"l{i}."
        h = rms(x, eps) * w[p + "norm2"]
        f = torch.nn.functional.gelu(h @ w[p + "mlp.gate"].T, approximate="tanh") * (h @ w[p + "mlp.up"].T)
        x = x + mult * (f @ w[p + "mlp.down"].T)
    logits = (rms(x[last], eps) * w["final.norm"]) @ w["head"].T
    cap = c["logit_softcap"]
    return cap * torch.tanh(logits / cap)
