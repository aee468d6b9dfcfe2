"""Cases that stand for the work users have the engine do: steps of live requests through `Engine.step` and
`Engine.choose`, over the layer sizes that `bench.py` and the tests know.

A case names a model, an arithmetic type and one of three passes:

  decode  one token each for `requests` live requests whose caches hold `context` tokens (with `ragged`: lengths between
          `shortest` and `context`, spread over their logarithm).  The next pass feeds the requests' next tokens, as
          generation does; the tokens are given, so that a pass's inputs do not hang on the rounding of the one before.
  prompt  `requests` new requests of `tokens` tokens each, fed whole or, where a prompt is longer than a step takes, in
          portions as `generate_tokens` feeds it; the first token is chosen and the requests are closed.
  mixed   a new request's first `tokens` tokens beside one token each of `requests` live ones: what a round of the
          scheduler is while a prompt arrives.

Outputs are the float32 logits of the wanted places.  The chosen tokens are read as a program reads them but not returned:
they are the logits' largest places, and random weights leave the two largest closer than bfloat16 rounding.

Models have fewer layers than their originals (every layer is alike; the head and the embedding are whole).
"""

from __future__ import annotations

import hashlib
import math

import torch

PAGE, STEP_TOKENS = 16, 2048

_QWEN3 = dict(architectures=["Qwen3ForCausalLM"], head_dim=128, rope_theta=1000000.0, rms_norm_eps=1e-6, hidden_act="silu")
_SINK = dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=128 ** -0.5,
             rot=dict(dims=64, base=1e6, scaling=dict(factor=4.0, original=4096, fast=32.0, slow=1.0)))
_DELTA = dict(heads=16, kv_heads=16, dim=128, vdim=128, conv=4, ranks=dict(decay=64, gate=64))
_TWO_MAPS = dict(heads=16, kv_heads=4, dim=64, vdim=128, diff=0.3, scale=0.125, mask=dict(size=1024),
                 rot=dict(dims=64, base=1e4, scaling=dict(factor=8.0, original=8192, low=1.0, high=4.0)))
MODELS = {
    # the layer sizes of bench.py's three dense models ...
    "qwen3-8b": dict(_QWEN3, num_hidden_layers=8, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8,
                     intermediate_size=12288, vocab_size=151936, tie_word_embeddings=False),
    "qwen3-14b": dict(_QWEN3, num_hidden_layers=6, hidden_size=5120, num_attention_heads=40, num_key_value_heads=8,
                      intermediate_size=17408, vocab_size=151936, tie_word_embeddings=False),
    "qwen3-32b": dict(_QWEN3, num_hidden_layers=4, hidden_size=5120, num_attention_heads=64, num_key_value_heads=8,
                      intermediate_size=25600, vocab_size=151936, tie_word_embeddings=False),
    # ... and the small one that its designs are held against
    "qwen3-s": dict(_QWEN3, num_hidden_layers=8, hidden_size=2048, num_attention_heads=16, num_key_value_heads=4,
                    intermediate_size=3072, vocab_size=32768, tie_word_embeddings=True),
    # the design whose mixers share most with the other designs (attention with a sink, differential attention over a
    # window, a matrix state per head).  Designs with routed experts are not among the cases: a rounding that turns a choice
    # of experts changes a token's output wholly, so two correct implementations cannot be held against each other.
    "lirulix-s": dict(
        architecture="Lirulix", vocab=32768, width=2048, norm=dict(eps=1e-6), loop=dict(start=0, stop=8, times=1),
        layers=[dict(type=kind, mixer=mixer, mlp=dict(kind="dense", ff=3072)) for kind, mixer in 2 * (
            ("attention", _SINK), ("channel_delta", _DELTA), ("attention", _SINK), ("attention_2", _TWO_MAPS))]),
}


def listed() -> list[dict]:
    bf16, f32 = "bfloat16", "float32"
    return [
        # a short chat with a small model: the smallest call, all launches and latency
        dict(name="chat small b1", kind="decode", model="qwen3-s", dtype=bf16, requests=1, context=210, ragged=False),
        # one user of the 8B model in the middle of a conversation
        dict(name="decode 8b b1", kind="decode", model="qwen3-8b", dtype=bf16, requests=1, context=2048, ragged=False),
        # the headline: a small batch with long contexts, where weights and cache weigh the same
        dict(name="decode 8b b8 long", kind="decode", model="qwen3-8b", dtype=bf16, requests=8, context=8192, ragged=False),
        # a full batch right after its prompts
        dict(name="decode 8b b64", kind="decode", model="qwen3-8b", dtype=bf16, requests=64, context=2048, ragged=False),
        # a served batch as it comes: an odd number of requests, contexts from a few lines to a book chapter
        dict(name="decode 14b b27 ragged", kind="decode", model="qwen3-14b", dtype=bf16, requests=27, context=16000, ragged=True),
        # the headline's prefill: a prompt of one whole step
        dict(name="prompt 8b 2048", kind="prompt", model="qwen3-8b", dtype=bf16, requests=1, tokens=2048),
        # a document with the largest model: a prompt of four portions, the last ones with a long history
        dict(name="prompt 32b 8192", kind="prompt", model="qwen3-32b", dtype=bf16, requests=1, tokens=8192),
        # a question of a few sentences that arrives beside decoding requests: a scheduler's round
        dict(name="mixed 8b 171 beside 8", kind="mixed", model="qwen3-8b", dtype=bf16, requests=8, context=8192, ragged=False, tokens=171),
        # the 32-bit path, which results are checked with: a few prompts fed together, and their decoding
        dict(name="prompt small f32", kind="prompt", model="qwen3-s", dtype=f32, requests=3, tokens=333),
        dict(name="decode small f32 b3", kind="decode", model="qwen3-s", dtype=f32, requests=3, context=700, ragged=True),
        # another design's prompt and its decoding batch
        dict(name="prompt lirulix 2000", kind="prompt", model="lirulix-s", dtype=bf16, requests=1, tokens=2000),
        dict(name="decode lirulix b8", kind="decode", model="lirulix-s", dtype=bf16, requests=8, context=2048, ragged=False),
    ]


def _spread(rng, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    """Batches of 1 to 64 with contexts of 64 to 16,384 tokens (at most 131,072 in all; less in the 32-bit path and the other
    design), prompts of 20 to 8,192 tokens (at most one step's in all where several are fed together), portions of 17 to 512
    tokens beside 1 to 32 requests; the 32-bit path at the small model's sizes."""
    kind = rng.choice(("decode", "decode", "prompt", "prompt", "mixed"))
    model = rng.choice(("qwen3-8b", "qwen3-8b", "qwen3-14b", "qwen3-32b", "qwen3-s", "qwen3-s", "lirulix-s"))
    dtype = rng.choice(("bfloat16", "float32")) if model == "qwen3-s" else "bfloat16"
    if kind == "prompt":
        requests = rng.choice((1, 1, 1, 2, 3, 4))
        most = 2048 // requests if requests > 1 else 2048 if dtype == "float32" or model.startswith("lirulix") else 8192
        return dict(kind=kind, model=model, dtype=dtype, requests=requests, tokens=_spread(rng, 20, most))
    requests = _spread(rng, 1, 64 if kind == "decode" else 32)
    most = 16384 if dtype == "float32" else 32768 if model.startswith("lirulix") else 131072
    long = 2048 if model.startswith("lirulix") or dtype == "float32" else 16384
    case = dict(kind=kind, model=model, dtype=dtype, requests=requests, context=_spread(rng, 64, min(long, most // requests)),
                ragged=rng.random() < 0.5)
    if kind == "mixed":
        case["tokens"] = _spread(rng, 17, 512)
    return case


# ---- what a user's program holds ----------------------------------------------------------------------------------------

SHORTEST = 64


def _contexts(case) -> list[int]:
    """The live requests' lengths: all alike, or spread evenly over the logarithm."""
    count, longest = case["requests"], case["context"]
    if not case["ragged"] or count == 1:
        return [longest] * count
    low = min(SHORTEST, longest)
    return [int(round(low * (longest / low) ** (i / (count - 1)))) for i in range(count)]


def _vocab(case) -> int:
    raw = MODELS[case["model"]]
    return raw.get("vocab_size") or raw["vocab"]


def _token_ids(case, seed: int) -> dict:
    """The token ids of a case: the live requests' contexts, the tokens they are fed pass after pass, the new prompts."""
    generator = torch.Generator().manual_seed(seed * 7919 + 17)
    ids = lambda *shape: torch.randint(0, _vocab(case), shape, generator=generator)
    if case["kind"] == "prompt":
        return dict(prompts=ids(case["requests"], case["tokens"]).tolist())
    held = dict(contexts=[ids(length).tolist() for length in _contexts(case)], fed=ids(64, case["requests"]).tolist())
    if case["kind"] == "mixed":
        held["prompts"] = ids(1, case["tokens"]).tolist()
    return held


def prepare(case, seed):
    from ampere_kv_engine_amd.config import EngineConfig, LirulixConfig, Qwen3Config
    from ampere_kv_engine_amd.engine import Engine, StepEntry
    raw = MODELS[case["model"]]
    held = _token_ids(case, seed)
    # room for the tokens that the passes add to the live requests
    grown = 0 if case["kind"] == "prompt" else 6144 if case["requests"] <= 4 else 3072
    lengths = [len(c) + grown for c in held.get("contexts", ())] + [len(p) for p in held.get("prompts", ())]
    engine = Engine.from_random(
        (LirulixConfig if "architecture" in raw else Qwen3Config).from_dict(raw), seed=seed, engine_config=EngineConfig(
            dtype=case["dtype"], page_size=PAGE, num_pages=sum(-(-length // PAGE) + 1 for length in lengths),
            max_seqs=len(lengths), max_batched_tokens=STEP_TOKENS, max_seq_len=max(max(lengths) + PAGE, STEP_TOKENS), device="cuda:0"))
    live = [engine.open(f"live{i}") for i in range(len(held.get("contexts", ())))]
    # the contexts enter the cache as any prompt does, as many in a step as it takes
    left = [(seq, ids) for seq, ids in zip(live, held.get("contexts", ()))]
    while left:
        room, entries, later = STEP_TOKENS, [], []
        for seq, ids in left:
            take = min(room, len(ids))
            if take:
                entries.append(StepEntry(seq, ids[:take], []))
                room -= take
            if take < len(ids):
                later.append((seq, ids[take:]))
        engine.step(entries)
        left = later
    return dict(case=case, engine=engine, live=live, passes=0, waiting=None, **{k: held.get(k) for k in ("fed", "prompts")})


def run(state):
    from ampere_kv_engine_amd.engine import StepEntry
    engine, kind = state["engine"], state["case"]["kind"]
    if kind == "prompt":
        seqs = [engine.open(f"new{i}") for i in range(len(state["prompts"]))]
        longest = len(state["prompts"][0])
        portion = STEP_TOKENS // len(seqs)
        for start in range(0, longest, portion):
            stop = min(start + portion, longest)
            logits = engine.step([StepEntry(seq, ids[start:stop], [stop - start - 1] if stop == longest else [])
                                  for seq, ids in zip(seqs, state["prompts"])], borrow_logits=True)
        engine.choose(logits)
        for seq in seqs:
            engine.close(seq)
        return logits
    fed = state["fed"][state["passes"] % len(state["fed"])]
    state["passes"] += 1
    entries = [StepEntry(seq, [token], [0]) for seq, token in zip(state["live"], fed)]
    if kind == "mixed":
        arriving = engine.open("new")
        ids = state["prompts"][0]
        logits = engine.step(entries + [StepEntry(arriving, ids, [len(ids) - 1])], borrow_logits=True)
        engine.choose(logits)
        engine.close(arriving)
        return logits
    logits = engine.step(entries, borrow_logits=True)
    # the tokens come to the host while the next step runs, as the scheduler reads them
    waiting, state["waiting"] = state["waiting"], engine.choose_later(logits)
    if waiting is not None:
        waiting.tokens()
    return logits


# ---- what a pass cannot do without --------------------------------------------------------------------------------------

def _spans(case) -> list[tuple[int, int]]:
    """(tokens a request holds before the pass, tokens it brings) of every request of the pass."""
    spans = [(length, 1) for length in _contexts(case)] if case["kind"] != "prompt" else []
    if case["kind"] == "prompt":
        spans = [(0, case["tokens"])] * case["requests"]
    elif case["kind"] == "mixed":
        spans.append((0, case["tokens"]))
    return spans


def _layers(raw) -> list[dict]:
    """Per layer: numbers of its matrices (`weights`), of its cache record (`record`, per token), of the multiplications a
    query and a key cost (`pair`), the window its queries see, of a state a request carries (`state`) and of the
    multiplications a token costs there."""
    if "architecture" not in raw:
        width, heads, groups, dim, ff = (raw[n] for n in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim",
                                                          "intermediate_size"))
        return [dict(weights=width * dim * (2 * heads + 2 * groups) + 3 * width * ff, record=2 * groups * dim, pair=2 * heads * dim,
                     window=None, state=0)] * raw["num_hidden_layers"]
    out, width = [], raw["width"]
    for layer in raw["layers"]:
        m, ff = layer["mixer"], 3 * width * layer["mlp"]["ff"]
        heads, groups, dim, vdim = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        if layer["type"] == "channel_delta":
            columns = 2 * groups * dim + heads * vdim
            low = sum(m["ranks"].values()) * width + m["ranks"]["decay"] * heads * dim + m["ranks"]["gate"] * heads * vdim
            out.append(dict(weights=width * (columns + heads * vdim + heads) + columns * m["conv"] + low + ff, record=0, pair=0,
                            window=None, state=heads * dim * vdim))
        else:
            maps = 2 if layer["type"] == "attention_2" else 1
            gate = heads * vdim if maps == 2 else 0
            out.append(dict(weights=width * (maps * (heads + groups) * dim + groups * vdim + heads * vdim + gate) + ff,
                            record=groups * (maps * dim + vdim), pair=maps * heads * (dim + vdim),
                            window=m["mask"]["size"] if m.get("mask") else None, state=0))
    return out


def work(case):
    """Every matrix of the layers and the head once, the cache records that the pass's queries see once, the new records and
    the logits once; two operations a multiplication."""
    raw, spans = MODELS[case["model"]], _spans(case)
    size = 4 if case["dtype"] == "float32" else 2
    tokens, wanted = sum(new for _, new in spans), len(spans)
    head = _vocab(case) * (raw.get("hidden_size") or raw["width"])
    moved, flops = size * head + 4 * wanted * _vocab(case), 2 * wanted * head
    for layer in _layers(raw):
        moved += size * layer["weights"]
        flops += 2 * tokens * layer["weights"]
        for before, new in spans:
            window = layer["window"] or before + new
            moved += size * layer["record"] * (min(before, window - 1) + new) + 8 * layer["state"]
            seen = sum(min(before + i + 1, window) for i in range(new))
            flops += 2 * layer["pair"] * seen + 6 * new * layer["state"]
    return dict(bytes=moved, flops=flops)


def tolerance(case):
    """Relative error of the logits, and the largest difference over their root mean square.  Against `exact` the engine shows
    4.5e-6 with 32-bit types; in bfloat16 0.007 (lirulix-s) and, growing with the layers, 0.014 to 0.025 (the qwen3 sizes: every
    branch's input, inner rows and output are rounded)."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits, in plain torch ------------------------------------------------------------------------------------

def _weight(name: str, shape, seed: int, dtype, mean: float = 0.0, std: float = 0.02) -> torch.Tensor:
    """A tensor of the engine's random weights (`Engine.from_random`): normal, drawn on the device by a generator seeded from
    the weights' seed and the tensor's name, rounded to the engine's type."""
    digest = hashlib.sha256(f"{seed}:{name}".encode()).digest()
    generator = torch.Generator(device="cuda:0").manual_seed(int.from_bytes(digest[:8], "little") >> 1)
    value = mean + torch.randn(tuple(shape), generator=generator, dtype=torch.float32, device="cuda:0") * std
    return value.to(dtype).double()


def _unit_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turned(x, freq, magnitude: float = 1.0):
    """x [n, heads, width]: dimension i turned with i + half by position * freq[i]; dimensions beyond 2 * half pass.  Angles are
    float32 products, as the model's definition forms them."""
    half = len(freq)
    angle = torch.arange(x.shape[0], dtype=torch.float32, device=x.device)[:, None] * freq.to(torch.float32).to(x.device)[None]
    cos, sin = (angle.cos() * magnitude).double()[:, None], (angle.sin() * magnitude).double()[:, None]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat((a * cos - b * sin, b * cos + a * sin, x[..., 2 * half:]), dim=-1)


def _attention(q, k, v, scale: float, sink=None, window=None):
    """q [n, heads, dim], k [n, groups, dim], v [n, groups, vdim] -> [n, heads, vdim], causal; a sink per head joins the
    denominator."""
    n, heads, groups = q.shape[0], q.shape[1], k.shape[1]
    share = heads // groups
    out = torch.empty(n, heads, v.shape[-1], dtype=q.dtype, device=q.device)
    rows = max(16, (1 << 27) // (n * share))
    for g in range(groups):
        keys, values = k[:, g].T.contiguous(), v[:, g].contiguous()
        for start in range(0, n, rows):
            stop = min(start + rows, n)
            scores = (q[start:stop, g * share:(g + 1) * share].reshape(-1, q.shape[-1]) @ keys[:, :stop] * scale).view(stop - start, share, stop)
            distance = torch.arange(start, stop, device=q.device)[:, None] - torch.arange(stop, device=q.device)[None]
            hidden = distance < 0 if window is None else (distance < 0) | (distance >= window)
            scores = scores.masked_fill(hidden[:, None], -math.inf)
            if sink is not None:
                extra = sink[g * share:(g + 1) * share].view(1, share, 1).expand(stop - start, share, 1)
                scores = torch.cat((scores, extra), dim=-1)
            weights = scores.softmax(-1)[..., :stop].reshape(-1, stop)
            out[start:stop, g * share:(g + 1) * share] = (weights @ values[:stop]).view(stop - start, share, -1)
    return out


def _exact_qwen3(raw, sequences, seed, dtype):
    """The last position's logits of every sequence."""
    width, heads, groups, dim = (raw[n] for n in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim"))
    ff, eps, vocab = raw["intermediate_size"], raw["rms_norm_eps"], raw["vocab_size"]
    draw_one = lambda name, *shape: _weight(name, shape, seed, dtype)
    norm = lambda name, n: _weight(name, (n,), seed, dtype, mean=1.0, std=0.1)
    freq = 1.0 / raw["rope_theta"] ** (torch.arange(0, dim, 2, dtype=torch.int64).float() / dim)
    ids = torch.tensor([t for s in sequences for t in s], device="cuda:0")
    edges = [0]
    for s in sequences:
        edges.append(edges[-1] + len(s))
    x = draw_one("model.embed_tokens.weight", vocab, width)[ids]
    parts = [slice(i, i + 8192) for i in range(0, len(ids), 8192)]
    for layer in range(raw["num_hidden_layers"]):
        at = f"model.layers.{layer}."
        first, second = norm(at + "input_layernorm.weight", width), norm(at + "post_attention_layernorm.weight", width)
        q_norm, k_norm = norm(at + "self_attn.q_norm.weight", dim), norm(at + "self_attn.k_norm.weight", dim)
        wq, wk, wv = (draw_one(f"{at}self_attn.{n}_proj.weight", h * dim, width).T for n, h in (("q", heads), ("k", groups), ("v", groups)))
        wo = draw_one(at + "self_attn.o_proj.weight", width, heads * dim).T
        for a, b in zip(edges, edges[1:]):
            h = _unit_rms(x[a:b], eps) * first
            q = _turned(_unit_rms((h @ wq).view(-1, heads, dim), eps) * q_norm, freq)
            k = _turned(_unit_rms((h @ wk).view(-1, groups, dim), eps) * k_norm, freq)
            x[a:b] += _attention(q, k, (h @ wv).view(-1, groups, dim), dim ** -0.5).reshape(b - a, -1) @ wo
        del wq, wk, wv, wo
        gate, up = (draw_one(f"{at}mlp.{n}_proj.weight", ff, width).T for n in ("gate", "up"))
        down = draw_one(at + "mlp.down_proj.weight", width, ff).T
        for part in parts:
            h = _unit_rms(x[part], eps) * second
            x[part] += (torch.nn.functional.silu(h @ gate) * (h @ up)) @ down
    last = _unit_rms(x[[b - 1 for b in edges[1:]]], eps) * norm("model.norm.weight", width)
    head = "model.embed_tokens.weight" if raw["tie_word_embeddings"] else "lm_head.weight"
    return last @ draw_one(head, vocab, width).T


def _stretched(rot):
    """(frequencies, factor on cos and sin) of a rotation whose frequencies a rule moves: a ramp between dimension indices
    (`fast`, `slow`), or by wavelength (`low`, `high`)."""
    dims, base, s = rot["dims"], rot["base"], rot["scaling"]
    freq = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    factor, original = s["factor"], s["original"]
    if "fast" in s:
        turned = lambda turns: dims * math.log(original / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(turned(s["fast"])), 0), min(math.ceil(turned(s["slow"])), dims - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
        return torch.tensor([f / factor * r + f * (1 - r) for f, r in zip(freq, ramp)], dtype=torch.float64), 0.1 * math.log(factor) + 1
    out = []
    for f in freq:
        share = (original * f / (2 * math.pi) - s["low"]) / (s["high"] - s["low"])
        share = min(max(share, 0.0), 1.0)
        out.append((1 - share) * f / factor + share * f)
    return torch.tensor(out, dtype=torch.float64), 1.0


def _exact_lirulix(raw, sequences, seed, dtype):
    """The last position's logits of every sequence (all of one length)."""
    width, vocab, eps = raw["width"], raw["vocab"], raw["norm"]["eps"]
    n, count = len(sequences[0]), len(sequences)
    get = lambda name, *shape: _weight(name, shape, seed, dtype)
    norm = lambda x, name: _unit_rms(x, eps) * (1.0 + _weight(name, (width,), seed, dtype, std=0.1))
    x = norm(get("embed", vocab, width)[torch.tensor(sequences, device="cuda:0")], "embed.norm")       # [count, n, width]
    x = x + get("loop.step", raw["loop"]["times"], width)[0]
    for index, layer in enumerate(raw["layers"]):
        at, m = f"l{index}.mix.", layer["mixer"]
        heads, groups, dim, vdim = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        h = norm(x, f"l{index}.norm1")
        wo = get(at + "o", width, heads * vdim).T
        if layer["type"] == "channel_delta":
            conv = {}
            for name, columns in (("q", groups * dim), ("k", groups * dim), ("v", heads * vdim)):
                z, taps = h @ get(at + name, columns, width).T, get(f"{at}{name}.conv", columns, m["conv"])
                reach = m["conv"] - 1
                z = torch.cat((torch.zeros_like(z[:, :1]).expand(-1, reach, -1), z), dim=1)
                conv[name] = torch.nn.functional.silu(sum(z[:, t:t + n] * taps[:, t] for t in range(m["conv"]))).view(count, n, -1, vdim if name == "v" else dim)
            q, k = (conv[name] / torch.sqrt((conv[name] ** 2).sum(-1, keepdim=True) + 1e-6) for name in "qk")
            q, k = ((z * s).repeat_interleave(heads // groups, dim=2) for z, s in ((q, dim ** -0.5), (k, 1.0)))
            beta = torch.sigmoid(h @ get(at + "b", heads, width).T)
            low = (h @ get(at + "a1", m["ranks"]["decay"], width).T) @ get(at + "a2", heads * dim, m["ranks"]["decay"]).T
            rate = torch.exp(get(at + "A_log", heads))[:, None]
            decay = torch.exp(-rate * torch.nn.functional.softplus(low + get(at + "dt_bias", heads * dim)).view(count, n, heads, dim))
            S = torch.zeros(count, heads, dim, vdim, dtype=x.dtype, device=x.device)
            o = torch.empty(count, n, heads, vdim, dtype=x.dtype, device=x.device)
            for t in range(n):
                S = S * decay[:, t, :, :, None]
                u = beta[:, t, :, None] * (conv["v"][:, t] - (S * k[:, t, :, :, None]).sum(2))
                S = S + k[:, t, :, :, None] * u[:, :, None, :]
                o[:, t] = (S * q[:, t, :, :, None]).sum(2)
            o = _unit_rms(o, eps) * _weight(at + "norm", (vdim,), seed, dtype, mean=1.0, std=0.1)
            gate = (h @ get(at + "g1", m["ranks"]["gate"], width).T) @ get(at + "g2", heads * vdim, m["ranks"]["gate"]).T
            mixed = (o * torch.sigmoid(gate).view(o.shape)).reshape(count, n, -1) @ wo
        else:
            maps = 2 if layer["type"] == "attention_2" else 1
            freq, magnitude = _stretched(m["rot"])
            wq, wk, wv = (get(at + name, columns, width).T for name, columns in (("q", maps * heads * dim), ("k", maps * groups * dim), ("v", groups * vdim)))
            sink = get(at + "sink", heads) if maps == 1 else None
            if maps == 2:
                lq1, lk1, lq2, lk2 = (get(at + name, dim) for name in ("lq1", "lk1", "lq2", "lk2"))
                lam = torch.exp((lq1 * lk1).sum()) - torch.exp((lq2 * lk2).sum()) + m["diff"]
                wg = get(at + "g", heads * vdim, width).T
            mixed = torch.empty_like(x)
            for s in range(count):
                q = _turned((h[s] @ wq).view(n, maps * heads, dim), freq, magnitude).view(n, heads, maps, dim)
                k = _turned((h[s] @ wk).view(n, maps * groups, dim), freq, magnitude).view(n, groups, maps, dim)
                v = (h[s] @ wv).view(n, groups, vdim)
                window = m["mask"]["size"] if m.get("mask") else None
                seen = [_attention(q[:, :, i], k[:, :, i], v, m["scale"], sink, window) for i in range(maps)]
                if maps == 1:
                    mixed[s] = seen[0].reshape(n, -1) @ wo
                else:
                    o = _unit_rms(seen[0] - lam * seen[1], eps) * (1.0 - m["diff"])
                    mixed[s] = (o.reshape(n, -1) * torch.sigmoid(h[s] @ wg)) @ wo
        x = x + mixed
        ff, mlp = layer["mlp"]["ff"], f"l{index}.mlp."
        h = norm(x, f"l{index}.norm2")
        gated = torch.nn.functional.gelu(h @ get(mlp + "gate", ff, width).T, approximate="tanh") * (h @ get(mlp + "up", ff, width).T)
        x = x + gated @ get(mlp + "down", width, ff).T
    return norm(x[:, -1], "final.norm") @ get("head", vocab, width).T


@torch.no_grad()
def exact(case, seed):
    raw, held = MODELS[case["model"]], _token_ids(case, seed)
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    sequences = [ids + [token] for ids, token in zip(held.get("contexts", ()), held["fed"][0])] if "fed" in held else []
    sequences += held.get("prompts", [])
    if sum(len(s) for s in sequences) > 140000:
        return None
    if "architecture" not in raw:
        return _exact_qwen3(raw, sequences, seed, dtype)
    out = []        # (sequences of one length together: the recurrence is a loop over tokens)
    for length in sorted({len(s) for s in sequences}):
        which = [i for i, s in enumerate(sequences) if len(s) == length]
        out += list(zip(which, _exact_lirulix(raw, [sequences[i] for i in which], seed, dtype)))
    return torch.stack([row for _, row in sorted(out, key=lambda pair: pair[0])])
