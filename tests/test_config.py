"""Typed configuration from config.json keys, and the architecture registry."""

import json

import pytest

from ampere_kv_engine_amd.config import (ConfigError, EngineConfig, Qwen3Config, known_architectures, load_config,
                                         register_architecture)
from conftest import TINY_A, TINY_B


def test_reads_every_size_from_the_keys():
    a, b = Qwen3Config.from_dict(TINY_A), Qwen3Config.from_dict(TINY_B)
    assert (a.num_hidden_layers, a.hidden_size, a.num_attention_heads, a.num_key_value_heads, a.head_dim) == (2, 64, 4, 2, 16)
    assert (a.intermediate_size, a.vocab_size, a.rope_theta, a.rms_norm_eps, a.tie_word_embeddings) == (128, 256, 1e4, 1e-6, True)
    assert (b.q_size, b.kv_size, b.group_size) == (192, 32, 6) and b.q_size != b.hidden_size
    assert not b.tie_word_embeddings and b.rms_norm_eps == 1e-5 and b.rope_theta == 1e6


def test_head_dim_defaults_to_hidden_over_heads_and_kv_heads_to_heads():
    raw = {k: v for k, v in TINY_A.items() if k not in ("head_dim", "num_key_value_heads")}
    c = Qwen3Config.from_dict(raw)
    assert c.head_dim == 16 and c.num_key_value_heads == 4


@pytest.mark.parametrize("key", ["vocab_size", "hidden_size", "num_hidden_layers", "num_attention_heads",
                                 "intermediate_size", "rope_theta", "rms_norm_eps"])
def test_a_missing_size_is_an_error_not_a_default(key):
    raw = {k: v for k, v in TINY_B.items() if k != key}
    with pytest.raises(ConfigError, match=key):
        Qwen3Config.from_dict(raw)


@pytest.mark.parametrize("change,match", [
    ({"hidden_act": "gelu"}, "hidden_act"), ({"use_sliding_window": True, "sliding_window": 128}, "sliding"),
    ({"rope_scaling": {"type": "yarn"}}, "rope_scaling"), ({"attention_bias": "yes"}, "attention_bias"),
    ({"num_key_value_heads": 4}, "multiple"), ({"head_dim": 31}, "odd"), ({"vocab_size": -1}, "vocab_size"),
    ({"num_hidden_layers": 2.5}, "num_hidden_layers"), ({"rope_theta": 0}, "rope_theta")])
def test_unsupported_options_are_refused(change, match):
    with pytest.raises(ConfigError, match=match):
        Qwen3Config.from_dict({**TINY_B, **change})


def test_round_trip_through_config_json(tmp_path):
    c = Qwen3Config.from_dict({**TINY_B, "eos_token_id": [7, 9]})
    (tmp_path / "config.json").write_text(json.dumps(c.to_dict()))
    again = load_config(str(tmp_path))
    assert again == c and again.eos_token_ids == (7, 9)
    (tmp_path / "generation_config.json").write_text(json.dumps({"eos_token_id": 3}))
    assert load_config(str(tmp_path)).eos_token_ids == (3,)


def test_registry_chooses_by_architecture_name(tmp_path):
    assert "Qwen3ForCausalLM" in known_architectures()
    (tmp_path / "config.json").write_text(json.dumps({**TINY_A, "architectures": ["NoSuchModel"]}))
    with pytest.raises(ConfigError, match="NoSuchModel.*Qwen3ForCausalLM"):
        load_config(str(tmp_path))
    (tmp_path / "config.json").write_text(json.dumps({k: v for k, v in TINY_A.items() if k != "architectures"}))
    with pytest.raises(ConfigError, match="architectures"):
        load_config(str(tmp_path))
    with pytest.raises(ValueError, match="already registered"):
        register_architecture("Qwen3ForCausalLM", Qwen3Config)


def test_model_spec_carries_sizes_layer_by_layer():
    spec = Qwen3Config.from_dict(TINY_B).to_model_spec()
    assert len(spec.layers) == 3 and [e.layer for e in spec.run_order] == [0, 1, 2]
    mixer = spec.layers[1].mixer
    assert mixer.kind == "attention" and mixer["q_heads"] == 6 and mixer["kv_heads"] == 1 and mixer["head_dim"] == 32
    assert mixer["position"].kind == "rope_half" and mixer["position"]["theta"] == 1e6
    assert mixer["qk_norm"]["eps"] == 1e-5 and mixer["scale"] == 32 ** -0.5
    assert spec.layers[2].feed_forward["intermediate_size"] == 200 and spec.layers[2].prefix == "model.layers.2."
    assert spec.head["tied_to"] is None
    assert Qwen3Config.from_dict(TINY_A).to_model_spec().head["tied_to"] == "model.embed_tokens.weight"


def test_engine_config_checks_its_numbers():
    with pytest.raises(ValueError):
        EngineConfig(dtype="float16")
    with pytest.raises(ValueError):
        EngineConfig(page_size=0)
    assert EngineConfig(page_size=16, max_seq_len=100).max_pages_per_seq == 7


def test_plan_memory_counts_weights_copies_and_pages():
    """Pages that fit beside a model, from its specification alone (no device)."""
    from ampere_kv_engine_amd.config import EngineConfig, Qwen3Config
    from ampere_kv_engine_amd.engine import plan_memory
    raw = dict(architectures=["Qwen3ForCausalLM"], vocab_size=1000, hidden_size=64, num_hidden_layers=3,
               num_attention_heads=4, num_key_value_heads=2, head_dim=16, intermediate_size=128, rope_theta=1e4,
               rms_norm_eps=1e-6, tie_word_embeddings=False, hidden_act="silu")
    spec = Qwen3Config.from_dict(raw).to_model_spec()
    layer = (4 + 2 + 2) * 16 * 64 + 64 * 64 + 3 * 128 * 64          # q/k/v, o, gate/up/down
    norms = 3 * (2 * 64 + 2 * 16) + 64
    config = EngineConfig(dtype="bfloat16", page_size=8, num_pages=1, max_seqs=2, max_batched_tokens=16, max_seq_len=64)
    plan = plan_memory(spec, config, 1 << 30)
    assert plan.weight_bytes == 2 * (3 * layer + norms + 2 * 1000 * 64)
    assert plan.second_copy_bytes == 2 * (3 * layer + 1000 * 64)        # every matrix but the embedding table
    assert plan.page_bytes == 3 * 2 * 2 * 16 * 8 * 2                     # layers x (k, v) x kv heads x dim x page x bytes
    assert plan.num_pages == ((1 << 30) - plan.weight_bytes - plan.second_copy_bytes - plan.fixed_bytes) // plan.page_bytes
    assert plan.tokens == plan.num_pages * 8
    own = plan_memory(spec, EngineConfig(dtype="bfloat16", page_size=8, num_pages=1, max_seqs=2, max_batched_tokens=16,
                                         max_seq_len=64, library_products_above=None), 1 << 30)
    assert own.second_copy_bytes == 0 and own.num_pages > plan.num_pages
    full = plan_memory(spec, EngineConfig(dtype="float32", page_size=8, num_pages=1, max_seqs=2, max_batched_tokens=16,
                                          max_seq_len=64), 1 << 30)
    assert full.weight_bytes == 2 * plan.weight_bytes and full.second_copy_bytes == 0 and full.page_bytes == 2 * plan.page_bytes
    with pytest.raises(ValueError, match="not a page"):
        plan_memory(spec, config, plan.weight_bytes + plan.second_copy_bytes + plan.fixed_bytes + plan.page_bytes)


def test_plan_memory_counts_a_second_copy_only_where_a_part_keeps_one():
    """The row-major copy for the BLAS library is `Linear`'s doing: it marks its tensors (`TensorSpec.library_copy`).
    A part with storage of its own - the toy routed feed-forward of the GPU tests, whose experts' matrices are plain
    `TensorSpec`s - is counted once."""
    import test_toy_parts_gpu as toy
    from ampere_kv_engine_amd.config import EngineConfig
    from ampere_kv_engine_amd.engine import plan_memory
    from ampere_kv_engine_amd.parts import register_part
    register_part("feed_forward", "routed", toy.RoutedFeedForward, replace=True)
    register_part("position", "adjacent_pair_rotary", toy.AdjacentPairRotary, replace=True)
    spec = toy.RoutedConfig(vocab_size=97, hidden_size=32, decay=0.0, eps=1e-5).to_model_spec()
    config = EngineConfig(dtype="bfloat16", page_size=8, num_pages=1, max_seqs=2, max_batched_tokens=16, max_seq_len=64)
    plan = plan_memory(spec, config, 1 << 30)
    attention = 3 * 2 * 16 * 32 + 32 * 2 * 16                       # q/k/v and o of one layer
    dense = 3 * 40 * 32
    experts = 3 * 32 + 3 * (2 * 24 * 32 + 32 * 24)                   # router and three experts
    head = 97 * 32
    assert plan.second_copy_bytes == 2 * (2 * attention + dense + head)
    assert plan.weight_bytes >= 2 * (2 * attention + dense + experts + 2 * head)


def test_layers_share_one_position_table_and_the_memory_plan_counts_it():
    """Every layer's rotary part is handed the same cos/sin table (ampere_kv/runner.py:41-44 builds its inverse
    frequencies once per model); `plan_memory` counts it once, sized by the longest sequence."""
    from ampere_kv_engine_amd.config import EngineConfig, Qwen3Config
    from ampere_kv_engine_amd.engine import plan_memory
    from ampere_kv_engine_amd.engine.dry import dry_runtime
    from ampere_kv_engine_amd.engine.model import Model
    raw = dict(architectures=["Qwen3ForCausalLM"], vocab_size=1000, hidden_size=64, num_hidden_layers=5,
               num_attention_heads=4, num_key_value_heads=2, head_dim=16, intermediate_size=128, rope_theta=1e4,
               rms_norm_eps=1e-6, tie_word_embeddings=False, hidden_act="silu")
    spec = Qwen3Config.from_dict(raw).to_model_spec()
    runtime = dry_runtime(max_seq_len=4096, page_size=8)
    model = Model(spec, runtime)
    tables = {id(block.mixer.position.table) for block in model.blocks}
    assert len(tables) == 1
    assert runtime.shared_bytes() == 4096 * 8 * 2 * 4
    sizes = dict(dtype="bfloat16", page_size=8, num_pages=1, max_seqs=2, max_batched_tokens=16)
    short = plan_memory(spec, EngineConfig(max_seq_len=64, **sizes), 1 << 30)
    long = plan_memory(spec, EngineConfig(max_seq_len=64 + 4096, **sizes), 1 << 30)
    assert long.fixed_bytes - short.fixed_bytes == 4096 * 8 * 2 * 4


@pytest.mark.parametrize("vectors,vdim,seqs", [(16, 128, 64), (64, 128, 64), (128, 256, 3), (16, 64, 1)])
@pytest.mark.parametrize("step", [1111, 64])
def test_partial_sums_of_growing_contexts_are_bounded_and_in_the_memory_plan(vectors, vdim, seqs, step):
    """Single tokens of gated attention leave a segment's sums per 256 keys.  Contexts that grow to 131,072 tokens, with exact
    lengths as eager steps have them, other activations before and behind: what the arena holds beside the first step's
    stays within what the plan counts."""
    from types import SimpleNamespace
    import torch
    from ampere_kv_engine_amd.config import EngineConfig
    from ampere_kv_engine_amd.engine.batch import Arena
    from ampere_kv_engine_amd.kernels import partial_sums
    config = EngineConfig(max_seqs=seqs, max_seq_len=131072, page_size=16)
    ctx = SimpleNamespace(arena=Arena("meta"))
    assert ctx.arena.chunk_bytes == partial_sums.ARENA_CHUNK
    held = None
    for length in list(range(200, 131072, step)) + [131072]:
        ctx.arena.reset()
        ctx.arena.take((seqs, 40000), torch.bfloat16)
        segments, at_once, floats = partial_sums.gated_cut(seqs, vectors, vdim, length, None, None, 0)
        assert segments * 256 >= length > (segments - 1) * 256 and floats == (at_once * vectors * segments * (vdim + 4) if segments > 1 else 0)
        assert at_once == 1 or floats * 4 <= partial_sums.BYTES
        if floats:
            assert partial_sums.take(ctx, floats, "meta").numel() >= floats
        ctx.arena.take((seqs, 40000), torch.bfloat16)
        now = sum(chunk.numel() for chunk in ctx.arena.chunks)
        held = held or now
    assert now - held <= partial_sums.gated_bytes(config, vectors, 128, vdim, None, None, 0) <= 1 << 30


@pytest.mark.parametrize("window", [None, 1000])
def test_partial_sums_of_float32_portions_are_bounded_and_in_the_memory_plan(window):
    """Float32 attention leaves a segment's sums per 256 keys where tiles of 16 (token, head) rows are few.  Portions of 200
    tokens (16 heads over 4: 200 blocks) of a prompt of 32,768, and single tokens at every length: with a window the sums stop
    growing at its segments, without one what the arena holds stays within what the plan counts."""
    from types import SimpleNamespace
    import torch
    from ampere_kv_engine_amd.config import EngineConfig
    from ampere_kv_engine_amd.engine.batch import Arena
    from ampere_kv_engine_amd.kernels import partial_sums
    config = EngineConfig(dtype="float32", max_seqs=64, max_seq_len=32768, page_size=16)
    ctx = SimpleNamespace(arena=Arena("meta"))
    asked = 0
    for tokens, lengths in ((200, range(200, 32769, 200)), (1, range(1, 32769, 61))):
        for length in lengths:
            ctx.arena.reset()
            segments = partial_sums.f32_segments(length, window)
            assert window is None or segments <= 5
            if segments > 1:
                floats = 16 * segments * 132
                launches = partial_sums.launches_of_tiles([0, tokens], 1, 4, partial_sums.at_once(tokens, floats))
                largest = max(end - first for first, end, _, _ in launches) * floats
                assert 4 * largest <= partial_sums.BYTES
                asked = max(asked, partial_sums.take(ctx, largest, "meta").numel())
    held = sum(chunk.numel() for chunk in ctx.arena.chunks)
    assert 4 * asked <= held <= partial_sums.f32_bytes(config, 16, 128, window)
    assert held <= (512 << 20 if window is None else 64 << 20)


@pytest.mark.parametrize("share", [1, 2, 3, 4, 6, 16, 20])
def test_launches_of_tiles_hold_whole_tiles(share):
    """Requests of all sizes, launches of every size: the launches' tokens and tiles follow each other, and a launch's tiles are those
    of its tokens."""
    from ampere_kv_engine_amd.kernels import partial_sums
    starts = [0, 1, 2, 19, 20, 100, 116, 117, 150]
    tiles = [(first + row // share, first + min(row + 15, (end - first) * share - 1) // share)      # a tile's first and last token
             for first, end in zip(starts, starts[1:]) for row in range(0, (end - first) * share, 16)]
    for at_once in range(1, 160):
        launches = partial_sums.launches_of_tiles(starts, len(starts) - 1, share, at_once)
        token = tile = 0
        for first, end, first_tile, count in launches:
            assert (first, first_tile) == (token, tile) and 0 < end - first <= max(at_once, partial_sums.tile_tokens(share))
            assert [t for t in tiles if first <= t[0] < end] == tiles[tile:tile + count]
            assert all(t[1] < end for t in tiles[tile:tile + count])
            token, tile = end, tile + count
        assert (token, tile) == (150, len(tiles))


def test_the_room_of_walked_states_covers_what_the_kernels_ask_for():
    """The memory plan's counts of floats against the kernel library's, over sizes, mixes of forms and of requests."""
    import ctypes
    import random
    from ampere_kv_engine_amd.csrc.build import parts_library_path
    from ampere_kv_engine_amd.kernels import walk_room
    path = parts_library_path()
    if path is None:
        pytest.skip("the kernel library is not built")
    lib = ctypes.CDLL(path)
    asks = [getattr(lib, f"akv_{name}_workspace") for name in ("delta_rule", "time_mixing", "matrix_memory")]
    for ask in asks:
        ask.restype = ctypes.c_long
    rng = random.Random(3)
    for _ in range(300):
        groups, dim, vdim = rng.choice((1, 2, 16)), rng.choice((24, 64, 128, 192, 256, 300)), rng.choice((16, 36, 128))
        heads, per_head, tokens, seqs = groups * rng.choice((1, 3, 16)), rng.random() < 0.5, rng.randrange(1, 5000), rng.randrange(1, 65)
        longest, walked = rng.randrange(1, tokens + 1), rng.randrange(0, tokens + 1)
        need = asks[0](tokens, seqs, heads, groups, dim, vdim, int(per_head), longest, walked)
        assert need <= walk_room.delta_rule_floats(tokens, seqs, heads, groups, dim, vdim, per_head)
        assert asks[1](tokens, heads, dim) <= walk_room.time_mixing_floats(tokens, heads, dim)
        assert asks[2](tokens, heads, dim, vdim) <= walk_room.matrix_memory_floats(tokens, heads, dim, vdim)


def test_the_room_of_walked_states_is_bounded_and_in_the_memory_plan(monkeypatch):
    """Steps that grow token by token: what is held - the buffer and what it outgrew - stays within the plan's count."""
    from types import SimpleNamespace
    import torch
    from ampere_kv_engine_amd.config import EngineConfig
    from ampere_kv_engine_amd.config.lirulix import LirulixConfig
    from ampere_kv_engine_amd.engine import plan_memory
    from ampere_kv_engine_amd.engine.dry import dry_runtime
    from ampere_kv_engine_amd.engine.model import Model
    from ampere_kv_engine_amd.engine.sizing import walk_bytes
    from ampere_kv_engine_amd.kernels import walk_room
    from ampere_kv_engine_amd.kernels.hip_parts import PartsKernels
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    kernels = SimpleNamespace(device="meta")
    sizes = (16, 1, 128, 128)                       # one key head for 16 heads: what the chunks hold is most beside the rows
    for tokens in range(1, 2049):
        PartsKernels._walk_workspace(kernels, walk_room.delta_rule_floats(tokens, 8, *sizes, False))
    held = 4 * sum(b.numel() for b in [kernels._walk_buffer, *kernels._walk_outgrown] if b is not None)
    assert held <= walk_room.held_bytes(walk_room.delta_rule_floats(2048, 8, *sizes, False)) <= 1 << 28
    raw = dict(architecture="Lirulix", vocab=256, width=64, norm=dict(eps=1e-6), loop=dict(start=0, stop=2, times=1), layers=[
        dict(type="channel_delta", mixer=dict(heads=16, kv_heads=1, dim=128, vdim=128, conv=4, ranks=dict(decay=8, gate=8)),
             mlp=dict(kind="dense", ff=64)),
        dict(type="attention", mixer=dict(heads=4, kv_heads=2, dim=32, vdim=32, scale=0.2, rot=dict(
            dims=16, base=1e4, scaling=dict(factor=4.0, original=64, fast=32.0, slow=1.0))), mlp=dict(kind="dense", ff=64))])
    spec = LirulixConfig.from_dict(raw).to_model_spec()
    config = EngineConfig(page_size=16, max_seqs=8, max_seq_len=4096, max_batched_tokens=2048, num_pages=8)
    assert walk_bytes(Model(spec, dry_runtime(4096, 16)), config) >= held
    small = EngineConfig(page_size=16, max_seqs=8, max_seq_len=4096, max_batched_tokens=64, num_pages=8)
    plans = [plan_memory(spec, c, 1 << 33) for c in (config, small)]
    assert plans[0].fixed_bytes - plans[1].fixed_bytes > held - walk_room.held_bytes(1)
    qwen3 = Model(Qwen3Config.from_dict(TINY_A).to_model_spec(), dry_runtime(8192, 16))
    assert walk_bytes(qwen3, config) == 0


def test_plan_memory_counts_the_partial_sums_of_cut_attention():
    """Once per arena, by the mixer with the largest; none where every key a token sees lies in one segment, nor for float32's gated
    attention, which is one kernel, or bfloat16's plain one, whose cut is sized by the device."""
    from ampere_kv_engine_amd.config import EngineConfig
    from ampere_kv_engine_amd.engine.sizing import partial_sum_bytes
    from ampere_kv_engine_amd.engine.dry import dry_runtime
    from ampere_kv_engine_amd.engine.model import Model
    from ampere_kv_engine_amd.config.lirulix import LirulixConfig
    raw = dict(architecture="Lirulix", vocab=256, width=64, norm=dict(eps=1e-6), loop=dict(start=0, stop=1, times=1), layers=[
        dict(type="attention", mixer=dict(heads=4, kv_heads=2, dim=32, vdim=32, scale=0.2, rot=dict(
            dims=16, base=1e4, scaling=dict(factor=4.0, original=64, fast=32.0, slow=1.0))), mlp=dict(kind="dense", ff=64))])
    model = Model(LirulixConfig.from_dict(raw).to_model_spec(), dry_runtime(8192, 16))
    sizes = dict(page_size=16, max_seqs=2, max_seq_len=8192)
    assert partial_sum_bytes(model, EngineConfig(**sizes)) == 2 * (64 << 20)
    assert partial_sum_bytes(model, EngineConfig(dtype="float32", **sizes)) == 0
    assert partial_sum_bytes(model, EngineConfig(page_size=8, max_seqs=2, max_seq_len=8192)) == 0
    assert partial_sum_bytes(model, EngineConfig(page_size=16, max_seqs=2, max_seq_len=128, graph_width_multiple=1)) == 0
    qwen3 = Model(Qwen3Config.from_dict(TINY_A).to_model_spec(), dry_runtime(8192, 16))
    assert partial_sum_bytes(qwen3, EngineConfig(**sizes)) == 0
    assert partial_sum_bytes(qwen3, EngineConfig(dtype="float32", **sizes)) >= 2 * (64 << 20)


def test_attention_bias_adds_the_four_bias_vectors_to_every_layer():
    """`attention_bias: true` (ampere_kv/runner.py:64-66, :165 hand each projection's bias to F.linear): every layer
    expects q/k/v/o biases beside the 11 tensors, 15 L + 3 in all; the key reads back from `to_dict`."""
    from ampere_kv_engine_amd.config import Qwen3Config
    from ampere_kv_engine_amd.engine.model import expected_tensors
    raw = dict(architectures=["Qwen3ForCausalLM"], vocab_size=100, hidden_size=64, num_hidden_layers=3,
               num_attention_heads=4, num_key_value_heads=2, head_dim=16, intermediate_size=128, rope_theta=1e4,
               rms_norm_eps=1e-6, tie_word_embeddings=False, hidden_act="silu", attention_bias=True)
    config = Qwen3Config.from_dict(raw)
    assert config.attention_bias and config.to_dict()["attention_bias"] is True
    assert Qwen3Config.from_dict(config.to_dict()) == config
    specs = {t.name: t for t in expected_tensors(config.to_model_spec())}
    assert len(specs) == 15 * 3 + 3
    assert specs["model.layers.1.self_attn.q_proj.bias"].shape == (64,)
    assert specs["model.layers.1.self_attn.k_proj.bias"].shape == (32,)
    assert specs["model.layers.2.self_attn.o_proj.bias"].shape == (64,) and specs["model.layers.2.self_attn.o_proj.bias"].role == "bias"
    assert not any("mlp" in name and name.endswith("bias") for name in specs)
    plain = Qwen3Config.from_dict({**raw, "attention_bias": False})
    assert len(expected_tensors(plain.to_model_spec())) == 11 * 3 + 3
