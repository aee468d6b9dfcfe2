"""Tukevik on the host: its configuration, and the engine's side of it - registry, loading, a cache layer with pages and
a state, chunks whose pages are given back, batching, the scheduler - with the torch double standing in for the HIP
kernels, against the plain implementation.  The HIP kernels meet the same cases in `test_tukevik_gpu.py`."""

import copy
import json
import math
import os

import pytest
import torch

import schedules
import tukevik_cases as T
from ampere_kv_engine_amd.cache.pages import BlockTable, PageAllocator
from ampere_kv_engine_amd.config import ConfigError, TukevikConfig, load_config
from ampere_kv_engine_amd.engine.model import expected_tensors
from conftest import random_ids
from plain import tukevik_plain as plain
from torch_kernels import TorchKernels


@pytest.fixture(scope="module", params=["A", "B"])       # (the third configuration, of served sizes, meets the GPU alone)
def case(request, tmp_path_factory):
    return T.make_case(request.param, str(tmp_path_factory.mktemp(f"tukevik_{request.param}")))


@pytest.fixture(scope="module")
def engine(case):
    return T.make_engine(case, "float32", "cpu", kernels=TorchKernels())


@pytest.mark.parametrize("cutting", T.CUTTINGS, ids=lambda f: f.__name__)
def test_cutting(engine, case, cutting):
    if cutting is T.case_long_decoding:
        cutting(engine, case, tokens=90)         # (the double steps through recurrences token by token on the host)
    else:
        cutting(engine, case)


@pytest.mark.parametrize("mechanism", T.MECHANISMS)
def test_one_mechanism_alone(mechanism, tmp_path):
    case = T.make_case(mechanism, str(tmp_path), T.alone(mechanism))
    engine = T.make_engine(case, "float32", "cpu", kernels=TorchKernels())
    T.case_whole(engine, case)
    T.case_portions_down_to_two_tokens(engine, case)
    T.case_mixed_with_pages_and_slots_used_again(engine, case)


def test_the_configuration_names_every_part_and_tensor(tmp_path):
    raw = copy.deepcopy(T.TUKEVIK_A)
    folder = str(tmp_path)
    with open(os.path.join(folder, "config.json"), "w") as handle:
        json.dump(raw, handle)
    config = load_config(folder)                     # found through the key "architecture"
    assert isinstance(config, TukevikConfig) and config.to_dict() == raw
    spec = config.to_model_spec()
    assert [layer.mixer.kind for layer in spec.layers] == ["rglru", "parallel", "parallel", "rglru"]
    assert [layer.feed_forward.kind for layer in spec.layers] == ["none", "routed_experts", "swiglu", "routed_experts"]
    assert all(layer.block.kind == "scaled_prenorm" and layer.block["residual_scale"] == 0.7 for layer in spec.layers)
    (left, left_scale), (right, right_scale) = spec.layers[1].mixer["branches"]
    assert (left.kind, left_scale, right.kind, right_scale) == ("gated_attention", 1.3, "retention", 0.6)
    assert left["chunk"] == 13 and left["softcap"] == 6.0 and left["sink"] and left["head_gate"] and right["rotary_dims"] == 8
    assert spec.head["tied_to"] == "embed"
    names = {t.name: tuple(t.shape) for t in expected_tensors(spec) if not t.optional}
    assert names["embed"] == (211, 96) and "head" not in names and names["final.norm"] == (96,)
    assert "l0.norm2" not in names and names["l0.mix.conv"] == (80, 4) and names["l0.mix.ra"] == (5, 16, 16)
    assert names["l0.mix.ri.b"] == (5, 16) and names["l0.mix.lam"] == (80,) and names["l0.mix.y.b"] == (80,)
    assert names["l1.mix.left.q"] == (144, 96) and names["l1.mix.left.k.b"] == (48,) and names["l1.mix.left.v"] == (32, 96)
    assert names["l1.mix.left.g"] == (6, 96) and "l1.mix.left.g.b" not in names and names["l1.mix.left.o"] == (96, 96)
    assert names["l1.mix.right.k"] == (48, 96) and names["l1.mix.right.g"] == (72, 96) and names["l1.mix.right.o"] == (96, 72)
    assert names["l1.mlp.e5.gate"] == (20, 96) and names["l1.mlp.router.b"] == (6,) and names["l1.mlp.shared.sg"] == (1, 96)
    assert names["l1.mlp.shared.down"] == (96, 28) and names["l2.mlp.down"] == (96, 72)
    assert "l3.mlp.shared.sg" not in names and names["l3.mlp.e3.down"] == (96, 16)


@pytest.mark.parametrize("change,message", [
    (lambda raw: raw["layers"][1].update(type="attention"), "type"),
    (lambda raw: raw["layers"][1]["mixer"]["left"].update(kv_heads=4), "kv_heads"),
    (lambda raw: raw["layers"][1]["mixer"]["right"].update(decay=[0.9]), "decay"),
    (lambda raw: raw["layers"][1]["mixer"]["right"]["rot"].update(dims=7), "rot.dims"),
    (lambda raw: raw["layers"][0]["mixer"].update(blocks=3), "blocks"),
    (lambda raw: raw["layers"][3]["mlp"]["router"].update(top=5), "experts"),
    (lambda raw: raw["layers"][2]["mlp"].update(kind="glu"), "kind"),
    (lambda raw: raw["layers"][1]["mixer"].pop("left_scale"), "left_scale"),
    (lambda raw: raw.pop("residual_mult"), "residual_mult"),
])
def test_configurations_the_design_does_not_allow_are_refused(change, message):
    raw = copy.deepcopy(T.TUKEVIK_A)
    change(raw)
    with pytest.raises(ConfigError, match=message):
        TukevikConfig.from_dict(raw)


def test_a_layer_with_pages_and_a_state_and_chunks_that_give_pages_back(case, engine):
    from ampere_kv_engine_amd.engine import StepEntry
    layers = case["raw"]["layers"]
    page = case["page_size"]
    for index, layer in enumerate(layers):
        view = engine.cache.layer_cache[index]
        m = layer["mixer"]
        if layer["type"] == "rglru":
            assert view.k is None and view.state.shape == (4, m["width"] * m["conv"])
        else:
            left, right = m["left"], m["right"]
            assert view.k.shape[1:] == (left["kv_heads"], page, left["dim"]) and view.v.shape[1:] == (left["kv_heads"], left["vdim"], page)
            assert view.state.shape == (4, right["heads"] * right["dim"] * right["vdim"])
    seq = engine.open("w")
    engine.step([StepEntry(seq, case["requests"]["d"], [])])
    engine.step([StepEntry(seq, case["requests"]["a"][:1], [])])    # (what a chunk has left behind is given back when tokens register)
    for table, group in zip(seq.tables, engine.cache.groups):
        assert table.num_held <= (group.need.chunk + page - 1) // page + 1
    slot = seq.slot
    engine.close(seq)
    seq = engine.open("again")           # the slot comes round again: nothing of its predecessor is left
    assert seq.slot == slot
    for index in range(len(layers)):
        assert not engine.cache.layer_cache[index].state[slot].any()
    engine.close(seq)


def test_block_table_with_chunks():
    pool = PageAllocator(16)
    table = BlockTable(pool, page_size=4, chunk=10)
    table.append_tokens(9)                      # positions 0..8: chunk 0
    assert table.num_held == 3
    table.append_tokens(3)                      # 9..11: position 10 opens chunk 1, whose first page also holds 8 and 9
    assert table.num_held == 3
    table.append_tokens(1)                      # the next position, 12, is of chunk 1 (from 10): pages 0 and 1 are passed
    assert table.num_held == 2 and table.pages[:2] == (-1, -1)
    table.append_tokens(9)                      # positions 13..21; 21 is of chunk 2 - but what is given back is decided
    assert table.num_held == 4                  # when tokens register: the portion's first position, 13, still reads from 10 on
    table.append_tokens(1)                      # the next position, 22, is of chunk 2 (from 20): page 5 holds 20..23
    assert table.num_held == 1 and pool.num_free == 15
    table.release()
    assert pool.num_free == 16


# ---- the plain implementation's own mechanisms, where a sentence of the design can be checked by hand -----------------

def test_plain_mechanisms_by_hand():
    assert plain.chunk_mask(5, 3).int().tolist() == [[1, 0, 0, 0, 0], [1, 1, 0, 0, 0], [1, 1, 1, 0, 0], [0, 0, 0, 1, 0], [0, 0, 0, 1, 1]]
    p = plain.sink_softmax(torch.tensor([[0.0, math.log(2.0), 5.0]]), torch.tensor([[True, True, False]]))
    torch.testing.assert_close(p, torch.tensor([[0.25, 0.5, 0.0]]))
    chosen, weights = plain.route(torch.eye(2), torch.tensor([[1.0, 0.0], [3.0, 0.0], [2.0, 0.0]]), torch.tensor([0.0, 0.0, 1.5]), 2)
    assert chosen[0].tolist() == [2, 1]        # logits 1, 3, 3.5 for the first token
    torch.testing.assert_close(weights[0], torch.softmax(torch.tensor([3.5, 3.0]), 0))
    out = plain.causal_conv(torch.tensor([[1.0], [2.0], [4.0]]), torch.tensor([[100.0, 10.0, 1.0]]), torch.tensor([0.5]))
    assert out[:, 0].tolist() == [1.5, 12.5, 124.5]
    u = torch.ones(3, 2)
    S = plain.rglru_scan(u, torch.full((3, 2), 0.5), torch.ones(3, 2), torch.zeros(2))
    a = math.exp(-8 * 0.5 * math.log(2.0))
    torch.testing.assert_close(S[1], torch.full((2,), a * math.sqrt(1 - a * a) + math.sqrt(1 - a * a)))
    turned = plain.rotate_first_dims(torch.arange(6.0).view(1, 1, 6), torch.tensor([2]), dims=4, base=100.0)
    assert torch.equal(turned[..., 4:], torch.tensor([[[4.0, 5.0]]]))
    torch.testing.assert_close(turned[0, 0, 0], torch.tensor(0 * math.cos(2.0) - 2 * math.sin(2.0)))
    torch.testing.assert_close(turned[0, 0, 3], torch.tensor(3 * math.cos(0.2) + 1 * math.sin(0.2)))


def test_a_far_key_at_the_chunks_edges_decides_the_output():
    """The plain attention with inputs made so that one key stands out: the first position of a chunk is seen by the
    chunk's last query and by no query of the next chunk."""
    n, size = 24, 8
    m = dict(heads=1, kv_heads=1, dim=4, vdim=2, mask=dict(size=size), scale=4.0, softcap=50.0)
    h = torch.zeros(n, 3)
    h[:, 0] = 1.0                      # every token: the same query direction
    h[8, 1] = 1.0                      # position 8, a chunk's first: a key along the queries, a value of its own
    w = {"q": torch.tensor([[1.0, 0, 0], [0, 0, 0], [0, 0, 0], [0, 0, 0]]), "q.b": torch.zeros(4),
         "k": torch.tensor([[0, 1.0, 0], [0.3, 0, 0], [0, 0, 0], [0, 0, 0]]), "k.b": torch.zeros(4),
         "v": torch.tensor([[0, 1.0, 0], [1.0, 0, 0]]), "v.b": torch.zeros(2), "g": torch.full((1, 3), 5.0),
         "o": torch.eye(2)}
    out = plain.chunked_attention(h, w, m, 1e-6)
    assert out[15, 0] > 0.9 and out[9, 0] > 0.9           # seen from the chunk's own last position, and from nearby
    assert out[16, 0].abs() < 1e-6 and out[7, 0].abs() < 1e-6      # not from the next chunk, nor from before


# us in the kernel that shares keys through LDS and in the one whose waves fetch their own, on 256 compute units:
# (heads, kv heads, maps, key width, value width, window), [(tokens, tokens before them)], shared, tiles
PORTIONS_MEASURED = [
    ((16, 4, 1, 128, 128, None), [(1024, 0)], 39, 38), ((16, 4, 1, 128, 128, None), [(2048, 0)], 75, 116),
    ((16, 4, 1, 128, 128, None), [(1024, 6000)], 233, 403), ((16, 4, 1, 128, 128, 1024), [(1024, 8000)], 41, 74),
    ((16, 4, 1, 128, 128, None), [(128, 0)] * 8, 10, 15), ((16, 4, 1, 128, 128, None), [(900, 0), (124, 6000)], 205, 175),
    ((32, 8, 1, 128, 128, None), [(512, 0)], 22, 25), ((32, 8, 1, 128, 128, None), [(512, 2048)], 89, 153),
    ((64, 8, 1, 128, 128, None), [(280, 0)], 16, 22), ((16, 16, 1, 64, 64, None), [(1024, 0)], 31, 28),
    ((16, 16, 1, 64, 64, None), [(256, 0)] * 4, 12, 14), ((16, 4, 1, 64, 64, None), [(1280, 0)], 38, 32),
    ((16, 4, 1, 64, 64, None), [(2048, 0)], 59, 68), ((16, 4, 1, 64, 64, None), [(1024, 4000)], 134, 142),
    ((16, 8, 2, 64, 128, 1024), [(512, 6000)], 40, 50), ((16, 4, 1, 32, 32, None), [(1024, 0)], 30, 17),
    ((16, 4, 1, 32, 32, None), [(1280, 0)], 36, 25), ((16, 4, 1, 32, 32, None), [(2048, 0)], 55, 49),
    ((16, 4, 1, 32, 32, None), [(1024, 4000)], 129, 111), ((32, 8, 1, 32, 32, None), [(2048, 0)], 55, 95),
    ((16, 4, 1, 32, 128, None), [(1280, 0)], 43, 39), ((16, 16, 1, 128, 64, None), [(1280, 0)], 42.6, 44.5)]


@pytest.mark.parametrize("sizes,portions,shared,tiles", PORTIONS_MEASURED)
def test_portions_go_to_the_faster_attention_kernel(sizes, portions, shared, tiles):
    """Whichever kernel the rule takes is within a twentieth of the faster one's measured time."""
    from ampere_kv_engine_amd.kernels.hip_parts import shared_blocks, shares_keys
    heads, kv_heads, maps, dim, vdim, window = sizes
    held = [(count, before + count) for count, before in portions]
    assert shared_blocks(held, heads * maps, kv_heads, maps) >= 256
    chosen = shared if shares_keys(256, held, heads * maps, kv_heads, maps, dim, vdim, window, None) else tiles
    assert chosen <= 1.05 * min(shared, tiles)


@pytest.mark.parametrize("vectors,kv_heads,maps,dim,vdim", [(64, 8, 1, 128, 128), (32, 8, 1, 128, 128), (64, 64, 1, 32, 32), (32, 8, 2, 64, 128)])
@pytest.mark.parametrize("window", [None, 40, 1024])
def test_a_recorded_step_goes_where_the_same_step_goes_unrecorded(vectors, kv_heads, maps, dim, vdim, window):
    """Steps of the sizes that may be recorded: their requests' lengths - as they are, or bounds - do not turn the choice.  Larger
    steps go by their lengths."""
    from types import SimpleNamespace
    from ampere_kv_engine_amd.config import EngineConfig
    from ampere_kv_engine_amd.kernels.hip_parts import PartsKernels
    kernels = PartsKernels.__new__(PartsKernels)
    kernels.compute_units = 256
    assert kernels.FEW_TOKENS == EngineConfig().record_max_tokens
    heads, seen = (vectors, kv_heads, maps, dim, vdim), set()
    for singles, counts in ((0, [512]), (0, [280]), (3, [300]), (1, [200, 311]), (2, [64] * 7)):
        starts = [0]
        for count in [1] * singles + counts:
            starts.append(starts[-1] + count)
        choices = set()
        for before in (0, 37, 2048, 30000):
            lengths = [before + 1] * singles + [before + count for count in counts]
            for bound in (None, 2048, 65536):
                ctx = SimpleNamespace(num_seqs=len(lengths), host_q_start=starts,
                                      host_seq_lens=lengths if bound is None else [65536] * singles + [bound] * len(counts))
                choices.add(kernels._shares_attention_keys(ctx, singles, heads, window, None))
                assert kernels._shares_attention_keys(ctx, singles, heads, window, None) in choices
        assert len(choices) == 1
        seen |= choices
    assert all(blocks >= 256 for blocks, shared in seen if shared)
    fresh, late = (kernels._shares_attention_keys(SimpleNamespace(num_seqs=1, host_q_start=[0, 1024], host_seq_lens=[length]), 0,
                                                  (16, 4, 1, 128, 128), None, None) for length in (1024, 7024))
    assert fresh == (256, False) and late == (256, True)


def test_requests_without_tokens_add_nothing_to_the_choice():
    """A request of a step may bring no token (a caller of the kernels alone): it makes no block and takes no time."""
    from ampere_kv_engine_amd.kernels.hip_parts import shared_blocks, shares_keys
    heads = (16, 4, 1, 128, 128)
    for portions in ([(2048, 2048)], [(1024, 7024)], [(900, 900), (124, 6124)]):
        for empty in ((0, 0), (0, 5000)):
            assert shared_blocks(portions + [empty], *heads[:3]) == shared_blocks(portions, *heads[:3])
            for window in (None, 1024):
                for order in (portions + [empty], [empty] + portions):
                    assert shares_keys(256, order, *heads, window, None) == shares_keys(256, portions, *heads, window, None)


@pytest.mark.parametrize("allowed", [64, 512, 513, 1024, 4096])
def test_an_engine_that_records_longer_portions_sends_them_the_same_way(allowed):
    """The line between steps that look at lengths and steps that do not follows what their engine may record."""
    from types import SimpleNamespace
    from ampere_kv_engine_amd.kernels.hip_parts import PartsKernels
    kernels = PartsKernels.__new__(PartsKernels)
    kernels.compute_units, turned = 256, False
    for heads in ((16, 4, 1, 128, 128), (64, 8, 1, 128, 128), (32, 8, 2, 64, 128)):
        for tokens in (280, 512, 513, 900, 1024, 1025):
            choices = {kernels._shares_attention_keys(
                SimpleNamespace(num_seqs=1, host_q_start=[0, tokens], host_seq_lens=[length], recordable_tokens=allowed),
                0, heads, None, None) for length in (tokens, tokens + 300, 2048, 7000, 65536)}
            turned |= len(choices) > 1
            assert len(choices) == 1 or tokens > max(allowed, 512)
    assert turned == (allowed < 1025)


# us in the faster of those two kernels and on the plain prompt attention's tiles, and whether the tiles are taken: steps that may be
# recorded (up to 512 tokens) are chosen as if as much lay before their portions as they bring, whatever does
PROMPT_TILES_MEASURED = [
    ((16, 4, 1, 128, 128, None), [(64, 0)], 6.5, 10.5, False), ((16, 4, 1, 128, 128, None), [(256, 0)], 11.9, 15.6, False),
    ((16, 4, 1, 128, 128, None), [(512, 0)], 20.5, 20.8, False), ((16, 4, 1, 128, 128, None), [(1024, 0)], 41, 32, True),
    ((16, 4, 1, 128, 128, None), [(2000, 0)], 76, 53, True), ((16, 4, 1, 128, 128, None), [(512, 2048)], 83, 61, False),
    ((16, 4, 1, 128, 128, None), [(1024, 6000)], 242, 157, True), ((16, 4, 1, 128, 128, None), [(500, 0)] * 4, 30, 22, True),
    ((16, 4, 1, 128, 128, None), [(128, 0)] * 8, 11.1, 13.3, False), ((16, 4, 1, 128, 128, 512), [(2000, 0)], 34, 28, True),
    ((16, 4, 1, 128, 128, 512), [(1024, 0)], 26.0, 25.8, True), ((32, 8, 1, 128, 128, None), [(2000, 0)], 84, 63, True),
    ((32, 8, 1, 128, 128, None), [(500, 0)] * 4, 40, 29, False), ((16, 4, 2, 64, 128, 1024), [(512, 0)], 22.3, 19.4, True),
    ((16, 4, 2, 64, 128, 1024), [(1024, 0)], 40, 31, True), ((16, 4, 2, 64, 128, 1024), [(2000, 0)], 59, 47, True),
    ((16, 4, 2, 64, 128, 1024), [(1024, 6000)], 51, 37, True), ((16, 4, 1, 64, 64, None), [(512, 0)], 14.4, 15.0, False),
    ((16, 4, 1, 64, 64, None), [(1024, 0)], 27, 23, True), ((16, 4, 1, 64, 64, None), [(2000, 0)], 60, 39, True),
    ((16, 4, 1, 64, 64, None), [(1024, 6000)], 189, 112, True), ((16, 16, 1, 64, 64, None), [(2000, 0)], 60, 39, True)]


def _prompt_tiles_chosen(sizes, portions, lengths=None, allowed=0, singles=0):
    from types import SimpleNamespace
    from ampere_kv_engine_amd.kernels.hip import HipKernels
    kernels = HipKernels.__new__(HipKernels)
    kernels.compute_units, kernels._attention_entry = 256, {("prompt tiles", 64): True, ("prompt tiles", 128): True}
    heads, kv_heads, maps, dim, vdim, window = sizes
    starts = [0]
    for count in [1] * singles + [count for count, _ in portions]:
        starts.append(starts[-1] + count)
    held = [9000] * singles + [before + count for count, before in portions] if lengths is None else lengths
    ctx = SimpleNamespace(num_seqs=len(held), host_q_start=starts, host_seq_lens=held, seq_lens=object(), recordable_tokens=allowed)
    chosen = kernels._takes_prompt_tiles(ctx, singles, (heads * maps, kv_heads, maps, dim, vdim), window, 16)
    assert kernels._takes_prompt_tiles(ctx, singles, (heads * maps, kv_heads, maps, dim, vdim), window, 16) == chosen
    return chosen


@pytest.mark.parametrize("sizes,portions,others,tiles,taken", PROMPT_TILES_MEASURED)
def test_portions_go_to_prompt_tiles_where_they_are_faster(sizes, portions, others, tiles, taken):
    """The choice as it stands, never for the slower kernel of the two where the tiles are it; the order of requests, requests without
    tokens and single tokens in front do not turn it."""
    assert not taken or tiles <= others
    for order in (portions, portions[::-1], portions + [(0, 0)], [(0, 5000)] + portions):
        assert _prompt_tiles_chosen(sizes, order) == taken
    if sum(count for count, _ in portions) > 512:
        assert _prompt_tiles_chosen(sizes, portions, singles=3) == taken


@pytest.mark.parametrize("allowed", [64, 512, 1024, 4096])
def test_recorded_steps_go_to_prompt_tiles_as_they_go_unrecorded(allowed):
    """Lengths - as they are, or bounds - do not turn the choice for a step that its engine may record; larger ones go by them."""
    turned, seen = False, set()
    for sizes in ((16, 4, 1, 128, 128, None), (16, 4, 2, 64, 128, 1024), (32, 8, 1, 64, 64, None)):
        for tokens in (200, 511, 512, 513, 1000, 1025):
            choices = {_prompt_tiles_chosen(sizes, [(tokens, 0)], lengths=[length], allowed=allowed)
                       for length in (tokens, tokens + 300, 2048, 7000, 65536)}
            seen |= choices
            turned |= len(choices) > 1
            assert len(choices) == 1 or tokens > max(allowed, 512)
    assert seen == {False, True} and (turned or allowed > 64)


def test_the_prompt_tiles_library_is_looked_for_by_bfloat16_engines_alone(monkeypatch):
    """A gated attention of float32, or of heads that the tiles do not take, asks for no library of a head size; where a bfloat16 one has
    none and none can be built, it says so once and its portions go to the other kernels."""
    from types import SimpleNamespace
    from ampere_kv_engine_amd.kernels import hip as module
    asked = []

    def absent(head_dim):
        asked.append(head_dim)
        raise RuntimeError("no compiler here")

    monkeypatch.setattr(module, "ensure_attention", absent)
    kernels = module.HipKernels.__new__(module.HipKernels)
    kernels._attention_entry, kernels.compute_units = {}, 256
    for dtype in (torch.float32, torch.bfloat16):
        kernels.check_gated_attention_sizes(16, 4, 128, 128, 16)
        kernels.find_gated_attention(1, 128, 128, 16, torch.float32)
        kernels.find_gated_attention(1, 128, 64, 16, dtype)
        kernels.find_gated_attention(1, 128, 128, 8, dtype)
    assert not asked
    with pytest.warns(UserWarning, match="no compiler here"):
        kernels.find_gated_attention(1, 128, 128, 16, torch.bfloat16)
    ctx = SimpleNamespace(num_seqs=1, host_q_start=[0, 2000], host_seq_lens=[2000], seq_lens=object())
    assert not kernels._takes_prompt_tiles(ctx, 0, (16, 4, 1, 128, 128), None, 16) and asked == [128]
    kernels._attention_entry[("prompt tiles", 128)] = True
    assert kernels._takes_prompt_tiles(ctx, 0, (16, 4, 1, 128, 128), None, 16)


def test_every_step_says_what_its_engine_may_record(engine, case):
    T.case_whole(engine, case)
    assert engine._last_step.recordable_tokens == engine.config.record_max_tokens
