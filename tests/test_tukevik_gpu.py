"""Tukevik on the GPU: every kernel of its own against the plain implementation's function of the same mechanism, and
the engine with the HIP kernels through the cuttings of `tukevik_cases` - float32 against tight limits, bfloat16 as
it is served."""

import json
import math
import os
import random
import subprocess
import sys
from types import SimpleNamespace

import pytest
import torch

import schedules
import tukevik_cases as T
from conftest import ROOT, random_ids
from plain import tukevik_plain as plain

pytestmark = pytest.mark.gpu
DEVICE = "cuda:0"


@pytest.fixture(scope="module")
def hip():
    from ampere_kv_engine_amd.kernels.hip import HipKernels
    return HipKernels(DEVICE)


@pytest.fixture(scope="module", params=list(T.TUKEVIK))
def case(request, tmp_path_factory):
    return T.make_case(request.param, str(tmp_path_factory.mktemp(f"tukevik_{request.param}")))


@pytest.fixture(scope="module", params=["float32", "bfloat16"])
def engine(request, case):
    return T.make_engine(case, request.param, DEVICE)


@pytest.mark.filterwarnings("ignore:a bfloat16 matrix")
@pytest.mark.parametrize("cutting", T.CUTTINGS, ids=lambda f: f.__name__)
def test_cutting(engine, case, cutting):
    if cutting is T.case_greedy_generation and engine.config.dtype != "float32":
        pytest.skip("greedy tokens are compared with the plain float32 implementation's")
    cutting(engine, case)
    assert engine.kernels.parts_library_path.endswith("libakv_parts.so")


@pytest.mark.filterwarnings("ignore:a bfloat16 matrix")
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("mechanism", T.MECHANISMS)
def test_one_mechanism_alone(mechanism, dtype, tmp_path):
    case = T.make_case(mechanism, str(tmp_path), T.alone(mechanism))
    engine = T.make_engine(case, dtype, DEVICE)
    T.case_whole(engine, case)
    T.case_prefill_then_token_by_token(engine, case)
    T.case_portions_down_to_two_tokens(engine, case)
    T.case_mixed_with_pages_and_slots_used_again(engine, case)


def test_steps_are_recorded_and_replayed(case):
    """Decode steps come again and again: the second is recorded, the later ones are replays; all agree with the plain
    implementation, and an engine that records nothing gives the same bits."""
    ids = case["requests"]["d"]
    want = case["expected"]["d"]
    outs = {}
    for graphs in (True, False):
        engine = T.make_engine(case, "float32", DEVICE, decode_graphs=graphs)
        got, _ = schedules.run(engine, {"d": ids}, schedules.last_one_by_one({"d": ids}, 60))
        T.assert_close(got["d"], want, "float32", f"graphs {graphs}")
        outs[graphs] = got["d"]
        if graphs:
            assert any(g is not None for g in engine._graphs.values()), "nothing was recorded"
    assert torch.equal(outs[True], outs[False])


def test_portions_whose_shape_comes_again_are_recorded(tmp_path):
    """Portions of 32 tokens, again and again, beside a request's single tokens - retention over chunks with a state of
    128 x 128 (its kernels ask for more than 64 KB of LDS), the matrix-core attention, the scan cut into runs: the
    recorded steps give the bits of an engine that records nothing, in both arithmetics."""
    raw = dict(architecture="Tukevik", vocab=200, width=64, norm=dict(eps=1e-6), residual_mult=0.9, layers=[
        dict(type="parallel", mlp=T.DENSE(64),
             mixer=T.PARALLEL(T.LEFT(4, 2, 64, 64, 50, 0.8, 10.0), T.RIGHT(1, 128, 128, [0.99], 64, 1e4), 1.0, 1.0)),
        dict(type="rglru", mixer=T.RGLRU(96, 2, 3), mlp=T.MOE(4, 2, 16, 16))])
    case = T.make_case("recorded portions", str(tmp_path), (raw, 41, 16))
    from ampere_kv_engine_amd.engine import StepEntry
    ids, single = case["requests"]["d"], case["requests"]["b"]
    for dtype in ("float32", "bfloat16"):
        outs = {}
        for graphs in (True, False):
            engine = T.make_engine(case, dtype, DEVICE, decode_graphs=graphs)
            d, b = engine.open("d"), engine.open("b")
            rows = []
            for step in range(3):          # a step is recorded when its shape comes again; each asks for two rows
                logits = engine.step([StepEntry(d, ids[32 * step:32 * step + 32], [31]), StepEntry(b, single[step:step + 1], [0])])
                rows.append(logits.float().cpu())
            engine.close(d), engine.close(b)
            got = torch.cat(rows)
            want = torch.stack([row for step in range(3) for row in (case["expected"]["d"][32 * step + 31], case["expected"]["b"][step])])
            T.assert_close(got, want, dtype, f"{dtype}, graphs {graphs}")
            outs[graphs] = got
            if graphs:
                assert any(g is not None for g in engine._graphs.values()), "nothing was recorded"
        assert torch.equal(outs[True], outs[False])


def test_trace_replay_of_a_random_model(case, tmp_path):
    """bin/trace_run on a configuration file and a seed: the mixed cutting, every position against the plain model."""
    from ampere_kv_engine_amd.config import TukevikConfig
    from ampere_kv_engine_amd.weights import write_random_model
    import numpy as np
    config_path = tmp_path / "config.json"
    config_path.write_text(json.dumps(case["raw"]))
    folder = write_random_model(str(tmp_path / "model"), TukevikConfig.from_dict(case["raw"]), 9)
    requests = {name: case["requests"][name] for name in ("a", "b", "e")}
    schedule = schedules.mixed(requests, T.PROMPTS, 16, 64, seed=3)
    out = tmp_path / "out"
    lines = "\n".join(json.dumps(r) for r in schedules.to_trace(requests, schedule)) + "\n"
    done = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--random-config", str(config_path),
                           "--weights-seed", "9", "--dtype", "float32", "--out", str(out), "--max-tokens", "1024"],
                          input=lines, capture_output=True, text=True, timeout=600)
    assert done.returncode == 0, done.stderr[-2000:]
    assert [l for l in done.stdout.splitlines() if l.startswith("done")] == [f"done {i}" for i in range(len(schedule))]
    fed = {name: 0 for name in requests}
    for number, (entries, _) in enumerate(schedule):
        got = torch.from_numpy(np.fromfile(out / f"{number}.f32", dtype="<f4").reshape(-1, case["raw"]["vocab"]).copy())
        row = 0
        for name, count in entries:
            want = T.plain_logits(folder, requests[name][:fed[name] + count])[fed[name]:]
            T.assert_close(got[row:row + count], want, "float32", f"step {number} request {name}")
            fed[name] += count
            row += count


def test_the_command_line_generates_with_a_tukevik_model(case, tmp_path):
    """`python -m ampere_kv_engine_amd.runner` on a configuration file and a seed: one request, and several through the
    scheduler, greedy; the tokens of the plain implementation.  `--mode check` holds the serving arithmetic against
    the engine's 32-bit path."""
    import re
    from ampere_kv_engine_amd.config import TukevikConfig
    from ampere_kv_engine_amd.weights import write_random_model
    config_path = tmp_path / "config.json"
    config_path.write_text(json.dumps(case["raw"]))
    folder = write_random_model(str(tmp_path / "model"), TukevikConfig.from_dict(case["raw"]), 5)
    prompts = [case["requests"]["a"][:19], case["requests"]["b"][:6], case["requests"]["c"][:31]]
    want = [T.plain_greedy(folder, ids, 6) for ids in prompts]
    base = [sys.executable, "-m", "ampere_kv_engine_amd.runner", "--random-config", str(config_path), "--weights-seed", "5",
            "--max-new-tokens", "6", "--ignore-eos"]
    run = lambda more: subprocess.run(base + more, capture_output=True, text=True, timeout=600, cwd=ROOT)
    one = run(["--mode", "generate", "--dtype", "float32", "--prompt-ids", " ".join(map(str, prompts[0])), "--prefill-chunk", "8"])
    assert one.returncode == 0, one.stderr[-2000:]
    assert json.loads(re.search(r"generated_token_ids = (\[.*\])", one.stdout).group(1)) == want[0]
    prompts_file = tmp_path / "prompts.txt"
    prompts_file.write_text("\n".join(" ".join(map(str, ids)) for ids in prompts) + "\n")
    many = run(["--mode", "generate", "--dtype", "float32", "--prompts-file", str(prompts_file), "--max-seqs", "2",
                "--prefill-chunk", "5"])
    assert many.returncode == 0, many.stderr[-2000:]
    got = [json.loads(line)["generated_token_ids"] for line in many.stdout.splitlines() if line.startswith("{")]
    assert got == want, many.stdout
    check = run(["--mode", "check", "--prompt-len", "40"])
    assert check.returncode == 0, check.stdout[-1500:] + check.stderr[-1500:]


def random_configuration(seed: int) -> tuple:
    """Sizes, constants and the order of layers drawn from a seed: any head counts and groupings, keys and values of
    different widths (some no multiple of 8), chunks from one position to longer than a request, any number of blocks
    and taps, layers without a feed-forward, routing with and without a shared expert."""
    rng = random.Random(seed)
    layers = []
    for _ in range(rng.choice((2, 3, 4, 5))):
        mlp = rng.choice((None, "dense", "moe", "moe"))
        if mlp == "dense":
            mlp = T.DENSE(rng.choice((40, 64, 100, 136)))
        elif mlp == "moe":
            experts = rng.choice((1, 2, 3, 5, 8, 17))
            mlp = T.MOE(experts, rng.randint(1, experts), rng.choice((8, 12, 32)), rng.choice((None, 8, 20, 48)))
        if rng.random() < 0.45:
            blocks = rng.choice((1, 2, 3, 4, 8))
            layers.append(dict(type="rglru", mlp=mlp, mixer=T.RGLRU(blocks * rng.choice((4, 8, 20, 32)), blocks, rng.choice((1, 2, 3, 4, 5)))))
            continue
        kv, group = rng.choice((1, 2, 3)), rng.choice((1, 2, 4, 5))
        left = T.LEFT(kv * group, kv, rng.choice((8, 12, 32, 64, 80)), rng.choice((4, 8, 24, 64, 72)),
                      rng.choice((1, 2, 5, 16, 31, 64, 100, 500)), rng.uniform(0.3, 1.2), rng.choice((2.0, 10.0, 30.0)))
        heads, dim = rng.choice((1, 2, 3, 5)), rng.choice((8, 12, 32, 64))
        right = T.RIGHT(heads, dim, rng.choice((4, 8, 24, 40)), [rng.choice((0.5, 0.9, 0.99, 0.999, 1.0)) for _ in range(heads)],
                        rng.choice([d for d in (2, 4, 8, 12, 32, 64) if d <= dim]), rng.choice((100.0, 1e4, 1e6)))
        layers.append(dict(type="parallel", mlp=mlp, mixer=T.PARALLEL(left, right, rng.uniform(0.3, 1.5), rng.uniform(0.3, 1.5))))
    raw = dict(architecture="Tukevik", vocab=rng.choice((97, 260, 1000)), width=rng.choice((40, 72, 96, 136, 192)),
               norm=dict(eps=rng.choice((1e-5, 1e-6))), residual_mult=rng.choice((0.3, 0.5, 1.0, 1.4)), layers=layers)
    return raw, seed, rng.choice((4, 8, 16, 32))


@pytest.mark.filterwarnings("ignore:a bfloat16 matrix")
@pytest.mark.parametrize("seed", range(500, 508))
def test_a_random_configuration_through_the_cuttings(seed, tmp_path):
    config = random_configuration(seed)
    print(f"seed {seed}: {config[0]}, pages of {config[2]}", flush=True)
    case = T.make_case(f"random {seed}", str(tmp_path), config)
    for dtype in ("float32", "bfloat16"):
        engine = T.make_engine(case, dtype, DEVICE)
        T.case_whole(engine, case)
        T.case_portions_down_to_two_tokens(engine, case)
        T.case_prefill_then_token_by_token(engine, case)
        T.case_mixed_with_pages_and_slots_used_again(engine, case)


# ---- the kernels one by one, against the plain functions ----------------------------------------------------------------

def _ctx(lengths_before, counts, device=DEVICE):
    """What the kernels read of a step: requests that hold `lengths_before` tokens and bring `counts` more."""
    q_start, positions, seq_of_token = [0], [], []
    for r, (before, count) in enumerate(zip(lengths_before, counts)):
        q_start.append(q_start[-1] + count)
        positions += list(range(before, before + count))
        seq_of_token += [r] * count
    ints = lambda values: torch.tensor(values, dtype=torch.int32, device=device)
    seqs = len(counts)
    singles = next((r for r, count in enumerate(counts) if count != 1), seqs)        # single tokens come first in a step
    return SimpleNamespace(num_decode_seqs=singles, max_new_tokens=max(counts), num_seqs=seqs, num_tokens=q_start[-1], q_start=ints(q_start), positions=ints(positions),
                           seq_of_token=ints(seq_of_token), seq_slots=ints(list(range(seqs))), host_q_start=q_start,
                           host_seq_slots=list(range(seqs)), host_seq_lens=[b + c for b, c in zip(lengths_before, counts)],
                           max_seq_len=max(b + c for b, c in zip(lengths_before, counts)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,chunk,page", [(4, 2, 16, 24, 11, 4), (3, 1, 40, 8, 64, 16), (8, 8, 64, 64, 7, 8),
                                                               (2, 1, 128, 256, 300, 16), (8, 2, 64, 32, 20, 16),
                                                               (4, 4, 32, 128, 48, 32), (1, 1, 64, 64, 5000, 16),
                                                               (2, 1, 256, 32, 40, 16)])
def test_attention_kernel_alone(hip, dtype, heads, kv_heads, dim, vdim, chunk, page):
    """Two requests in two portions each, through the unit norm with its cache write and the attention, against the plain
    attention of the whole sequences.  Scores are made sharp, and one key a request - the first of a chunk - is made to
    stand out for every later query: it counts up to its chunk's last position and not beyond."""
    torch.manual_seed(heads * 100 + dim)
    lengths, eps, scale, softcap = (75, 2 * chunk + 3 if chunk < 100 else 330 if chunk < 1000 else 2100), 1e-6, 1.2, 9.0
    m = dict(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, mask=dict(size=chunk), scale=scale, softcap=softcap)
    width = heads * dim + kv_heads * (dim + vdim) + heads
    rows = [torch.randn(n, width) for n in lengths]
    for projected, n in zip(rows, lengths):
        needle = min(chunk, n - 2) if chunk < n else 0
        projected[needle, heads * dim:heads * dim + kv_heads * dim] = projected[needle + 1:, :dim].mean(0).repeat(kv_heads) * 30
    rows = [r.to(dtype).float() for r in rows]
    pages_needed = sum((n + page - 1) // page for n in lengths)
    k_pages = torch.zeros(pages_needed + 2, kv_heads, page, dim, dtype=dtype, device=DEVICE)
    v_pages = torch.zeros(pages_needed + 2, kv_heads, vdim, page, dtype=dtype, device=DEVICE)
    order = torch.randperm(pages_needed + 2).tolist()
    table = torch.full((2, max((n + page - 1) // page for n in lengths)), -1, dtype=torch.int32)
    for r, n in enumerate(lengths):
        for i in range((n + page - 1) // page):
            table[r, i] = order.pop()
    got = [torch.zeros(n, heads * vdim) for n in lengths]
    # two portions each, then the last token of each alone (sixteen waves share a row whose request is long)
    for step, befores in enumerate([(0, 0), (41, 5), (lengths[0] - 1, lengths[1] - 1)]):
        counts = [[41, 5], [lengths[0] - 42, lengths[1] - 6], [1, 1]][step]
        ctx = _ctx(befores, counts)
        projected = torch.cat([rows[r][b:b + c] for r, (b, c) in enumerate(zip(befores, counts))]).to(dtype).to(DEVICE)
        slot_map = torch.tensor([int(table[r, p // page]) * page + p % page for r, (b, c) in enumerate(zip(befores, counts))
                                 for p in range(b, b + c)], dtype=torch.int32, device=DEVICE)
        meta = SimpleNamespace(block_table=table.to(DEVICE), rows=None, width=table.shape[1], slot_map=slot_map)
        q = torch.empty(ctx.num_tokens, heads * dim, dtype=dtype, device=DEVICE)
        out = torch.empty(ctx.num_tokens, heads * vdim, dtype=dtype, device=DEVICE)
        hip.unit_norm_write(projected, heads, kv_heads, dim, vdim, eps, slot_map, k_pages, v_pages, q)
        hip.gated_attention(q, k_pages, v_pages, projected, heads * dim + kv_heads * (dim + vdim), ctx, meta, heads, kv_heads,
                            dim, vdim, scale, softcap, chunk, None, True, out)
        at = 0
        for r, (b, c) in enumerate(zip(befores, counts)):
            got[r][b:b + c] = out[at:at + c].float().cpu()
            at += c
    for r, n in enumerate(lengths):
        x = rows[r]
        qk = heads * dim + kv_heads * dim
        identity = lambda size: torch.eye(size)
        # the plain function with identity projections: its input IS the projected row, cut by selecting matrices
        pick = lambda lo, hi: torch.eye(width)[lo:hi]
        w = {"q": pick(0, heads * dim), "q.b": torch.zeros(heads * dim), "k": pick(heads * dim, qk), "k.b": torch.zeros(kv_heads * dim),
             "v": pick(qk, qk + kv_heads * vdim), "v.b": torch.zeros(kv_heads * vdim), "g": pick(qk + kv_heads * vdim, width),
             "o": identity(heads * vdim)}
        want = plain.chunked_attention(x, w, m, eps)
        limit = 2e-5 if dtype == torch.float32 else 0.03
        error = (got[r] - want).abs().max() / want.abs().max()
        assert error < limit, f"request {r}: {error:.2e}"


SINGLES = [     # heads, kv heads, dim, vdim, page, maps, options
    (4, 2, 32, 32, 16, 1, dict(softcap=9.0, chunk=48, sink="zero", gates=True)), (16, 4, 128, 128, 16, 1, dict(sink="learned")),
    (8, 8, 64, 256, 32, 1, dict(window=700)), (6, 2, 64, 128, 16, 2, dict(window=33)), (20, 1, 128, 64, 48, 1, dict(chunk=300)),
    (8, 2, 256, 128, 16, 1, dict(window=40, keep_first=20)), (36, 2, 32, 64, 16, 1, dict(bias=True, sink="zero")), (2, 1, 256, 256, 16, 1, dict())]


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,page,maps,options", SINGLES)
def test_single_tokens_on_the_matrix_cores(hip, heads, kv_heads, dim, vdim, page, maps, options):
    """Single tokens whose keys end at every edge of a step, of a wave's share and of a segment, and the same in the kernel that
    takes a wave's tiles in turn: both against the double.  Weights are exact in float32 in all of them, so what is left is one
    rounding of an output - two results on either side of a rounding's edge lie one unit in the last of eight bits apart, at
    most 2^-7 of them - and float32 sums (1e-4).  Slots beyond a request's tokens
    hold NaN; one key of weight zero has an infinite value, which nobody takes."""
    from torch_kernels import TorchKernels
    torch.manual_seed(dim + heads)
    befores = [0, 1, 15, 16, 62, 63, 64, 255, 256, 257, 300, 511, 512, 1037]
    counts = [1] * len(befores)
    ctx = _ctx(befores, counts)
    need = [(b + page) // page for b in befores]
    order = torch.randperm(sum(need) + 2).tolist()
    table = torch.full((len(befores), max(need)), -1, dtype=torch.int32)
    k_pages = torch.full((sum(need) + 2, kv_heads, page, maps * dim), float("nan"))
    v_pages = torch.full((sum(need) + 2, kv_heads, vdim, page), float("nan"))
    for r, before in enumerate(befores):
        for p in range(before + 1):
            if p % page == 0:
                table[r, p // page] = order.pop()
            at = int(table[r, p // page])
            k_pages[at, :, p % page], v_pages[at, :, :, p % page] = torch.randn(kv_heads, maps * dim), torch.randn(kv_heads, vdim)
    vectors = heads * maps
    q = torch.randn(len(befores), vectors * dim).bfloat16()
    k_pages, v_pages = k_pages.bfloat16(), v_pages.bfloat16()
    width = vectors * vdim + 12
    gates = torch.randn(len(befores), vectors + 3).bfloat16() if options.get("gates") else None
    sinks = torch.randn(vectors) * 3 if options.get("sink") == "learned" else None
    bias = torch.rand(2, vectors) if options.get("bias") else None
    meta = SimpleNamespace(block_table=table.to(DEVICE), rows=None, width=table.shape[1])

    def through(kernels, device, v, c, m):
        out = torch.zeros(len(befores), width, dtype=torch.bfloat16, device=device)
        move = lambda t: t.to(device) if t is not None else None
        kernels.gated_attention(move(q), move(k_pages), move(v), move(gates), 2, c, m, heads, kv_heads, dim, vdim, 1.7 * dim ** -0.5,
                                options.get("softcap"), options.get("chunk"), options.get("window"), "sink" in options, out,
                                out_at=4, out_scale=0.7, sink_logits=move(sinks), maps=maps,
                                keep_first=options.get("keep_first", 0), distance_bias=move(bias))
        return out.float().cpu()

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = through(TorchKernels(), "cpu", v_pages, host, SimpleNamespace(block_table=table, rows=None, width=table.shape[1]))
    got = through(hip, DEVICE, v_pages, ctx, meta)
    portion = SimpleNamespace(**dict(vars(ctx), num_decode_seqs=0))          # (the same rows through the portions' kernel)
    assert ((got - want).abs() <= want.abs() * 2.0 ** -7 + 1e-4).all(), (got - want).abs().max()
    assert ((through(hip, DEVICE, v_pages, portion, meta) - want).abs() <= want.abs() * 2.0 ** -7 + 5e-3).all()
    if options or maps > 1:
        return
    # the last request's key 700 points away from every query by so much that its weight is zero; its value is infinite
    at, place = int(table[-1, 700 // page]), 700 % page
    k_pages[at, :, place] = -q[-1].view(heads, dim).float().sum(0).bfloat16() * 1000
    clean = through(hip, DEVICE, v_pages, ctx, meta)
    v_pages[at, :, :, place] = float("inf")
    assert torch.equal(through(hip, DEVICE, v_pages, ctx, meta)[:-1], clean[:-1])
    last = through(hip, DEVICE, v_pages, ctx, meta)[-1]
    assert torch.isfinite(last).all()
    assert ((last - clean[-1]).abs() <= clean[-1].abs() * 2.0 ** -7 + 1e-4).all()


@pytest.mark.parametrize("askew", ["q", "k_pages", "v_pages", "out"])
@pytest.mark.parametrize("counts", [[1, 1], [70, 3]])
def test_gated_attention_of_operands_that_are_not_aligned(hip, monkeypatch, askew, counts):
    """A tensor that begins one element behind the boundary that wide accesses need, as a view into a larger one may, goes to the
    plain kernel - single tokens and portions, whichever matrix-core kernel they would go to.  (2^-7 |out| + 2e-3 as above.)"""
    from torch_kernels import TorchKernels
    torch.manual_seed(9)
    heads, kv_heads, dim, vdim, page = 4, 2, 64, 32, 16
    ctx = _ctx([300, 17], counts)
    ctx.seq_lens = torch.tensor(ctx.host_seq_lens, dtype=torch.int32, device=DEVICE)
    pages = max(ctx.host_seq_lens) // page + 1
    table = torch.randperm(2 * pages, dtype=torch.int32).view(2, pages)
    given = dict(q=torch.randn(ctx.num_tokens, heads * dim), k_pages=torch.randn(2 * pages, kv_heads, page, dim),
                 v_pages=torch.randn(2 * pages, kv_heads, vdim, page), out=torch.zeros(ctx.num_tokens, heads * vdim))
    given = {name: t.bfloat16() for name, t in given.items()}

    def attend(kernels, device, c, q, k_pages, v_pages, out):
        meta = SimpleNamespace(block_table=table.to(device), rows=None, width=pages)
        kernels.gated_attention(q, k_pages, v_pages, None, 0, c, meta, heads, kv_heads, dim, vdim, 0.1, None, None, None, True, out)
        return out.float().cpu()

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = attend(TorchKernels(), "cpu", host, **given)
    given = {name: t.to(DEVICE) for name, t in given.items()}
    room = torch.empty(given[askew].numel() + 1, dtype=torch.bfloat16, device=DEVICE)
    given[askew] = room[1:].view(given[askew].shape).copy_(given[askew])
    assert given[askew].data_ptr() % 16 == 2
    for blocks in (1, 1 << 30):
        monkeypatch.setattr(hip, "shared_attention_blocks", blocks, raising=False)
        given["out"].zero_()
        assert ((attend(hip, DEVICE, ctx, **given) - want).abs() <= want.abs() * 2.0 ** -7 + 2e-3).all()


@pytest.mark.parametrize("singles,portions", [(63, []), (64, []), (65, [40, 2])])
def test_many_single_tokens_of_wide_heads_of_their_own(hip, singles, portions):
    """On both sides of the line from which single tokens whose heads have keys of their own and values of 256 go to the plain kernel
    (512 rows on 256 units), with portions behind them: against the double.  (2^-7 |out| + 2e-3 as above.)"""
    from torch_kernels import TorchKernels
    torch.manual_seed(singles)
    heads, dim, vdim, page = 8, 32, 256, 16
    ctx = _ctx([(37 * r) % 300 for r in range(singles)] + [20] * len(portions), [1] * singles + portions)
    ctx.seq_lens = torch.tensor(ctx.host_seq_lens, dtype=torch.int32, device=DEVICE)
    seqs, pages = ctx.num_seqs, max(ctx.host_seq_lens) // page + 1
    table = torch.randperm(seqs * pages, dtype=torch.int32).view(seqs, pages)
    k_pages = torch.randn(seqs * pages, heads, page, dim).bfloat16()
    v_pages = torch.randn(seqs * pages, heads, vdim, page).bfloat16()
    q, gates = torch.randn(ctx.num_tokens, heads * dim).bfloat16(), torch.randn(ctx.num_tokens, heads).bfloat16()

    def attend(kernels, device, c):
        out = torch.full((ctx.num_tokens, heads * vdim), float("nan"), dtype=torch.bfloat16, device=device)
        meta = SimpleNamespace(block_table=table.to(device), rows=None, width=pages)
        kernels.gated_attention(q.to(device), k_pages.to(device), v_pages.to(device), gates.to(device), 0, c, meta, heads, heads, dim, vdim,
                                0.2, None, None, None, True, out)
        return out.float().cpu()

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = attend(TorchKernels(), "cpu", host)
    assert ((attend(hip, DEVICE, ctx) - want).abs() <= want.abs() * 2.0 ** -7 + 2e-3).all()


@pytest.mark.parametrize("tokens_at_once", [1, 2, 5, 9])
@pytest.mark.parametrize("dim,vdim,window,keep_first", [(64, 128, None, 0), (128, 32, 6000, 40), (256, 256, None, 0)])
def test_single_tokens_whose_partial_sums_do_not_fit(hip, monkeypatch, tokens_at_once, dim, vdim, window, keep_first):
    """Nine single tokens of one to 33 segments whose partial sums would be more than a launch may leave: they are taken so many at
    a time through one buffer, and have the bits they have in one launch."""
    from ampere_kv_engine_amd.kernels import partial_sums
    torch.manual_seed(3)
    heads, kv_heads, page = 6, 2, 16
    befores = [8300, 0, 300, 255, 256, 4095, 17, 4096, 7000]
    ctx = _ctx(befores, [1] * 9)
    pages = max(befores) // page + 1
    table = torch.randperm(9 * pages, dtype=torch.int32).view(9, pages).to(DEVICE)
    meta = SimpleNamespace(block_table=table, rows=None, width=pages)
    k_pages = torch.randn(9 * pages, kv_heads, page, dim, device=DEVICE).bfloat16()
    v_pages = torch.randn(9 * pages, kv_heads, vdim, page, device=DEVICE).bfloat16()
    q, gates = torch.randn(9, heads * dim, device=DEVICE).bfloat16(), torch.randn(9, heads + 5, device=DEVICE).bfloat16()
    cuts, cut = [], partial_sums.gated_cut
    monkeypatch.setattr(partial_sums, "gated_cut", lambda *args: cuts.append(cut(*args)) or cuts[-1])

    def attend():
        out = torch.full((9, heads * vdim + 8), 7.0, dtype=torch.bfloat16, device=DEVICE)
        hip.gated_attention(q, k_pages, v_pages, gates, 3, ctx, meta, heads, kv_heads, dim, vdim, 0.1, None, None, window, True, out, out_at=4,
                            keep_first=keep_first)
        return out

    want = attend()
    floats = heads * cuts[0][0] * (vdim + 4)
    monkeypatch.setattr(partial_sums, "BYTES", 4 * floats * tokens_at_once)
    asked = []
    monkeypatch.setattr(partial_sums, "take", lambda ctx, count, device: asked.append(count) or torch.empty(count, device=device))
    assert torch.equal(attend(), want)
    assert [c[1] for c in cuts] == [9, tokens_at_once] and asked == [tokens_at_once * floats]


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,page,maps,eps,rot,keyed", [
    (4, 2, 64, 64, 16, 1, 1e-6, 0, False), (16, 4, 128, 128, 16, 1, None, 64, False), (2, 1, 40, 72, 8, 2, None, 16, False),
    (3, 3, 8, 8, 64, 1, 1e-5, 0, True), (1, 1, 512, 256, 32, 1, 1e-6, 512, False), (6, 2, 24, 200, 24, 1, None, 0, False)])
@pytest.mark.parametrize("lead", [0, 3, 8])
def test_norm_and_rotation_in_eights(hip, heads, kv_heads, dim, vdim, page, maps, eps, rot, keyed, lead):
    """Vectors whose widths come in eights, against the oracle on the same rows in float32: `lead` tokens of other requests and
    a portion of 29 - so that eight tokens are a run of a page, cross into one, or lie askew -, some tokens without a
    slot or beyond the pages, with and without the cache write.  Queries and keys: a rounding to bfloat16 is at most 2^-8 of the value, and float32's
    own roundings (a norm of at most 512 terms, a turn of two) at most 2^-16 of the magnitudes that meet; values the same bits;
    nothing else in the pages changes."""
    from torch_kernels import TorchKernels
    generator = torch.Generator().manual_seed(heads * 1000 + dim + lead)
    tokens, num_pages = lead + 29, 29 // page + 12
    columns = (heads + kv_heads) * maps * dim + (0 if keyed else kv_heads * vdim)
    rows = torch.randn(tokens, 16 + columns, generator=generator).bfloat16()
    positions = torch.randint(0, 300, (tokens,), generator=generator, dtype=torch.int32)
    slots = torch.cat([torch.arange(lead) * (page + 1) + 5 * page, torch.arange(29) + page]).int()
    slots[[lead + 9, tokens - 1]] = torch.tensor([-1, num_pages * page + 3], dtype=torch.int32)
    slots[:lead] += 29 // page * page + page * 2 - 5 * page + page
    slots[:lead] = torch.where(slots[:lead] < num_pages * page, slots[:lead], -1)
    angles = torch.rand(300, max(rot, 2) // 2, generator=generator) * 6
    table = torch.stack([angles.cos(), angles.sin()], -1).float() if rot else None
    more = dict(at=16, maps=maps, rot_dims=rot, keyed_values=keyed)
    k_pages = torch.full((num_pages, kv_heads, page, maps * dim), 7.0)
    v_pages = torch.full((num_pages, kv_heads, vdim, page), 7.0)
    want_q, oracle = torch.empty(tokens, heads * maps * dim), TorchKernels()
    oracle.unit_norm_write(rows.float(), heads, kv_heads, dim, vdim, eps, None, k_pages, v_pages, want_q, table=table,
                           positions=positions, **more)
    kept = (slots >= 0) & (slots < num_pages * page)
    got_k, got_v = k_pages.bfloat16().to(DEVICE), v_pages.bfloat16().to(DEVICE)
    oracle.unit_norm_write(rows[kept].float(), heads, kv_heads, dim, vdim, eps, slots[kept], k_pages, v_pages,
                           want_q[kept], table=table, positions=positions[kept], **more)
    for slot_map in (None, slots.to(DEVICE)):
        if slot_map is not None:
            assert (got_k == 7).all() and (got_v == 7).all()
        q = torch.empty(tokens, heads * maps * dim, dtype=torch.bfloat16, device=DEVICE)
        hip.unit_norm_write(rows.to(DEVICE), heads, kv_heads, dim, vdim, eps, slot_map, got_k, got_v, q,
                            table=table.to(DEVICE) if rot else None, positions=positions.to(DEVICE), **more)
        reach = 2.0 ** -16 * 2 * (want_q.abs().max())
        assert ((q.cpu().float() - want_q).abs() <= want_q.abs() * 2.0 ** -8 + reach).all()
    reach = 2.0 ** -16 * 2 * k_pages.abs().max()
    assert ((got_k.cpu().float() - k_pages).abs() <= k_pages.abs() * 2.0 ** -8 + reach).all()
    assert torch.equal(got_v.cpu().float(), v_pages)


@pytest.mark.parametrize("heads,kv_heads,dim,vdim,page,maps,options", [c for c in SINGLES if c[2] <= 128 and c[3] <= 128] + [
    (12, 4, 128, 128, 16, 1, dict(sink="learned", gates=True)), (3, 3, 64, 64, 64, 1, dict(window=70, keep_first=40)),
    (4, 2, 64, 128, 16, 2, dict(window=50, sink="zero"))])
def test_portions_that_share_their_keys_through_lds(hip, monkeypatch, heads, kv_heads, dim, vdim, page, maps, options):
    """Portions whose first and last columns fall inside tiles of 64, with and without history, beside single tokens - in the
    kernel that shares keys through LDS, whatever the number of blocks, and in the one in which every wave fetches its own: both
    against the double.  A weight is two bfloat16 (2^-17 of it is left out: times values of up to 5 sigma, below 1e-4 of the
    largest), an output is rounded once (an ulp apart at a rounding's edge: 2^-7 of it), exponentials are the hardware's (a
    few 2^-23 of scores of up to 60 in base 2): 2^-7 |out| + 2e-3.  Slots beyond a request's tokens hold NaN."""
    from torch_kernels import TorchKernels
    torch.manual_seed(dim + heads + vdim)
    befores, counts = [7, 0, 33, 300, 16, 0], [1, 1, 3, 90, 64, 331]
    ctx = _ctx(befores, counts)
    ctx.seq_lens = torch.tensor(ctx.host_seq_lens, dtype=torch.int32, device=DEVICE)
    need = [(n + page - 1) // page for n in ctx.host_seq_lens]
    order = torch.randperm(sum(need) + 2).tolist()
    table = torch.full((len(befores), max(need)), -1, dtype=torch.int32)
    k_pages = torch.full((sum(need) + 2, kv_heads, page, maps * dim), float("nan"))
    v_pages = torch.full((sum(need) + 2, kv_heads, vdim, page), float("nan"))
    for r, length in enumerate(ctx.host_seq_lens):
        for p in range(length):
            if p % page == 0:
                table[r, p // page] = order.pop()
            at = int(table[r, p // page])
            k_pages[at, :, p % page], v_pages[at, :, :, p % page] = torch.randn(kv_heads, maps * dim), torch.randn(kv_heads, vdim)
    vectors, tokens = heads * maps, ctx.num_tokens
    q = torch.randn(tokens, vectors * dim).bfloat16()
    k_pages, v_pages = k_pages.bfloat16(), v_pages.bfloat16()
    gates = torch.randn(tokens, vectors + 3).bfloat16() if options.get("gates") else None
    sinks = torch.randn(vectors) * 3 if options.get("sink") == "learned" else None
    bias = torch.rand(2, vectors) if options.get("bias") else None

    def through(kernels, device, c):
        out = torch.zeros(tokens, vectors * vdim + 12, dtype=torch.bfloat16, device=device)
        move = lambda t: t.to(device) if t is not None else None
        meta = SimpleNamespace(block_table=move(table), rows=None, width=table.shape[1])
        kernels.gated_attention(move(q), move(k_pages), move(v_pages), move(gates), 2, c, meta, heads, kv_heads, dim, vdim, 1.7 * dim ** -0.5,
                                options.get("softcap"), options.get("chunk"), options.get("window"), "sink" in options, out,
                                out_at=4, out_scale=0.7, sink_logits=move(sinks), maps=maps,
                                keep_first=options.get("keep_first", 0), distance_bias=move(bias))
        return out.float().cpu()

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = through(TorchKernels(), "cpu", host)
    for blocks in (1, 1 << 30):
        monkeypatch.setattr(hip, "shared_attention_blocks", blocks, raising=False)
        got = through(hip, DEVICE, ctx)
        assert ((got - want).abs() <= want.abs() * 2.0 ** -7 + 2e-3).all(), (blocks, (got - want).abs().max())


@pytest.mark.parametrize("singles,portions", [(0, 65), (3, 64), (5, 140)])
def test_portions_that_share_their_keys_of_many_requests(hip, monkeypatch, singles, portions):
    """A block finds its tile's request by adding up 64 requests' tiles at a time, from the first portion on: more of them than that,
    of uneven lengths, behind single tokens.  (2^-7 |out| + 2e-3 as above.)"""
    from torch_kernels import TorchKernels
    torch.manual_seed(portions)
    heads, kv_heads, dim, vdim, page = 6, 2, 32, 64, 16
    counts = [1] * singles + [2 + (7 * r) % 41 for r in range(portions)]
    ctx = _ctx([(29 * r) % 90 for r in range(len(counts))], counts)
    ctx.seq_lens = torch.tensor(ctx.host_seq_lens, dtype=torch.int32, device=DEVICE)
    seqs, pages = ctx.num_seqs, max(ctx.host_seq_lens) // page + 1
    table = torch.randperm(seqs * pages, dtype=torch.int32).view(seqs, pages)
    k_pages = torch.randn(seqs * pages, kv_heads, page, dim).bfloat16()
    v_pages = torch.randn(seqs * pages, kv_heads, vdim, page).bfloat16()
    q = torch.randn(ctx.num_tokens, heads * dim).bfloat16()

    def attend(kernels, device, c):
        out = torch.full((ctx.num_tokens, heads * vdim), float("nan"), dtype=torch.bfloat16, device=device)
        meta = SimpleNamespace(block_table=table.to(device), rows=None, width=pages)
        kernels.gated_attention(q.to(device), k_pages.to(device), v_pages.to(device), None, 0, c, meta, heads, kv_heads, dim, vdim, 0.2,
                                None, None, None, False, out)
        return out.float().cpu()

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = attend(TorchKernels(), "cpu", host)
    for blocks in (1, 1 << 30):
        monkeypatch.setattr(hip, "shared_attention_blocks", blocks, raising=False)
        assert ((attend(hip, DEVICE, ctx) - want).abs() <= want.abs() * 2.0 ** -7 + 2e-3).all(), blocks


@pytest.mark.parametrize("poison", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,maps,options", [
    (4, 4, 64, 64, 1, {}), (16, 4, 128, 128, 1, dict(sink=True)), (8, 2, 32, 64, 1, dict(softcap=9.0)), (4, 2, 64, 128, 2, dict(window=40)),
    (6, 2, 64, 32, 1, dict(chunk=48)), (2, 1, 128, 64, 1, dict(window=33, keep_first=20))])
def test_portions_that_share_their_keys_keep_clear_of_values_they_do_not_see(hip, monkeypatch, poison, heads, kv_heads, dim, vdim, maps,
                                                                             options):
    """One dimension of a position's value is infinite or NaN - a position inside a portion, one in its history, one among the
    kept first keys.  Tokens that do not see it share steps and tiles with tokens that do: they have the result without
    it in every dimension, as those that see it have in all dimensions but that one, which is not finite.  (2^-7 |out| + 2e-3 as
    for `test_portions_that_share_their_keys_through_lds`.)"""
    from torch_kernels import TorchKernels
    torch.manual_seed(dim + heads)
    page, befores, counts = 16, [0, 70], [131, 90]
    ctx = _ctx(befores, counts)
    ctx.seq_lens = torch.tensor(ctx.host_seq_lens, dtype=torch.int32, device=DEVICE)
    need = [(n + page - 1) // page for n in ctx.host_seq_lens]
    order, table = torch.randperm(sum(need)).tolist(), torch.full((2, max(need)), -1, dtype=torch.int32)
    for r, pages in enumerate(need):
        table[r, :pages] = torch.tensor([order.pop() for _ in range(pages)])
    k_pages = torch.randn(sum(need), kv_heads, page, maps * dim).bfloat16()
    v_pages = torch.randn(sum(need), kv_heads, vdim, page).bfloat16()
    vectors, tokens = heads * maps, ctx.num_tokens
    q = torch.randn(tokens, vectors * dim).bfloat16()
    window, chunk, kept = options.get("window"), options.get("chunk"), options.get("keep_first", 0)

    def through(kernels, device, values, c):
        out = torch.zeros(tokens, vectors * vdim, dtype=torch.bfloat16, device=device)
        meta = SimpleNamespace(block_table=table.to(device), rows=None, width=table.shape[1])
        kernels.gated_attention(q.to(device), k_pages.to(device), values.to(device), None, 0, c, meta, heads, kv_heads, dim, vdim, dim ** -0.5,
                                options.get("softcap"), chunk, window, options.get("sink", False), out, maps=maps, keep_first=kept)
        return out.float().cpu().view(tokens, vectors, vdim)

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = through(TorchKernels(), "cpu", v_pages, host)
    reach = want.abs() * 2.0 ** -7 + 2e-3
    monkeypatch.setattr(hip, "shared_attention_blocks", 1, raising=False)
    for request, at in ((0, 37), (0, 100), (1, 9), (1, 64), (1, 120)):
        values = v_pages.clone()
        values[int(table[request, at // page]), :, 3, at % page] = poison
        got = through(hip, DEVICE, values, ctx)
        pos = ctx.positions.cpu()
        sees = (ctx.seq_of_token.cpu() == request) & (pos >= at)
        inside = torch.ones_like(sees) if window is None else pos - at < window
        if chunk is not None:
            inside &= pos // chunk == at // chunk
        sees &= inside | (at < kept)
        assert not torch.isfinite(got[sees][:, :, 3]).any(), (request, at)
        got[sees, :, 3] = want[sees, :, 3]
        assert torch.isfinite(got).all(), (request, at)
        assert ((got - want).abs() <= reach).all(), (request, at)


@pytest.mark.parametrize("poison", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,maps,page,options", [
    (4, 4, 64, 64, 1, 16, {}), (16, 4, 128, 128, 1, 32, dict(sink=True)), (40, 1, 64, 64, 1, 64, dict(window=40)),
    (6, 2, 128, 128, 1, 16, dict(window=33, sink=True)), (4, 2, 64, 128, 2, 16, dict(window=40)), (3, 1, 64, 128, 2, 32, {}),
    (2, 2, 64, 128, 2, 64, dict(window=70))])
def test_portions_on_prompt_tiles_keep_clear_of_what_they_do_not_see(hip, monkeypatch, poison, heads, kv_heads, dim, vdim, maps, page, options):
    """As above on the plain prompt attention's tiles: one dimension of a position's value is not finite - inside a portion, in its history,
    the last position of a request -, and in every case keys and values of slots that no token sees are not finite at all: those
    behind a request's last token in its last page, and those that lie behind every token's window."""
    from torch_kernels import TorchKernels
    torch.manual_seed(dim + heads)
    befores, counts = [0, 170], [131, 90]
    ctx = _ctx(befores, counts)
    ctx.seq_lens = torch.tensor(ctx.host_seq_lens, dtype=torch.int32, device=DEVICE)
    need = [(n + page - 1) // page for n in ctx.host_seq_lens]
    order, table = torch.randperm(sum(need)).tolist(), torch.full((2, max(need)), -1, dtype=torch.int32)
    for r, pages in enumerate(need):
        table[r, :pages] = torch.tensor([order.pop() for _ in range(pages)])
    k_pages = torch.randn(sum(need), kv_heads, page, maps * dim).bfloat16()
    v_pages = torch.randn(sum(need), kv_heads, vdim, page).bfloat16()
    vectors, tokens, window = heads * maps, ctx.num_tokens, options.get("window")
    q = torch.randn(tokens, vectors * dim).bfloat16()

    def through(kernels, device, keys, values, c):
        out = torch.zeros(tokens, vectors * vdim, dtype=torch.bfloat16, device=device)
        meta = SimpleNamespace(block_table=table.to(device), rows=None, width=table.shape[1])
        kernels.gated_attention(q.to(device), keys.to(device), values.to(device), None, 0, c, meta, heads, kv_heads, dim, vdim, dim ** -0.5,
                                None, None, window, options.get("sink", False), out, maps=maps)
        return out.float().cpu().view(tokens, vectors, vdim)

    host = SimpleNamespace(**{k: (v.cpu() if isinstance(v, torch.Tensor) else v) for k, v in vars(ctx).items()})
    want = through(TorchKernels(), "cpu", k_pages, v_pages, host)
    reach = want.abs() * 2.0 ** -7 + 2e-3
    ctx.num_decode_seqs = 0
    monkeypatch.setattr(hip, "gated_prompt_tiles", True, raising=False)
    for r, length in enumerate(ctx.host_seq_lens):
        unseen = list(range(length, need[r] * page))
        if window is not None:
            unseen += range(max(befores[r] - window + 1, 0))
        for at in unseen:
            k_pages[int(table[r, at // page]), :, at % page] = poison
            v_pages[int(table[r, at // page]), :, :, at % page] = poison
    for request, at in ((None, None), (0, 37), (0, 100), (0, 130), (1, 150), (1, 200), (1, 259)):
        values, got = v_pages.clone(), None
        sees = torch.zeros(tokens, dtype=torch.bool)
        if request is not None:
            values[int(table[request, at // page]), :, 3, at % page] = poison
            pos = ctx.positions.cpu()
            sees = (ctx.seq_of_token.cpu() == request) & (pos >= at)
            if window is not None:
                sees &= pos - at < window
        got = through(hip, DEVICE, k_pages, values, ctx)
        assert not torch.isfinite(got[sees][:, :, 3]).any(), (request, at)
        got[sees, :, 3] = want[sees, :, 3]
        assert torch.isfinite(got).all(), (request, at)
        assert ((got - want).abs() <= reach).all(), (request, at)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,dim,vdim,rot", [(2, 16, 12, 8), (1, 64, 32, 64), (3, 24, 40, 0), (2, 128, 128, 32), (1, 256, 256, 2)])
def test_retention_kernel_alone(hip, dtype, heads, dim, vdim, rot):
    torch.manual_seed(dim + vdim)
    lengths, eps, base = (70, 9), 1e-6, 1000.0
    m = dict(heads=heads, dim=dim, vdim=vdim, decay=[0.9, 0.99, 1.0][:heads], rot=dict(dims=rot or 2, base=base))
    width = 2 * heads * (dim + vdim)
    rows = [torch.randn(n, width).to(dtype).float() for n in lengths]
    table = None
    if rot:
        freq = torch.tensor([base ** (-2.0 * i / rot) for i in range(rot // 2)], dtype=torch.float32, device=DEVICE)
        table = torch.empty(128, rot // 2, 2, dtype=torch.float32, device=DEVICE)
        hip.rope_table(freq, table)
    state = torch.zeros(3, heads * dim * vdim, dtype=torch.float32, device=DEVICE)
    decay = torch.tensor(m["decay"], dtype=torch.float32, device=DEVICE)
    got = [torch.zeros(n, heads * vdim) for n in lengths]
    for befores, counts in (((0, 0), (33, 2)), ((33, 2), (1, 1)), ((34, 3), (36, 6))):
        ctx = _ctx(befores, counts)
        projected = torch.cat([rows[r][b:b + c] for r, (b, c) in enumerate(zip(befores, counts))]).to(dtype).to(DEVICE)
        out = torch.empty(ctx.num_tokens, heads * vdim, dtype=dtype, device=DEVICE)
        hip.retention(projected, heads, dim, vdim, rot, table, dim ** -0.5, decay, eps, state, ctx, out)
        at = 0
        for r, (b, c) in enumerate(zip(befores, counts)):
            got[r][b:b + c] = out[at:at + c].float().cpu()
            at += c
    assert not state[2].any()
    qk, vs = heads * dim, heads * vdim
    pick = lambda lo, hi: torch.eye(width)[lo:hi]
    w = {"q": pick(0, qk), "k": pick(qk, 2 * qk), "v": pick(2 * qk, 2 * qk + vs), "g": pick(2 * qk + vs, width), "o": torch.eye(vs)}
    for r, n in enumerate(lengths):
        want = plain.retention(rows[r], w, m, eps) if rot else _retention_without_rotation(rows[r], w, m, eps)
        error = (got[r] - want).abs().max() / want.abs().max()
        assert error < (3e-5 if dtype == torch.float32 else 0.03), f"request {r}: {error:.2e}"


def _retention_without_rotation(x, w, m, eps):
    heads, dim, vdim = m["heads"], m["dim"], m["vdim"]
    n = x.shape[0]
    q, k = (x @ w["q"].T).view(n, heads, dim), (x @ w["k"].T).view(n, heads, dim) * dim ** -0.5
    v = (x @ w["v"].T).view(n, heads, vdim)
    S = torch.zeros(heads, dim, vdim)
    out = torch.zeros(n, heads, vdim)
    for t in range(n):
        S = torch.tensor(m["decay"])[:, None, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out[t] = torch.einsum("hdv,hd->hv", S, q[t])
    return plain.unit_rms(out, eps).reshape(n, -1) * plain.silu(x @ w["g"].T)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,blocks,taps", [(80, 5, 4), (64, 1, 1), (300, 3, 2)])
def test_recurrent_unit_kernels_alone(hip, dtype, width, blocks, taps):
    """Convolution without an activation, the gates' block-diagonal product and the scan, three steps of two requests."""
    torch.manual_seed(width)
    lengths = (50, 12)
    bw = width // blocks
    xy = [torch.randn(n, 2 * width).to(dtype).float() for n in lengths]
    conv, conv_b = (torch.randn(width, taps) * 0.5).to(dtype), (torch.randn(width) * 0.1).to(dtype)
    ra, ri = (torch.randn(blocks, bw, bw) * 0.3).to(dtype), (torch.randn(blocks, bw, bw) * 0.3).to(dtype)
    ra_b, ri_b = (torch.randn(blocks, bw) * 0.3).to(dtype), (torch.randn(blocks, bw) * 0.3).to(dtype)
    lam = (-5.0 + 4.0 * torch.rand(width)).to(dtype)
    gate_weight = torch.cat((ra.transpose(1, 2), ri.transpose(1, 2)), dim=2).contiguous().to(DEVICE)
    gate_bias = torch.cat((ra_b, ri_b), dim=1).float().contiguous().to(DEVICE)
    rate = (-8.0 * torch.nn.functional.softplus(lam.float())).to(DEVICE)
    state = torch.zeros(2, width * taps, dtype=torch.float32, device=DEVICE)
    got = [torch.zeros(n, width) for n in lengths]
    for befores, counts in (((0, 0), (20, 2)), ((20, 2), (1, 1)), ((21, 3), (29, 9))):
        ctx = _ctx(befores, counts)
        both = torch.cat([xy[r][b:b + c] for r, (b, c) in enumerate(zip(befores, counts))]).to(dtype).to(DEVICE)
        tokens = both.shape[0]
        u = torch.empty(tokens, width, dtype=dtype, device=DEVICE)
        hip.conv_silu(both, width, conv.to(DEVICE), conv_b.to(DEVICE), state, 1, ctx, u, activation="none")
        gates = torch.empty(tokens, blocks, 2 * bw, dtype=torch.float32, device=DEVICE)
        hip.heads_linear(u.view(tokens, blocks, bw), bw, gate_weight, gates, 2 * bw)
        out = torch.empty(tokens, width, dtype=dtype, device=DEVICE)
        hip.gated_linear_scan(u, gates, gate_bias, rate, both, blocks, state, taps, ctx, out)
        at = 0
        for r, (b, c) in enumerate(zip(befores, counts)):
            got[r][b:b + c] = out[at:at + c].float().cpu()
            at += c
    for r, n in enumerate(lengths):
        x, y = xy[r][:, :width], xy[r][:, width:]
        u = plain.causal_conv(x, conv.float(), conv_b.float())
        S = plain.rglru_scan(u, plain.block_gate(u, ra.float(), ra_b.float()), plain.block_gate(u, ri.float(), ri_b.float()), lam.float())
        want = S * plain.gelu_tanh(y)
        error = (got[r] - want).abs().max() / want.abs().max()
        assert error < (2e-5 if dtype == torch.float32 else 0.04), f"request {r}: {error:.2e}"


@pytest.mark.parametrize("experts,top,ff,shared", [(6, 3, 20, 28), (4, 1, 16, 0), (2, 2, 8, 8), (70, 5, 4, 12), (1, 1, 8, 0),
                                                   (5, 2, 24, 40)])
def test_routing_and_the_experts_activation(hip, experts, top, ff, shared):
    torch.manual_seed(experts)
    tokens = 37
    scored = experts + (1 if shared else 0)
    logits = torch.randn(tokens, scored) * 3
    logits[0, :min(experts, 2)] = 1.25                 # equal logits: the lower index wins
    gates = torch.empty(tokens, scored, device=DEVICE)
    hip.route_chosen(logits.to(DEVICE), gates, experts, top)
    want = torch.zeros(tokens, scored)
    for t in range(tokens):
        order = sorted(range(experts), key=lambda e: (-float(logits[t, e]), e))[:top]
        weights = torch.softmax(logits[t, order], 0)
        want[t, order] = weights
    chosen, weights = plain.route(logits[1:, :experts], torch.eye(experts), torch.zeros(experts), top)      # (rows without equal logits)
    torch.testing.assert_close(torch.zeros(tokens - 1, experts).scatter_(1, chosen, weights), want[1:, :experts])
    if shared:
        want[:, experts] = torch.sigmoid(logits[:, experts])
    torch.testing.assert_close(gates.cpu(), want, rtol=1e-5, atol=1e-6)
    columns = experts * ff + shared
    for dtype in (torch.float32, torch.bfloat16):
        gate_up = torch.randn(tokens, 2 * columns).to(dtype)
        act = torch.empty(tokens, columns, dtype=dtype, device=DEVICE)
        hip.gate_silu_mul(gate_up.to(DEVICE), gates, act, experts, ff)
        g, u = gate_up[:, :columns].float(), gate_up[:, columns:].float()
        weight = torch.cat([want[:, :experts].repeat_interleave(ff, dim=1)] + ([want[:, experts:].expand(-1, shared)] if shared else []), dim=1)
        torch.testing.assert_close(act.float().cpu(), (weight * plain.silu(g) * u).to(dtype).float(), rtol=2e-2 if dtype == torch.bfloat16 else 1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scaled_residual_norm_and_scaled_sum(hip, dtype):
    torch.manual_seed(3)
    for hidden in (96, 100, 4096):
        stream = torch.randn(9, hidden, device=DEVICE)
        delta = torch.randn(9, hidden, device=DEVICE).to(dtype)
        weight = 1 + 0.1 * torch.randn(hidden, device=DEVICE)
        want_stream = stream + 0.7 * delta.float()
        want = plain.rms_norm(want_stream, weight, 1e-6)
        out = torch.empty(9, hidden, dtype=dtype, device=DEVICE)
        hip.norm_add_norm(stream, delta, None, 0.0, weight, 1e-6, out, delta_scale=0.7)
        torch.testing.assert_close(stream, want_stream, rtol=1e-6, atol=1e-6)
        torch.testing.assert_close(out.float(), want.to(dtype).float(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-5, atol=1e-5)
        a, b = torch.randn(9, hidden, device=DEVICE).to(dtype), torch.randn(9, hidden, device=DEVICE).to(dtype)
        total = torch.empty_like(a)
        hip.scaled_sum(a, 0.8, b, 1.1, total)
        torch.testing.assert_close(total.float(), (a.float() * 0.8 + b.float() * 1.1).to(dtype).float(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-6, atol=1e-6)


@pytest.mark.parametrize("heads,kv_heads,maps,dim,vdim", [(16, 4, 1, 128, 128), (4, 4, 1, 32, 256), (3, 1, 2, 64, 64), (20, 1, 1, 256, 32)])
@pytest.mark.parametrize("softcap", [None, 9.0])
@pytest.mark.parametrize("sink", [False, True])
def test_single_tokens_of_short_contexts_beside_a_long_one(hip, heads, kv_heads, maps, dim, vdim, softcap, sink):
    """Where one segment holds all keys, waves have no step of 16 keys, one or several, and take what they have; beside a longer request they
    take four always: the same bits.  One value in a short request is infinite: it reaches its own request alone."""
    torch.manual_seed(dim + heads)
    page, befores = 16, [0, 1, 15, 16, 17, 40, 63, 64, 65, 100, 127, 128, 200, 255, 500]
    need = [before // page + 1 for before in befores]
    table = torch.full((len(befores), max(need)), -1, dtype=torch.int32)
    order = torch.randperm(sum(need)).tolist()
    for r, pages in enumerate(need):
        table[r, :pages] = torch.tensor([order.pop() for _ in range(pages)])
    k_pages = torch.randn(sum(need), kv_heads, page, maps * dim, device=DEVICE).bfloat16()
    v_pages = torch.randn(sum(need), kv_heads, vdim, page, device=DEVICE).bfloat16()
    q = torch.randn(len(befores), heads * maps * dim, device=DEVICE).bfloat16()

    def of(count):
        out = torch.full((count, heads * maps * vdim), float("nan"), dtype=torch.bfloat16, device=DEVICE)
        meta = SimpleNamespace(block_table=table[:count].contiguous().to(DEVICE), rows=None, width=table.shape[1])
        hip.gated_attention(q[:count].contiguous(), k_pages, v_pages, None, 0, _ctx(befores[:count], [1] * count), meta, heads, kv_heads, dim,
                            vdim, dim ** -0.5, softcap, None, None, sink, out, maps=maps)
        return out

    short, beside = of(len(befores) - 1), of(len(befores))
    assert torch.isfinite(beside).all()
    assert torch.equal(short, beside[:-1])
    v_pages[table[6, 2], :, 1, 3] = float("inf")           # position 35 of the request of 64 keys
    poisoned = of(len(befores) - 1)
    assert not torch.isfinite(poisoned[6]).all()
    assert torch.equal(poisoned[:6], short[:6]) and torch.equal(poisoned[7:], short[7:])
    assert torch.equal(poisoned.view(torch.int16), of(len(befores))[:-1].view(torch.int16))
