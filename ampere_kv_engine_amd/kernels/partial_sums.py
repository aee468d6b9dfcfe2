"""Attention that cuts a token's keys over blocks leaves every segment's sums in memory until a second kernel has folded them.  How
a token's keys are cut follows from its position alone (its bits then do not depend on the rest of the step), so what a step of
many long requests leaves would grow with tokens times length: 64 requests of 131,072 tokens with 64 query vectors of 128 make
1.1 GB.  A launch therefore takes only as many of the step's tokens as fit `BYTES`, and the launches of a step use one buffer in
turn.  (64 requests of 32,768 tokens, 64 query and 8 key heads of 128, 277 MB, us a layer: 1,840 in one launch, 1,900 in two,
2,487 in nine of 32 MB - each waits for its last blocks and its fold.  Blocks that take 16 segments each leave a 16th of it
and take 2,173.)"""

from __future__ import annotations

import math

import torch

BYTES = 256 << 20           # of one launch's sums
ARENA_CHUNK = 64 << 20      # what an arena grows by
SEGMENT_KEYS = 256          # `kSegment` of attention_f32.hip, `kSegmentSteps` steps of 16 keys of gated_attention.hip


def at_once(tokens: int, floats_a_token: int) -> int:
    """How many of `tokens` a launch takes (one at least)."""
    return max(1, min(tokens, BYTES // (4 * floats_a_token)))


def room(floats: int) -> int:
    """The floats to ask an arena for.  What fits half of its chunk is asked for as it is; more as a power of two: an arena keeps
    every chunk it has made, so that buffers that grow with the context have to grow by doubling."""
    return floats if 4 * floats <= ARENA_CHUNK // 2 else 1 << (floats - 1).bit_length()


def take(ctx, floats: int, device) -> torch.Tensor:
    """The buffer: from the step's arena, or - a context without one - of its own."""
    arena = getattr(ctx, "arena", None)
    count = room(floats)
    return arena.take((count,), torch.float32) if arena is not None else torch.empty(count, dtype=torch.float32, device=device)


def held_bytes(floats: int) -> int:
    """What an arena holds at most for buffers of up to `floats` (the memory plan's share): a chunk, or all the doublings - and
    what is asked for behind a doubling may need a chunk of its own."""
    if floats == 0:
        return 0
    held, size = ARENA_CHUNK, 4 * room(floats)
    while size > ARENA_CHUNK // 2:
        held += max(size, ARENA_CHUNK) + ARENA_CHUNK
        size //= 2
    return held


def longest_bound(config) -> int:
    """The largest bound on a request's length that a step is launched for (a recorded step's is rounded up)."""
    return config.max_seq_len + config.page_size * config.graph_width_multiple


# ---- single tokens of gated attention ---------------------------------------------------------------------------------
GATED_HEAD_DIMS = (32, 64, 128, 256)      # widths of keys and of values that gated attention's matrix-core kernels are built for


def gated_on_matrix_cores(dim: int, vdim: int, page_size: int) -> bool:
    return dim in GATED_HEAD_DIMS and vdim in GATED_HEAD_DIMS and page_size % 16 == 0


def gated_segments(span: int, window: int | None, chunk: int | None, keep_first: int) -> int:
    """Segments that the keys of a single token touch at most, of `span` keys that it can see: they are counted in steps of 16 keys,
    and where the first key that is seen need not be a step's first, in one step more."""
    aligned = window is None and (chunk is None or chunk % 16 == 0)
    steps = (span + 15) // 16 + (0 if aligned else 1) + (keep_first + 15) // 16
    return (steps * 16 + SEGMENT_KEYS - 1) // SEGMENT_KEYS


def gated_cut(tokens: int, vectors: int, vdim: int, span: int, window: int | None, chunk: int | None,
              keep_first: int) -> tuple[int, int, int]:
    """(segments a token, tokens a launch, floats of the buffer)"""
    segments = gated_segments(span, window, chunk, keep_first)
    if segments <= 1:
        return 1, tokens, 0
    floats = vectors * segments * (vdim + 4)
    tokens = at_once(tokens, floats)
    return segments, tokens, tokens * floats


def gated_bytes(config, vectors: int, dim: int, vdim: int, window: int | None, chunk: int | None, keep_first: int) -> int:
    """What an arena of an engine of this configuration holds at most for single tokens of `vectors` query vectors."""
    if config.dtype != "bfloat16" or not gated_on_matrix_cores(dim, vdim, config.page_size):
        return 0
    span = min(x for x in (chunk, window, longest_bound(config)) if x is not None)
    return held_bytes(gated_cut(config.max_seqs, vectors, vdim, span, window, chunk, keep_first)[2])


# ---- float32 attention (attention_f32.hip) ------------------------------------------------------------------------------
def tile_tokens(share: int) -> int:
    """The fewest tokens after which a tile of 16 (token, head) rows ends where a token's does (`share` query heads a key head)."""
    return 16 // math.gcd(16, share)


def tiles_before(starts, seqs: int, share: int, token: int) -> int:
    """The tiles of the tokens before `token`, request by request (inside a request: a multiple of `tile_tokens`)."""
    return sum((max(0, min(starts[r + 1], token) - starts[r]) * share + 15) // 16 for r in range(seqs))


def launches_of_tiles(starts, seqs: int, share: int, tokens_at_once: int) -> list[tuple[int, int, int, int]]:
    """A step's tokens as launches of about so many: (first token, token end, first tile, tiles).  A launch ends where a request
    does or a tile of its does - after `tile_tokens` at least."""
    whole = tile_tokens(share)
    limit, tokens = max(tokens_at_once, whole), starts[seqs]
    launches, first, tile = [], 0, 0
    request = 0
    while first < tokens:
        end = min(first + limit, tokens)
        while starts[request + 1] <= end and request + 1 < seqs:
            request += 1
        if end < tokens:        # (inside `request`, or where it starts)
            end = starts[request] + (end - starts[request]) // whole * whole
        upto = tiles_before(starts, seqs, share, end)
        launches.append((first, end, tile, upto - tile))
        first, tile = end, upto
    return launches


def f32_segments(longest: int, window: int | None) -> int:
    """Segments that a token's keys touch at most (`akv_attention_f32_segments`, of steps that it cuts)."""
    segments = (longest + SEGMENT_KEYS - 1) // SEGMENT_KEYS
    return min(segments, (window + SEGMENT_KEYS - 2) // SEGMENT_KEYS + 1) if window else segments


def f32_bytes(config, q_heads: int, dim: int, window: int | None) -> int:
    """What an arena of an engine of this configuration holds at most: keys are cut only in steps whose tiles of 16 (token, head)
    rows leave some of 256 units without a block, which is up to 4,096 rows."""
    if config.dtype != "float32":
        return 0
    segments = f32_segments(longest_bound(config), window)
    if segments <= 1:
        return 0
    tokens, floats = min(config.max_batched_tokens, 4096 // q_heads + 1), q_heads * segments * (dim + 4)
    return held_bytes(min(tokens, max(at_once(tokens, floats), 16)) * floats)
