"""The buffer in which matrix states that walk over a step's tokens (delta rule, time mixing, matrix memory) find the tokens'
vectors and leave their outputs: one for all mixers of a kernel set.  Recorded steps keep what it has outgrown, so it grows by
doubling: steps that grow token by token then hold twice the largest at most, where buffers of exactly their size would add up to
many times that.  The counts of floats are upper bounds on what the kernels ask for (`akv_*_workspace`), for the memory plan."""

from __future__ import annotations

LEAST = 1 << 22             # floats
ROWS_BEHIND = 32            # `kRowsBehind` of state_walk.h
CHUNK = 16                  # `kChunk` of delta_rule.hip, whose chunked form takes heads of CHUNK_DIMS
CHUNK_DIMS = (64, 128, 192, 256)


def room(floats: int) -> int:
    """The floats to ask for."""
    return max(LEAST, 1 << max(floats - 1, 0).bit_length())


def held_bytes(floats: int) -> int:
    """What is held at most for steps that need up to `floats`: the buffer and all that it outgrew."""
    return 4 * (2 * room(floats) - LEAST) if floats else 0


def _rows(tokens: int, heads: int, groups: int, dim: int, outputs: int, head_decay: bool) -> int:
    width = 2 * groups * dim + (0 if head_decay else heads * dim) + (3 if head_decay else 2) * heads
    return (tokens + ROWS_BEHIND) * ((width + 3) // 4 * 4 + outputs)


def delta_rule_floats(tokens: int, seqs: int, heads: int, groups: int, dim: int, vdim: int, per_head: bool) -> int:
    """Every token's row, output and chunk: some requests may walk while others go in chunks."""
    chunks = 0
    if dim in CHUNK_DIMS:
        chunks = (tokens // CHUNK + seqs + 1) * heads * (3 * CHUNK * dim + dim + 2 * CHUNK * CHUNK)
    return chunks + _rows(tokens, heads, groups, dim, heads * vdim, per_head)


def time_mixing_floats(tokens: int, heads: int, dim: int) -> int:
    return _rows(tokens, heads, heads, dim, heads * dim, False)


def matrix_memory_floats(tokens: int, heads: int, dim: int, vdim: int) -> int:
    return _rows(tokens, heads, heads, dim, heads * (vdim + 2), True)
