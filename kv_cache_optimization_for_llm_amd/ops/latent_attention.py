"""Kernel choice for attention over low-rank entries and for the per-head products around it."""
from __future__ import annotations

import torch

from . import kernels as K


def heads_product(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor, gates=None, rotate=None) -> torch.Tensor:
    """``out[t, h] = w[h] @ x[t, h]`` for ``w`` ``[heads, N, K]``; ``x`` and ``out`` may be views into
    wider buffers.  ``gates`` ``[T, heads]``: head h of row t times ``sigmoid(gates[t, h])``;
    gates ``[T, heads, N]``: every element times its own.  ``rotate``: rows rotated in the same launch
    (``kernels.heads_matmul``)."""
    return K.heads_matmul(x, w, out, gates, rotate)


# Workgroups (of four wavefronts) a launch should have before keys stop being cut into ranges: one a compute
# unit; two where two fit one (small ranks).
_TARGET_WORKGROUPS = 256
_SMALL_RANK = 128
_MIN_KEYS_PER_RANGE = 128       # a block of 32 keys for each wavefront of an item of few rows
FEW_ROWS, MANY_ROWS = 16, 64    # rows of a work item of the two kernels


def mfma_supported(rank: int, key_dim: int, page_size: int = 16) -> bool:
    """Whether the matrix-core kernels have an instance for these sizes."""
    return K.latent_attention_mfma_supported(rank, key_dim, page_size)


def choose_ranges(items: int, max_context: int, visible: int = 0, workgroups: int = _TARGET_WORKGROUPS) -> tuple:
    """(ranges, keys per range) for ``items`` work items over at most ``max_context`` keys: ranges
    of at least 128 keys until the launch has ``workgroups`` workgroups.  ``visible``
    > 0: a row sees at most so many keys (a window and the kept first positions), wherever they
    lie: the ranges are sized as if the context were that long, and most of them stay empty."""
    want = max(1, workgroups // max(1, items))
    span = min(max_context, visible) if visible > 0 else max_context
    ranges = max(1, min(want, span // _MIN_KEYS_PER_RANGE))
    if ranges == 1:
        return 1, 0
    per = (-(-span // ranges) + 31) // 32 * 32
    return -(-max_context // per), per


# Steps whose entries all have so many tokens, and contexts of at most so many times as many, expand keys and values
# (ops.kernels.latent_prompt) while the expanded contexts stay below so many bytes.  Whole steps of 8 layers (16 heads of
# 128 + 64 / 128, rank 512), over the cached rows -> expanded, ms: one prompt of 64 / 128 / 256 / 2,048 tokens 1.36 / 1.61 /
# 1.67 / 4.77 -> 1.30 / 1.51 / 1.51 / 3.44; four of 128 / 256 behind 1,024: 2.41 / 3.16 -> 1.98 / 2.57; 128 / 192 / 256
# behind 2,048: 1.87 / 2.36 / 2.21 -> 1.95 / 2.21 / 1.95; 256 behind 6,000: 2.82 -> 2.86; 512 behind 7,000: 4.17 -> 3.26.
# Error of the logits against 64 bits: 0.0084 / 0.0082 and 0.0085 / 0.0081 (eight prompts of 512 / one of 2,048).
EXPAND_FROM = 64
EXPAND_CONTEXTS = 16
EXPAND_BYTES = 512 << 20


def expanded_bytes(shortest: int, entries: int, max_context: int, heads: int, dim: int, rot: int, vdim: int, rank: int, window: int,
                   dtype) -> int:
    """Bytes of expanded keys and values over which a step's prompt portions attend; 0: they attend over the cached rows.  A
    captured step knows its contexts to the power of two above them (at least 256): every step goes by that, so that it
    asks for the same work items with and without."""
    context = 1 << max(8, (max_context - 1).bit_length())
    size = entries * context * (heads * (dim + vdim) + rot) * 2
    return size if (dtype == torch.bfloat16 and window <= 0 and heads <= 1024 and shortest >= EXPAND_FROM
                    and context <= EXPAND_CONTEXTS * shortest and size <= EXPAND_BYTES
                    and K.latent_prompt_supported(dim, rot, vdim, rank)) else 0


def expanded_bytes_limit(tokens: int, positions: int, heads: int, dim: int, rot: int, vdim: int) -> int:
    """The most any step of up to ``tokens`` tokens and contexts of up to ``positions`` expands."""
    if tokens < EXPAND_FROM:
        return 0
    rows = min(EXPAND_CONTEXTS * tokens, (tokens // EXPAND_FROM) << max(8, (positions - 1).bit_length()))
    return min(EXPAND_BYTES, rows * (heads * (dim + vdim) + rot) * 2)


def expands(batch, heads: int, dim: int, rot: int, vdim: int, rank: int, window: int, dtype) -> bool:
    """Whether a step's prompt portions attend over expanded keys and values."""
    return expanded_bytes(batch.min_q_len, batch.num_entries, batch.max_context, heads, dim, rot, vdim, rank, window, dtype) > 0


def latent_attention(q_lat: torch.Tensor, out: torch.Tensor, kv, batch, scale: float, window: int = 0,
                     keep_first: int = 0, sinks=None) -> torch.Tensor:
    """Causal attention of the step's tokens over the rows of ``kv.arrays["latent"]``
    (``[pages, page_size, key_dim]``): ``q_lat`` ``[T, heads, key_dim]``, ``out`` ``[T, heads, rank]``."""
    if window <= 0:
        keep_first = 0
    cache = kv.arrays["latent"]
    if q_lat.dtype == torch.bfloat16 and mfma_supported(out.shape[2], q_lat.shape[2], cache.shape[1]):
        # entries of at most 16 rows (decoded tokens) and longer ones (prompt portions) have a kernel each
        heads = q_lat.shape[1]
        if batch.max_q_len * heads <= FEW_ROWS:
            launches = [(*batch.attention_items(heads, 1, "all")[:2], FEW_ROWS)]
        elif batch.min_q_len * heads > FEW_ROWS:
            launches = [(*batch.attention_items(heads, MANY_ROWS // 16, "all")[:2], MANY_ROWS)]
        else:
            launches = [(*batch.attention_items(heads, MANY_ROWS // 16, "long")[:2], MANY_ROWS),
                        (*batch.attention_items(heads, 1, "short")[:2], FEW_ROWS)]
        ranges, per = choose_ranges(sum(l[0].shape[0] for l in launches), batch.max_context,
                                    window + keep_first if window > 0 else 0,
                                    _TARGET_WORKGROUPS * (2 if out.shape[2] <= _SMALL_RANK else 1))
        (item_entry, item_row0, rows), *more = launches
        return K.latent_attention_mfma(q_lat, out, cache, kv.block_table, item_entry, item_row0,
                                       batch.entry_seat, batch.entry_q_start, batch.entry_start_pos, scale, window,
                                       keep_first, sinks, ranges, per, rows, more)
    return K.latent_attention_rowwise(q_lat, out, kv.arrays["latent"], kv.block_table, batch.tok_seat,
                                      batch.positions, scale, window, keep_first, sinks)
