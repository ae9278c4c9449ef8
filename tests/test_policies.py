"""Host-side decisions that need no GPU: how attention keys are cut into splits, and how large a
cache pool is made from leftover device memory."""
import pytest

from kv_cache_optimization_for_llm_amd.engine.engine import EngineError, pool_pages_from_memory
from kv_cache_optimization_for_llm_amd.ops.attention import (choose_decode_ranges, choose_left_ranges, choose_lds_splits, choose_splits,
                                                             use_lds_kernel)

KERNEL_MAX_SPLITS = 256         # what the kernels and their merge take (kva_attention_max_splits)


@pytest.mark.parametrize("nkv", [1, 2, 4, 8])
@pytest.mark.parametrize("items", [1, 2, 3])
@pytest.mark.parametrize("context", [4096, 32768, 65536, 100000, 131072])
def test_key_splits_never_exceed_what_the_kernels_take(nkv, items, context):
    """Few kv heads, one or two decoding requests and a long context ask for many splits; the
    policy must stop at the kernels' limit, and its ranges must still cover every key."""
    for splits, per in (choose_splits(items, nkv, context, KERNEL_MAX_SPLITS),
                        choose_splits(items, nkv, context, KERNEL_MAX_SPLITS, decoding=True),
                        choose_lds_splits(items * nkv, context, KERNEL_MAX_SPLITS),
                        choose_lds_splits(items * nkv, context, KERNEL_MAX_SPLITS, head_dim=128)):
        assert 1 <= splits <= KERNEL_MAX_SPLITS
        if splits > 1:
            assert per % 32 == 0 and splits * per >= context and (splits - 1) * per < context


def test_the_clamp_is_what_bites_for_few_kv_heads():
    # one request on one kv head at 131,072 keys would ask for 1,024 ranges of 128 keys
    assert choose_splits(1, 1, 131072, 4096)[0] == 1024
    assert choose_splits(1, 1, 131072, KERNEL_MAX_SPLITS) == (256, 512)
    assert choose_splits(1, 4, 65536, KERNEL_MAX_SPLITS) == (256, 256)
    assert choose_splits(4096, 8, 2048, KERNEL_MAX_SPLITS) == (1, 0)      # a big prompt fills the GPU by itself
    assert choose_splits(1, 8, 100, KERNEL_MAX_SPLITS) == (1, 0)          # too short to split


@pytest.mark.parametrize("nkv", [1, 2, 5, 8])
@pytest.mark.parametrize("items", [1, 2, 8, 17, 31, 48, 64, 100, 128, 300])
@pytest.mark.parametrize("context", [1, 40, 200, 768, 4096, 8192, 131072])
@pytest.mark.parametrize("head_dim", [64, 128, 256])
def test_key_ranges_of_decoded_tokens_and_the_wavefronts_that_share_them(nkv, items, context, head_dim):
    """Whatever the batch: the ranges cover every key, there are no more of them than the kernels
    take, the wavefronts of a workgroup divide them, and head sizes above 128 get one."""
    splits, per, waves = choose_decode_ranges(items, nkv, context, head_dim, KERNEL_MAX_SPLITS)
    assert 1 <= splits <= KERNEL_MAX_SPLITS and waves in (1, 2, 4) and splits % waves == 0
    if splits > 1:
        # every key in a range, and no workgroup (of `waves` neighbouring ranges) without a key
        assert per % 32 == 0 and splits * per >= context and (splits - waves) * per < context
    if head_dim > 128:
        assert waves == 1


def test_where_decoded_tokens_need_no_merge_launch():
    # 17 to 63 requests of 8 kv heads: four ranges, all in one workgroup
    for items in (17, 24, 32, 48, 63):
        assert choose_decode_ranges(items, 8, 768, 64, KERNEL_MAX_SPLITS) == (4, 192, 4)
    assert choose_decode_ranges(64, 8, 768, 64, KERNEL_MAX_SPLITS) == (1, 0, 1)          # enough wavefronts as they are
    assert choose_decode_ranges(64, 8, 8192, 64, KERNEL_MAX_SPLITS) == (4, 2048, 4)      # but not for long contexts
    for context, want in ((1023, 1), (1024, 4), (4095, 4)):                                # as many as the chip takes at once, long enough
        assert choose_decode_ranges(64, 8, context, 64, KERNEL_MAX_SPLITS)[2] == want
        assert choose_decode_ranges(65, 8, context, 64, KERNEL_MAX_SPLITS) == (1, 0, 1)
    assert choose_decode_ranges(20, 8, 100, 64, KERNEL_MAX_SPLITS) == (2, 64, 2)
    # many ranges share a workgroup only where the merge has much to read
    assert choose_decode_ranges(8, 8, 8192, 64, KERNEL_MAX_SPLITS) == (16, 512, 4)
    assert choose_decode_ranges(8, 8, 768, 64, KERNEL_MAX_SPLITS) == (4, 192, 4)
    # three to fifteen requests above 2,048 keys (from six requests on above 1,024): four ranges to a
    # workgroup, and no more workgroups than compute units
    assert choose_decode_ranges(8, 8, 4096, 64, KERNEL_MAX_SPLITS) == (16, 256, 4)
    assert choose_decode_ranges(3, 8, 8192, 64, KERNEL_MAX_SPLITS) == (40, 224, 4)
    assert choose_decode_ranges(7, 8, 8192, 64, KERNEL_MAX_SPLITS) == (16, 512, 4)          # 224 workgroups, not 280
    assert choose_decode_ranges(12, 8, 2048, 64, KERNEL_MAX_SPLITS) == (8, 256, 4)
    assert choose_decode_ranges(5, 8, 2048, 64, KERNEL_MAX_SPLITS)[2] == 1 and choose_decode_ranges(6, 8, 2048, 64, KERNEL_MAX_SPLITS)[2] == 4
    assert choose_decode_ranges(5, 8, 768, 64, KERNEL_MAX_SPLITS)[2] == 1
    assert choose_decode_ranges(16, 8, 4096, 64, KERNEL_MAX_SPLITS) == (8, 512, 1)
    assert choose_decode_ranges(5, 8, 8192, 128, KERNEL_MAX_SPLITS)[2] == 1                 # head size 128: not measured
    assert choose_decode_ranges(1, 8, 8192, 64, KERNEL_MAX_SPLITS) == (64, 128, 4)
    assert choose_decode_ranges(1, 8, 768, 64, KERNEL_MAX_SPLITS) == (12, 64, 1)
    # short contexts: four ranges from 8 requests of 8 kv heads on
    assert choose_decode_ranges(8, 8, 768, 64, KERNEL_MAX_SPLITS) == (4, 192, 4)
    assert choose_decode_ranges(7, 8, 768, 64, KERNEL_MAX_SPLITS)[2] == 1
    assert choose_decode_ranges(8, 8, 2048, 64, KERNEL_MAX_SPLITS) == (16, 128, 4)
    assert choose_decode_ranges(32, 8, 768, 256, KERNEL_MAX_SPLITS)[2] == 1               # head size 256: one wavefront
    # one request and a long context: twice the ranges the merge kernel is given otherwise, four to a
    # workgroup, so that there is still a workgroup for every compute unit
    assert choose_decode_ranges(1, 8, 32768, 64, KERNEL_MAX_SPLITS) == (128, 256, 4)
    assert choose_decode_ranges(1, 8, 131072, 64, KERNEL_MAX_SPLITS) == (128, 1024, 4)
    assert choose_decode_ranges(1, 1, 65536, 64, KERNEL_MAX_SPLITS) == (256, 256, 1)      # 64 workgroups would be too few
    assert choose_decode_ranges(16, 8, 8192, 64, KERNEL_MAX_SPLITS) == (8, 1024, 1)
    # head size 128: four ranges up to 256 pairs only, and many ranges keep a wavefront each
    assert choose_decode_ranges(32, 8, 768, 128, KERNEL_MAX_SPLITS) == (4, 192, 4)
    assert choose_decode_ranges(33, 8, 768, 128, KERNEL_MAX_SPLITS) == (1, 0, 1)
    assert choose_decode_ranges(47, 8, 2048, 128, KERNEL_MAX_SPLITS) == (1, 0, 1)
    assert choose_decode_ranges(33, 8, 768, 64, KERNEL_MAX_SPLITS) == (4, 192, 4)
    # ... and from 128 pairs on, where head size 64 shares from 64
    assert choose_decode_ranges(8, 8, 768, 64, KERNEL_MAX_SPLITS) == (4, 192, 4)
    assert choose_decode_ranges(12, 8, 768, 128, KERNEL_MAX_SPLITS) == (8, 96, 1)
    assert choose_decode_ranges(16, 8, 768, 128, KERNEL_MAX_SPLITS) == (4, 192, 4)
    assert choose_decode_ranges(48, 8, 768, 128, KERNEL_MAX_SPLITS) == (1, 0, 1)
    assert choose_decode_ranges(64, 8, 8192, 128, KERNEL_MAX_SPLITS) == (1, 0, 1)
    assert choose_decode_ranges(8, 8, 8448, 128, KERNEL_MAX_SPLITS)[2] == 1


def test_which_prompt_rows_go_to_the_workgroup_kernel():
    """Workgroups (128 query rows x kv heads) and mean keys a row decide; head size 128 goes there
    earlier, and with shorter key ranges."""
    # a 2,048-token prompt from position 0 on 8 kv heads, 4 query heads each: 512 workgroups, 1,024 keys a row
    assert not use_lds_kernel(512, 1024.5, 64) and use_lds_kernel(512, 1024.5, 128)
    assert use_lds_kernel(1024, 2048.5, 64) and use_lds_kernel(1024, 2048.5, 96)
    assert use_lds_kernel(768, 10, 64)                       # three workgroups per compute unit: whatever they visit
    assert use_lds_kernel(576, 1152.5, 64) and not use_lds_kernel(576, 500, 64)      # a 2,304-token prompt; many short ones
    # a 256-token portion at position 4,096: 64 workgroups
    assert not use_lds_kernel(64, 4224.5, 64) and use_lds_kernel(64, 4224.5, 128)
    assert not use_lds_kernel(64, 1152.5, 128)               # the same portion at position 1,024
    # head size 128, 24 heads on 8 kv heads: a 2,048-token prompt (384 workgroups) and one of 2,560 (480)
    # stay with the one-wavefront kernel, 3,072 tokens (576) do not; nor does a portion whose rows visit 2,048 keys
    assert not use_lds_kernel(384, 1024.5, 128) and not use_lds_kernel(480, 1280.5, 128)
    assert use_lds_kernel(576, 1536.5, 128) and use_lds_kernel(192, 2560.5, 128)
    assert not use_lds_kernel(8, 8000, 128)                  # a 32-token portion: too few rows to share a key block
    assert choose_lds_splits(64, 4352, KERNEL_MAX_SPLITS, head_dim=128) == (8, 544)
    assert choose_lds_splits(128, 4608, KERNEL_MAX_SPLITS, head_dim=64) == (4, 1152)
    assert choose_lds_splits(512, 2048, KERNEL_MAX_SPLITS, head_dim=128) == (1, 0)


def test_pool_from_leftover_memory():
    GiB = 1 << 30
    # Llama-3.2-1B: 16 layers x 2 x 8 heads x 64 x 16 tokens x 2 bytes = 512 KiB a page
    page_bytes = 16 * 2 * 8 * 64 * 16 * 2
    # config.json says 131,072 positions and the server has 64 seats: every seat at its longest
    # would be 256 GiB; the pool takes what is free instead
    pages = pool_pages_from_memory(200 * GiB, page_bytes, page_size=16, max_seqs=64, max_seq_len=131072,
                                   margin_bytes=2 * GiB, step_bytes=4 * GiB)
    assert pages == (200 - 2 - 4) * GiB // page_bytes
    assert pages * page_bytes <= 194 * GiB < 64 * 131072 // 16 * page_bytes
    # a small model on a big device: never more than every seat at its longest
    assert pool_pages_from_memory(200 * GiB, 4096, page_size=16, max_seqs=8, max_seq_len=100,
                                  margin_bytes=GiB) == 8 * 7
    with pytest.raises(EngineError) as e:
        pool_pages_from_memory(3 * GiB, page_bytes, page_size=16, max_seqs=8, max_seq_len=8192,
                               margin_bytes=2 * GiB, step_bytes=2 * GiB)
    assert "no room for a cache pool" in str(e.value)


def test_row_counts_timed_for_decode_batches_cover_every_batch_above_the_few_rows_kernels():
    """Every batch from 17 seats up to the largest has a timed row count at or above it and at
    most twice its size (the sharing rule of the vendor product's plans)."""
    from kv_cache_optimization_for_llm_amd.ops.gemm_bf16 import decode_tune_rows
    assert decode_tune_rows(1) == [] and decode_tune_rows(16) == []
    assert decode_tune_rows(17) == [17] and decode_tune_rows(32) == [32]
    assert decode_tune_rows(64) == [32, 64] and decode_tune_rows(100) == [32, 64, 100]
    for seats in (17, 40, 64, 200, 384):
        rows = decode_tune_rows(seats)
        for batch in range(17, seats + 1):
            assert any(batch <= r <= 2 * batch for r in rows), (seats, batch)


def test_which_products_of_one_or_two_tokens_take_the_matrix_vector_kernel():
    from kv_cache_optimization_for_llm_amd.ops.gemm_bf16 import use_gemv
    # the four products of a layer and the head at the 1B and 8B sizes: every one the kernel has an instance for
    for n, k in ((3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192), (128256, 2048),
                 (6144, 4096), (4096, 4096), (28672, 4096), (128256, 4096)):
        assert use_gemv(1, n, k) and use_gemv(2, n, k), (n, k)
    assert not use_gemv(1, 4096, 14336)                 # no instance for that K
    assert not use_gemv(3, 2048, 2048)
    # the 3B sizes: all but the down projection, whose rows are long and many
    for n, k in ((5120, 3072), (3072, 3072), (16384, 3072), (128256, 3072)):
        assert use_gemv(1, n, k) and use_gemv(2, n, k), (n, k)
    assert not use_gemv(1, 3072, 8192) and not use_gemv(2, 3072, 8192)
    # long rows cost a second token more than a first one
    assert use_gemv(1, 4096, 5120) and not use_gemv(2, 4096, 5120)
    assert use_gemv(1, 2048, 8192) and use_gemv(2, 2048, 8192)


@pytest.mark.parametrize("context", [512, 513, 600, 768, 769, 1000, 1024, 1500, 2048])
@pytest.mark.parametrize("items", [1, 2])
def test_key_ranges_left_for_an_output_projection_that_adds_them_up(items, context, ):
    ranges, per, waves = choose_left_ranges(items, context, 64, 4)
    assert waves == 4 and ranges % 4 == 0 and 2 <= ranges // 4 <= 4          # what the consumer takes
    assert per % 32 == 0 and per >= 64 and ranges * per >= context           # every key in a range
    assert (ranges - 4) * per < context                                     # no workgroup without a key


def test_where_no_key_ranges_are_left_to_the_output_projection():
    assert choose_left_ranges(3, 768, 64, 4) is None            # the matrix-vector kernel takes two tokens
    assert choose_left_ranges(1, 300, 64, 4) is None            # too short for two workgroups of four ranges
    assert choose_left_ranges(1, 4096, 64, 4) is None           # too long for 16 ranges
    assert choose_left_ranges(1, 768, 128, 4) is None           # measured at head sizes up to 64
    assert choose_left_ranges(1, 768, 64, 1) is None and choose_left_ranges(1, 768, 64, 0) is None
    assert choose_left_ranges(1, 768, 64, 2) == (8, 96, 4)


def test_workgroups_a_pair_at_long_contexts_even_out_the_compute_units():
    """17 to 63 requests on 8 kv heads at 4,096 keys or more: one workgroup of four ranges a pair
    where that fills the compute units' turns well (192, 448 of 256), two or three where it
    leaves most units idle in the last turn (264, 320 of 512)."""
    from kv_cache_optimization_for_llm_amd.ops.attention import _workgroups_a_pair
    assert [_workgroups_a_pair(p, 8192) for p in (136, 160, 176, 192, 264, 320, 384, 448, 504)] == [3, 3, 1, 1, 3, 3, 2, 1, 1]
    assert [_workgroups_a_pair(p, 4096) for p in (136, 192, 264, 320, 384, 448)] == [1, 1, 2, 2, 2, 1]
    assert choose_decode_ranges(33, 8, 8192, 64, KERNEL_MAX_SPLITS) == (12, 704, 4)
    assert choose_decode_ranges(48, 8, 8192, 64, KERNEL_MAX_SPLITS) == (8, 1024, 4)
    assert choose_decode_ranges(56, 8, 8192, 64, KERNEL_MAX_SPLITS) == (4, 2048, 4)
    assert choose_decode_ranges(40, 8, 4096, 64, KERNEL_MAX_SPLITS) == (8, 512, 4)
    assert choose_decode_ranges(40, 8, 2048, 64, KERNEL_MAX_SPLITS) == (4, 512, 4)          # shorter contexts: as before
    assert choose_decode_ranges(40, 8, 131072, 64, KERNEL_MAX_SPLITS) == (12, 10944, 4)


def test_portions_that_share_an_item():
    from kv_cache_optimization_for_llm_amd.ops.attention import MEAN_KEYS_STEPS, choose_portion_waves
    assert [choose_portion_waves(n, n / 2, 64) for n in (64, 256, 512, 1024, 2048, 2560, 3072)] == [1, 2, 2, 2, 2, 2, 1]
    assert [choose_portion_waves(256, mean, 64) for mean in (1152, 8128, 30128)] == [4, 4, 1]
    assert [choose_portion_waves(n, mean, 64) for n, mean in ((1600, 100), (1536, 255), (1024, 2512), (2048, 7024))] == [1, 2, 2, 4]
    assert [choose_portion_waves(n, mean, 128) for n, mean in ((256, 128), (256, 1152), (768, 384), (640, 50), (1024, 512), (512, 7256))] \
        == [2, 4, 2, 1, 1, 1]
    assert choose_portion_waves(512, 256, 160) == 1
    for head_dim in (64, 128):          # nothing but the step below the mean decides: a captured step's shape names it
        for n in range(1, 4000, 61):
            for mean in range(1, 5000, 83):
                step = max([s for s in MEAN_KEYS_STEPS if s <= mean], default=0)
                assert choose_portion_waves(n, mean, head_dim) == choose_portion_waves(n, step, head_dim)


def test_recurrences_go_in_chunks_where_that_is_the_faster_way():
    """One entry from the table's lines on; many prompts at once or a long one among many decoded tokens by what both ways cost."""
    from kv_cache_optimization_for_llm_amd.ops import kernels as K

    def chunks(lengths, heads, dim, vdim, delta, channel=False):
        table = K.DELTA_RULE_CHUNKS_FROM if delta else K.LINEAR_ATTENTION_CHUNKS_FROM
        return K.recurrent_chunks_pay(lengths, K.recurrent_chunks_from(table, dim, vdim, channel), heads, dim, vdim, delta, channel)
    # (us, walk / chunks: 38/59, 75/67; 53/79, 99/87; 33/44, 149/53; 56/57, 85/61)
    for shape, at in (((8, 128, 128, True), 176), ((8, 128, 128, True, True), 224), ((16, 64, 128, False, True), 224), ((16, 128, 128, False), 144)):
        assert chunks([at], *shape) and not chunks([at - 1], *shape)
        assert chunks([at, 1], *shape) and not chunks([at - 1, 1], *shape)
    # (248/308, 123/184, 243/328; 186/144, 717/218; 338/432, 435/502, 404/322, 1,160/590)
    for lengths, shape in (([512] + [1] * 256, (8, 128, 128, True)), ([176] + [1] * 128, (8, 128, 128, True)), ([512] + [1] * 256, (8, 128, 128, True, True)),
                           ([200] * 40, (16, 64, 128, False, True)), ([225] * 40, (8, 128, 128, True, True))):
        assert not chunks(lengths, *shape)
    for lengths, shape in (([512] + [1] * 64, (8, 128, 128, True)), ([2048] + [1] * 64, (8, 128, 128, True)), ([256] * 32, (8, 128, 128, True)),
                           ([200] * 40, (16, 128, 128, False)), ([2048], (32, 128, 128, True))):
        assert chunks(lengths, *shape)
    assert K.recurrent_chunks_from(K.DELTA_RULE_CHUNKS_FROM, 96, 128, False) == 0 == K.recurrent_chunks_from(K.DELTA_RULE_CHUNKS_FROM, 64, 40, True)
    assert not K.recurrent_chunks_pay([], 64, 8, 128, 128, True, False)


def test_a_steps_workspace_is_reserved_and_counts_against_the_graphs_kept(monkeypatch):
    """Keys and values expanded per head go by entries x contexts, not by tokens: the engine's estimate covers every step that
    expands, and a captured step counts as the tokens whose activations take as much."""
    from collections import OrderedDict
    from types import SimpleNamespace

    import torch
    from kv_cache_optimization_for_llm_amd.engine.graphs import PortionGraphs
    from kv_cache_optimization_for_llm_amd.ops import kernels as K
    from kv_cache_optimization_for_llm_amd.ops import latent_attention as lat
    monkeypatch.setattr(K, "latent_prompt_supported", lambda *sizes: True)
    for heads, tokens, positions in ((16, 512, 8192), (16, 8192, 8192), (16, 100, 3000), (128, 2048, 40000), (64, 4096, 700), (16, 63, 8192)):
        limit, seen = lat.expanded_bytes_limit(tokens, positions, heads, 128, 64, 128), 0
        for entries in (1, 2, 3, 7, 20, 64, 128):
            for shortest in (1, 63, 64, 100, 255, 256, 512, tokens // entries):
                for context in (shortest, 256, 300, 1024, 4097, 16 * shortest, positions):
                    if entries * shortest <= tokens and shortest <= context <= positions:
                        seen = max(seen, lat.expanded_bytes(shortest, entries, context, heads, 128, 64, 128, 512, 0, torch.bfloat16))
        assert (seen > 0) == (tokens >= 64) and seen <= limit <= lat.EXPAND_BYTES
    # 64 KB of activations a token; a portion of 512 tokens expands its context of 8,192 positions, 8,320 bytes each: 1,040 tokens more
    model = SimpleNamespace(token_activation_bytes=lambda: 65536, step_workspace_bytes=lambda lens, context:
                            lat.expanded_bytes(min(lens), len(lens), context, 16, 128, 64, 128, 512, 0, torch.bfloat16))
    graphs = PortionGraphs(model, None, "cpu")
    assert isinstance(graphs.slots, OrderedDict)
    for i in range(40):
        kept = graphs.make_room((512,), 8192)
        assert kept == 512 + 1040
        graphs.slots[i] = SimpleNamespace(kept=kept)
        assert sum(s.kept for s in graphs.slots.values()) <= graphs.MAX_KEPT_TOKENS
    assert list(graphs.slots) == list(range(30, 40))
    assert graphs.make_room((512,) + (1,) * 8, 8192) == 520 and len(graphs.slots) == 10        # (decoded tokens beside it: nothing expanded)
    model.step_workspace_bytes = lambda lens, context: 17000 * 65536
    assert graphs.make_room((512,), 8192) is None and len(graphs.slots) == 10


def test_portions_that_do_better_without_sharing_an_item():
    """Measured (us, without / with): short shares, few pairs far behind, pages looked up key by key, windows; and a captured step's
    shape, which names the step below the mean and the tokens of its entries, decides all of it."""
    from kv_cache_optimization_for_llm_amd.ops.attention import MEAN_KEYS_STEPS, choose_portion_waves
    for args in ((256, 32.5, 64, 32.0), (1024, 32.5, 64, 32.0), (800, 50, 80, 50.0), (256, 32.5, 128, 32.0), (40, 1017, 64, 16.5), (64, 4032, 64, 32.0),
                 (80, 1150, 64, 150.0, 16, 1), (192, 2384, 64, 383.0, 16, 1), (1536, 20768, 64, 768.0), (128, 4064, 64, 64.0, 32), (304, 8150, 64, 150.0, 8),
                 (512, 3050, 128, 50.0, 16, 1), (512, 2500, 128, 500.0, 16, 1), (40, 1017, 128, 16.5), (2048, 1024, 64, 1024.0, 16, 4, 128)):
        assert choose_portion_waves(*args) == 1, args
    for args, waves in (((512, 256.5, 64, 256.0), 2), ((256, 128.5, 64, 128.0), 2), ((256, 1152, 64, 128.0), 4), ((200, 2100, 64, 100.0), 4), ((512, 2256, 128, 256.0), 2),
                        ((128, 64.5, 64, 64.0), 2), ((1536, 20768, 64, 768.0, 8), 4), ((64, 2032, 64, 32.0, 16, 4, 256), 2), ((64, 300, 64, 32.0, 16, 4, 256), 1),
                        ((128, 1064, 128, 64.0, 16, 4, 1024), 4)):
        assert choose_portion_waves(*args) == waves, args
    for n in range(1, 3000, 131):
        for mean in (20, 127, 129, 300, 511, 513, 900, 1500, 3000, 7000, 30000):
            step = max([s for s in MEAN_KEYS_STEPS if s <= mean], default=0)
            for rest in ((64, 30.0), (64, 50.0, 8), (128, 100.0, 16, 1), (64, 20.0, 16, 4, 256), (64, 400.0, 16, 2, 128), (128, 100.0, 32, 4, 700)):
                assert choose_portion_waves(n, mean, *rest) == choose_portion_waves(n, step, *rest)


def test_captured_shapes_are_told_apart_by_what_is_decided():
    """Steps of the same entries whose attention is decided alike share a shape, whatever their mean number of keys; those decided
    otherwise do not.  The head layouts come from the first eager step, which is noted under the shape its next step asks for."""
    from types import SimpleNamespace

    import numpy as np
    from kv_cache_optimization_for_llm_amd.engine.graphs import PortionGraphs
    from kv_cache_optimization_for_llm_amd.ops.attention import portion_choice
    for heads, dim in ((32, 64), (32, 128), (24, 128)):
        graphs = PortionGraphs(None, None, "cpu")
        lens, rows = (512,) + (1,) * 8, tuple(range(511, 520))

        def key(start):
            return graphs.shape_key(lens, [start] + [8000] * 8, rows)
        batch = SimpleNamespace(attention_plans={(heads, 8, dim, 16, 0, 0): [], (heads, 8, dim, 16, 12, 0): [], (heads, 8, dim, 16, 0, 256): []},
                                h_entry_start_pos=np.asarray([1536] + [8000] * 8, dtype=np.int32), _items={})
        graphs.note(key(1536), batch)
        assert list(graphs.seen) == [key(1536)] and graphs.times[key(1536)] == 1
        assert len(graphs.layouts) == 2
        keys, choices = {}, set()
        for start in range(0, 7680, 128):
            decided = tuple(portion_choice(lens, start + 256.5, heads // 8, 8, dim, 16, visible) for visible in (0, 256))
            assert keys.setdefault(key(start), decided) == decided
            choices.add(decided)
        assert len(keys) == len(choices) <= 3
    assert PortionGraphs(None, None, "cpu").shape_key([5000], [0], [4999]) is None


def test_experts_products_take_256_outputs_a_workgroup_where_128_would_not_fit_the_chip_at_once():
    """By the groups that are in use, measured (us, 128 / 256 outputs), not by those the list has room for."""
    from kv_cache_optimization_for_llm_amd.ops.kernels import moe_tiles, moe_wide
    for slots, experts, outputs, wide in ((8192, 4, 1024, False), (8192, 4, 2048, True),                    # 56/75, 53/43
                                          (3356, 16, 1536, False), (6400, 16, 1536, True), (12800, 16, 768, True),      # 44/59, 82/71, 84/73
                                          (7680, 32, 1024, True), (5120, 32, 1024, False), (10240, 64, 512, False),     # 82/73, 48/61, 48/61
                                          (15360, 64, 512, True), (20480, 128, 512, True), (10240, 64, 768, True)):     # 80/73, 120/100, 86/75
        assert moe_wide(outputs, moe_tiles(slots, experts, 8), 8, experts) == wide, (slots, experts, outputs)
    assert not moe_wide(4096, moe_tiles(20000, 16, 4), 4, 16)


def test_the_experts_first_product_goes_to_tiles_where_they_are_faster():
    """By sizes and activation, measured (us, groups of 8 or 4 tiles / blocks of as many rows as an expert has)."""
    from kv_cache_optimization_for_llm_amd.ops.kernels import moe_tiles_plan
    for slots, experts, top, n, k, act, gated, tiles in (
            (8192, 16, 4, 1536, 2048, "silu", True, True),          # 64.7/62.3
            (8192, 16, 4, 1024, 2048, "gelu", False, True),         # 68.5/49.6
            (2048, 4, 4, 1024, 2048, "gelu", False, True),          # 24.8/18.9
            (8192, 4, 4, 1024, 2048, "gelu", False, False),         # 43.4/44.6
            (8192, 4, 4, 1024, 2048, "gelu_tanh", False, False),    # 43.1/48.5
            (8192, 16, 4, 1024, 2048, "gelu_tanh", False, True),    # 67.7/48.9
            (4812, 32, 4, 1024, 1024, "gelu", False, False),        # 27.3/33.3
            (4767, 8, 1, 2816, 2048, "gelu", True, False),          # 71/107
            (17436, 32, 4, 768, 1536, "gelu_tanh", False, False),   # 66/98
            (12000, 4, 4, 2048, 1024, "gelu", False, False),        # 74/89
            (24000, 4, 4, 1024, 2048, "gelu", False, False),        # 103/127
            (16384, 4, 4, 1536, 2048, "silu", True, False)):        # 98/104
        assert (moe_tiles_plan(slots, experts, top, n, k, False, act, gated) >= 0) == tiles, (slots, experts, n, k, act)


def test_rotated_tokens_share_a_workgroup_where_that_is_faster():
    """By tokens and the elements of V of one, measured (us, a workgroup a token / sixteen tokens a workgroup)."""
    from kv_cache_optimization_for_llm_amd.ops.kernels import rope_tokens_wide
    for tokens, heads, dim, cached, wide in (
            (65, 8, 64, True, False),           # 3.5/4.9; decoded tokens 3.4/5.4
            (256, 8, 64, True, False),          # 4.0/4.4; decoded 4.3/6.0
            (512, 2, 64, True, False),          # decoded 4.2/5.4
            (256, 8, 128, True, False),         # decoded 5.6/7.0
            (512, 16, 64, True, True),          # 6.5/4.9
            (1024, 8, 64, True, True),          # 6.9/5.7
            (2048, 1, 128, True, True),         # 6.3/5.0
            (2048, 8, 32, True, True),          # 7.9/5.8
            (2048, 8, 64, False, False),        # no cache: 4.8/5.2
            (64, 64, 256, True, False)):
        assert rope_tokens_wide(tokens, heads, dim, cached) == wide, (tokens, heads, dim, cached)


def test_the_choice_of_experts_is_made_inside_the_first_product_where_workgroups_and_tokens_are_few():
    """By workgroups of the launch and tokens, measured (us, in a launch of its own / inside)."""
    from kv_cache_optimization_for_llm_amd.ops.kernels import moe_choice_inside
    for workgroups, tokens, inside in ((384, 1, True), (384, 8, True), (384, 16, False),            # 18.5/15.7, 20.3/19.1, 22.6/24.0
                                       (480, 8, True), (480, 16, False), (768, 1, False),           # 22.3/21.7, 25.0/26.8, 41.0/42.2
                                       (1536, 1, False), (1536, 16, False), (256, 8, True), (256, 16, False)):   # 41.2/47.8, 46.5/64.8, 15.6/14.5, 16.4/17.0
        assert moe_choice_inside(workgroups, tokens) == inside, (workgroups, tokens)


def test_products_timed_at_start_up_run_the_way_that_was_faster(monkeypatch):
    """Whole or in two, both timed; rows that were not timed go by the nearest above, up to twice as many; others by the rule."""
    import torch
    from kv_cache_optimization_for_llm_amd.ops import gemm_bf16 as G
    calls, us = [], {}
    monkeypatch.setattr(G, "_TIMED_CUTS", {})
    monkeypatch.setattr(G.K, "gemm_vendor_tune", lambda rows, ws, dtype, columns_of=0: calls.append((rows, ws[0].shape[0], columns_of)) or us[ws[0].shape[0]])
    ws, dev = [torch.empty((8208, 64), dtype=torch.bfloat16)] * 2, torch.device("cpu")
    # the rest begins a turn of the compute units, or does not, or is too much for the small product
    assert [G.vendor_cut(m, n) for m, n in ((2048, 8208), (1793, 8208), (1792, 8208), (2049, 8208), (4096, 4128), (2048, 4128), (4096, 4129), (2048, 8192))] \
        == [8192, 8192, 0, 0, 4096, 0, 0, 0]
    assert G.chosen_cut(2048, 8208, 64, dev) == 8192
    us.update({8208: (84.0, 50.0, 9), 8192: (56.0, 48.0, 8), 16: (8.0, 6.0, 7)})
    assert G.tune_linear(2048, ws) == (64.0, 50.0, 24) and calls == [(2048, 8208, 0), (2048, 8192, 8208), (2048, 16, 8208)]
    assert [G.chosen_cut(m, 8208, 64, dev) for m in (4096, 2048, 1793, 1792)] == [8192, 0, 0, 0]
    assert G.chosen_cut(2048, 8208, 32, dev) == G.chosen_cut(2048, 8208, 64, dev, torch.float32) == 8192
    us[8208] = (84.0, 60.0, 9)
    assert G.tune_linear(1900, ws) == (64.0, 54.0, 24) and G.chosen_cut(1800, 8208, 64, dev) == 8192 and G.chosen_cut(1901, 8208, 64, dev) == 0
    us[16] = (-1.0, -1.0, 0)                # the library has nothing for the rest: one product
    assert G.tune_linear(4096, ws) == (84.0, 60.0, 17) and G.chosen_cut(4096, 8208, 64, dev) == 0
    calls.clear()
    us[8192 + 64] = (5.0, 4.0, 3)
    assert G.tune_linear(2048, [torch.empty((8192 + 64, 64))]) == (5.0, 4.0, 3) and calls == [(2048, 8256, 0)]


class _Operand:
    """As much of a tensor on the GPU as the choice of a product looks at."""
    is_cuda, device = True, "cuda:0"

    def __init__(self, *shape):
        import torch
        self.shape, self.dtype = shape, torch.bfloat16

    def is_contiguous(self):
        return True

    def data_ptr(self):
        return 0

    def stride(self, _):
        return 1

    def __getitem__(self, _):
        return self


def test_the_librarys_algorithms_are_timed_where_the_library_takes_rows(monkeypatch):
    """What linear_bf16 hands to the library at a row count, or at one that what was timed there serves (down to half of it), is timed; and
    nothing else is."""
    from types import SimpleNamespace
    from kv_cache_optimization_for_llm_amd.models.builder import Model
    from kv_cache_optimization_for_llm_amd.ops import gemm_bf16 as G
    taken, timed = [], []
    monkeypatch.setattr(G, "_TIMED_CUTS", {})
    monkeypatch.setattr(G.K, "gemm_tiles_takes", lambda x, w: True)
    for kernel in ("gemm_tiles", "gemm_skinny", "gemv", "gemm_vendor"):
        monkeypatch.setattr(G.K, kernel, lambda *a, _k=kernel, **kw: taken.append(_k) or True)
    monkeypatch.setattr(G, "tune_linear", lambda rows, ws: timed.append(rows) or (1.0, 1.0, 1))

    def takes(m, n, k):
        taken.clear()
        G.linear_bf16(_Operand(m, k), _Operand(n, k), _Operand(m, n), SimpleNamespace(halves=1))
        return set(taken)

    # outputs a little past whole columns, which the library takes in two; others that it takes whole at some of the rows; none
    for n, k, asked in ((8208, 2048, (2048, 1024)), (16400, 2048, (2048,)), (4112, 2048, (4096,)), (6144, 4096, (256, 128, 80)), (3072, 8192, (512,)),
                        (2048, 2048, (64, 512, 2048)), (2048, 8192, (100, 1203)), (40000, 2048, (96,))):
        for rows in asked:
            library = any("gemm_vendor" in takes(m, n, k) for m in range((rows + 1) // 2, rows + 1))
            timed.clear()
            lin = SimpleNamespace(weight=_Operand(n, k), tiled=SimpleNamespace(halves=1), out_features=n, in_features=k, halves=1)
            Model.tune_products(SimpleNamespace(linears=lambda: [lin]), [rows])
            assert timed == ([rows] if library else []), (rows, n, k)
    assert takes(2048, 8208, 2048) == {"gemm_vendor"} and takes(256, 6144, 4096) == {"gemm_tiles"} and takes(200, 6144, 4096) == {"gemm_vendor"}
    # a joined [gate; up] matrix: by the plan of the product with its activation
    for rows in (96, 300, 8190):
        timed.clear()
        lin = SimpleNamespace(weight=_Operand(28672, 4096), tiled=SimpleNamespace(halves=2), out_features=28672, in_features=4096, halves=2)
        Model.tune_products(SimpleNamespace(linears=lambda: [lin]), [rows])
        assert timed == ([rows] if any(G.K.gemm_tiles_plan(m, 28672, 4096, G.K.TILES_GATED) < 0 for m in range(max(65, (rows + 1) // 2), rows + 1)) else [])
