"""Plain attention of few rows: which entries of the block table its wavefronts look up (on the CPU; the kernel's own rule).

A window's pages go back to the pool once no later token sees a key of theirs, and their entries name no page.  A key that is read
and not used leaves the result as it is, so only the entries can show that none of those is looked up."""
import numpy as np
import pytest

from kv_cache_optimization_for_llm_amd.cache.manager import CacheManager
from kv_cache_optimization_for_llm_amd.ops.library import hip_lib
from kv_cache_optimization_for_llm_amd.parts.base import attention_cache_spec


def reads(pos, block, window=0, keep_first=0, chunk=0):
    keys, values = np.empty(64, dtype=np.int32), np.empty(64, dtype=np.int32)
    assert hip_lib().kva_attention_few_reads(pos, window, keep_first, chunk, block, keys.ctypes.data, values.ctypes.data) == 0
    return keys, values


def sees(pos, window=0, keep_first=0, chunk=0):
    """Whether a token at ``pos`` sees key 0 .. pos."""
    key = np.arange(pos + 1)
    if chunk:
        return key // chunk == pos // chunk
    return (pos - key < window) | (key < keep_first) if window else key >= 0


@pytest.mark.parametrize("page", [4, 16, 32, 64])
@pytest.mark.parametrize("mask", [{}, dict(window=65), dict(window=100), dict(window=70, keep_first=3), dict(window=130, keep_first=70), dict(chunk=96)])
def test_every_page_looked_up_holds_a_key_that_is_seen(page, mask):
    for pos in range(0, 420):
        seen = sees(pos, **mask)
        pages = set((np.nonzero(seen)[0] // page).tolist())
        for block in range(pos // 64 + 3):
            inside = np.arange(64 * block, min(64 * block + 64, pos + 1))
            keys, values = reads(pos, block, **mask)
            if not inside.size or not seen[inside].any():
                assert (keys == -1).all() and (values == -1).all()
                continue
            assert set((keys // page).tolist()) <= pages and set((values // page).tolist()) <= pages, (pos, block)
            assert (keys[inside - 64 * block] == inside)[seen[inside]].all()         # a key that is seen is read itself
            assert (values[inside - 64 * block] == inside)[seen[inside]].all()


@pytest.mark.parametrize("keep_first", [0, 5, 70])
def test_no_entry_that_the_cache_has_given_back(keep_first):
    """A request decoded past several windows: at every step, by the table as the cache leaves it."""
    window, page = 100, 16
    cache = CacheManager([(attention_cache_spec(1, 64, kind="window", window=window, keep_first=keep_first), [0])], {}, page_size=page, num_pages=64,
                         max_seqs=1, max_seq_len=640)
    seat, given_back = cache.admit("a"), 0
    for pos in range(520):
        assert cache.grow(seat, pos + 1)
        row = cache.groups[0].table_host[seat]
        given_back += int((row[:pos // page] < 0).any())
        for block in range(pos // 64 + 1):
            keys, values = reads(pos, block, window, keep_first)
            if keys[0] >= 0:
                assert (row[keys // page] >= 0).all() and (row[values // page] >= 0).all(), (pos, block)
        cache.commit(seat, pos + 1)
    assert given_back > 300
