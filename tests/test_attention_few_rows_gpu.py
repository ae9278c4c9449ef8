"""Plain attention of few rows, four wavefronts a token and head: the bits of the kernel with one."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

# at the edges of blocks of 64 keys and of rounds of four, short ones among them (whose block the others' wavefronts pass by)
POSITIONS = [0, 31, 32, 63, 64, 127, 128, 191, 255, 256, 319, 600]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nq, nkv, d, dv", [(8, 2, 64, 64), (3, 3, 128, 128), (4, 1, 64, 100), (2, 1, 128, 24)])
@pytest.mark.parametrize("mask", [{}, dict(window=65), dict(window=70, keep_first=3), dict(window=130, keep_first=70), dict(chunk=96)])
@pytest.mark.parametrize("sink", [False, True])
def test_four_wavefronts_have_the_bits_of_one(dtype, nq, nkv, d, dv, mask, sink, gpu):
    g = torch.Generator(device=gpu).manual_seed(2)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu).to(dtype)
    T, page, blocks = len(POSITIONS), 16, 40
    # what lies behind a token is no number; pages without a key that is seen are not in the table, as the cache leaves them (and what
    # such an entry would lead to is a page in front of the others)
    kc = torch.full((1 + T * blocks, nkv, page, d), float("nan"), dtype=dtype, device=gpu)
    vc = torch.full((1 + T * blocks, nkv, dv, page), float("nan"), dtype=dtype, device=gpu)[1:]
    table = torch.randperm(T * blocks, generator=torch.Generator().manual_seed(1)).to(torch.int32).view(T, blocks).to(gpu)
    for t, pos in enumerate(POSITIONS):
        at = torch.arange(pos + 1, device=gpu)
        kc[1 + table[t].long()[at // page], :, at % page] = rnd(pos + 1, nkv, d)
        vc[table[t].long()[at // page], :, :, at % page] = rnd(pos + 1, nkv, dv)
        lo = pos - pos % mask["chunk"] if "chunk" in mask else max(0, pos - mask.get("window", pos + 1) + 1)
        seen = (at >= lo) | (at < mask.get("keep_first", 0))
        unseen = torch.ones(blocks, dtype=torch.bool, device=gpu)
        unseen[at[seen] // page] = False
        table[t, unseen] = -1
    kc = K.keys_to_pages(kc)[1:]
    q, sinks = rnd(T, nq * d) * 2, torch.randn(nq, generator=g, device=gpu) if sink else None
    seat, pos = torch.arange(T, dtype=torch.int32, device=gpu), torch.tensor(POSITIONS, dtype=torch.int32, device=gpu)

    def run(longest):
        out = torch.full((T, nq * dv), 7.0, dtype=dtype, device=gpu)
        return K.attention_rowwise(q, nq * d, out, kc, vc, table, seat, pos, nq, nkv, d, d ** -0.5, sinks=sinks, value_dim=dv, longest=longest, **mask)
    one, four = run(64), run(601)            # (one block of keys at most: a wavefront; it decides nothing else)
    assert one.isfinite().all() and torch.equal(one, four)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nq, nkv, d, dv", [(8, 2, 64, 64), (8, 2, 128, 100), (6, 2, 64, 128), (2, 1, 128, 24), (4, 4, 64, 64)])
@pytest.mark.parametrize("mask", [{}, dict(window=70, keep_first=3)])
@pytest.mark.parametrize("page", [16, 6])            # (6: keys one by one, a wavefront a head or several)
def test_many_rows_have_the_bits_of_few(dtype, nq, nkv, d, dv, mask, page, gpu):
    """Four, three, two and one query heads a wavefront, as a prompt's tokens take them, against the same tokens alone."""
    g = torch.Generator(device=gpu).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu).to(dtype)
    T, blocks, times = len(POSITIONS), 601 // page + 1, 12288 // nq // len(POSITIONS) + 1
    kc, vc = K.keys_to_pages(rnd(blocks, nkv, page, d)), rnd(blocks, nkv, dv, page)
    table = torch.randperm(blocks, generator=torch.Generator().manual_seed(1)).to(torch.int32).view(1, blocks).to(gpu)
    q, sinks = rnd(T, nq * d) * 2, torch.randn(nq, generator=g, device=gpu)
    pos = torch.tensor(POSITIONS, dtype=torch.int32, device=gpu)

    def run(n):
        out = torch.full((n * T, nq * dv), 7.0, dtype=dtype, device=gpu)
        return K.attention_rowwise(q.repeat(n, 1), nq * d, out, kc, vc, table, torch.zeros(n * T, dtype=torch.int32, device=gpu), pos.repeat(n), nq, nkv,
                                   d, d ** -0.5, sinks=sinks, value_dim=dv, **mask)
    few, many = run(1), run(times)
    assert few.isfinite().all() and torch.equal(few.repeat(times, 1), many)
