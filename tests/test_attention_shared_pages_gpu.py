"""The workgroup kernel of prompt portions where its list of pages ends: it holds 512 blocks of 32 keys (16,384 keys) at a time."""
import math

import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

# (first position, tokens): up to one key short of a list, exactly one, one and a key, over two of them, nearly none
ENTRIES = [(16384 - 40, 39), (16384 - 7, 7), (16384 - 20, 21), (33000, 9), (0, 5)]


@pytest.mark.parametrize("nq, nkv, d", [(4, 2, 32), (8, 2, 64), (3, 1, 96), (8, 1, 128)])
@pytest.mark.parametrize("window, pair, per", [(0, False, 0), (0, True, 0), (16500, False, 0), (90, True, 0), (0, False, 16416), (0, True, 3008)])
def test_contexts_longer_than_the_pages_a_workgroup_holds(nq, nkv, d, window, pair, per, gpu):
    g = torch.Generator(device=gpu).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=gpu).to(torch.bfloat16)
    page, group, scale = 16, nq // nkv, 1.0 / math.sqrt(d)
    blocks = [(s + n + page - 1) // page for s, n in ENTRIES]
    total = sum(blocks) + 3
    # what no entry has written holds NaN and infinities
    kc = torch.full((total, nkv, page, d), float("nan"), dtype=torch.bfloat16, device=gpu)
    vc = torch.full((total, nkv, d, page), float("inf"), dtype=torch.bfloat16, device=gpu)
    vc[:, :, ::2] = float("nan")
    perm = torch.randperm(total, generator=torch.Generator().manual_seed(4))
    table = torch.zeros((len(ENTRIES), max(blocks) + 1), dtype=torch.int32)
    rows, wants, bounds, queries, used, q0 = [], [], [], [], 0, 0
    for e, ((start, n), nb) in enumerate(zip(ENTRIES, blocks)):
        ctx, own = start + n, perm[used:used + nb]
        used += nb
        table[e, :nb] = own.to(torch.int32)
        k, v = rnd(ctx, nkv, d), rnd(ctx, nkv, d)
        pg, at = own.to(gpu)[torch.arange(ctx, device=gpu) // page], torch.arange(ctx, device=gpu) % page
        kc[pg, :, at] = k
        vc[pg, :, :, at] = v
        q = rnd(n, nq, d) * 3                       # sharp: some keys of every row matter
        queries.append(q)
        pos = torch.arange(start, ctx, device=gpu)[:, None]
        key = torch.arange(ctx, device=gpu)[None]
        seen = (key <= pos) & ((key > pos - window) if window else True)
        kk, vv = (x.float().repeat_interleave(group, 1).transpose(0, 1).contiguous() for x in (k, v))
        s = torch.matmul(q.float().transpose(0, 1).contiguous(), kk.transpose(1, 2).contiguous()).double() * scale
        p = torch.softmax(s.masked_fill(~seen, float("-inf")), dim=-1)
        wants.append(torch.matmul(p, vv.double()).transpose(0, 1).reshape(n, nq * d))
        bounds.append(torch.matmul(p, vv.double().abs()).transpose(0, 1).reshape(n, nq * d))
        rows += [(q0, n, start, e, r0, 0, 0, 0) for r0 in range(0, n * group, 128)]
        q0 += n
    rows.sort(key=lambda m: -m[2])
    meta = torch.tensor(rows, dtype=torch.int32, device=gpu)
    qkv = torch.cat(queries).reshape(q0, nq * d)
    out = torch.full((q0, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    splits = -(-max(s + n for s, n in ENTRIES) // per) if per else 1          # (ranges of more than a list, or many; some are empty)
    K.attention_lds(qkv, nq * d, out, K.keys_to_pages(kc.cpu()).to(gpu), vc, table.to(gpu), meta, nq, nkv, d, scale, window, pair,
                    splits, per)
    # a probability, the denominator and the result are each rounded to 8 bits once (half a unit: 2**-9); the scores in fp32 add
    # d * 2**-24 of their terms' size, under 2**-13 of a probability here
    err = (out.double() - torch.cat(wants)).abs()
    assert bool((err <= 3.2 * 2 ** -9 * torch.cat(bounds)).all()), (err / torch.cat(bounds)).max().item() * 2 ** 9
