"""Attention of prompts over expanded keys and values: every way its workgroups share tokens and keys, at the edges of their blocks."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K
from kv_cache_optimization_for_llm_amd.parts.rotary import RotaryEncoding

pytestmark = pytest.mark.gpu


# heads and entries (first position, tokens): 16 tokens a wavefront (short contexts; many workgroups), two parts of the keys (with few and
# with many heads to expand), four parts (one token past a block of 128 keys, one short of it, entries that differ)
@pytest.mark.parametrize("heads, entries", [(3, [(0, 65), (447, 64), (31, 1)]), (56, [(0, 897)]), (20, [(13, 900)]), (40, [(3, 830), (0, 64)]),
                                            (2, [(0, 1025), (895, 128)]), (3, [(639, 128), (700, 67), (0, 5)]), (1, [(2100, 63)])])
@pytest.mark.parametrize("scale", [192 ** -0.5, -0.05, 0.0])
def test_every_share_of_tokens_and_keys(heads, entries, scale, gpu):
    d, rot, rank, page, T = 128, 64, 64, 16, sum(n for _, n in entries)
    g = torch.Generator(device=gpu).manual_seed(heads)
    rnd = lambda *s, by=1.0: (torch.randn(*s, generator=g, device=gpu) * by).to(torch.bfloat16)
    context = max(s + n for s, n in entries)
    blocks = -(-context // page)
    cache = rnd(len(entries) * blocks, page, rank + rot)
    table = torch.arange(len(entries) * blocks, dtype=torch.int32, device=gpu).flip(0).view(len(entries), blocks)
    q, up_k, up_v = rnd(T, heads, d + rot), rnd(heads * d, rank, by=rank ** -0.5), rnd(heads * d, rank, by=rank ** -0.5)
    cos, sin = RotaryEncoding(head_dim=rot, max_positions=4096, theta=10000.0, frequencies="plain_f64", pairing="half").tables(gpu)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)
    first = [0]
    for _, n in entries:
        first.append(first[-1] + n)
    out = torch.full((T, heads * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    K.latent_prompt(q, cache, K.moe_tiled_weight(torch.cat([up_k, up_v])[None])[0], out, table, i32(list(range(len(entries)))), i32(first),
                    i32([s for s, _ in entries]), cos, sin, False, scale, context, max(n for _, n in entries))
    for e, (start, n) in enumerate(entries):
        rows = cache[table[e].long()].reshape(-1, rank + rot)[:start + n].double()
        k = torch.cat([(rows[:, :rank] @ up_k.double().T).view(-1, heads, d), rows[:, None, rank:].expand(-1, heads, -1)], -1)
        v = (rows[:, :rank] @ up_v.double().T).view(-1, heads, d)
        x, pos = q[first[e]:first[e] + n].double(), torch.arange(start, start + n, device=gpu)
        c, s = cos.double()[pos][:, None], sin.double()[pos][:, None]
        a, b = x[..., d:d + rot // 2], x[..., d + rot // 2:]
        x = torch.cat([x[..., :d], a * c - b * s, b * c + a * s], -1)
        score = torch.matmul(x.transpose(0, 1).contiguous(), k.permute(1, 2, 0).contiguous()) * scale
        score = score.masked_fill(torch.arange(start + n, device=gpu)[None, None, :] > pos[None, :, None], float("-inf"))
        want = torch.matmul(torch.softmax(score, -1), v.transpose(0, 1).contiguous()).transpose(0, 1).reshape(n, heads * d)
        got = out[first[e]:first[e] + n].double()
        # keys, values, rotated queries, probabilities and results are rounded to bf16 (2^-9 each, relative): their squares add up
        assert (got - want).norm() <= 2.0 ** -9 * 5 ** 0.5 * 1.5 * want.norm(), e
