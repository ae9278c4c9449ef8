"""Rotation and cache write of many tokens at a time (csrc/rope_cache.hip) against the same tokens a few at a time, bit for bit."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


def _slots(page, pages):
    """Decoded tokens, tokens without a slot, and portions that begin and end anywhere in a page and go to the next one; as often as
    takes 1,536 tokens, from which the kernel for many takes any geometry."""
    g = torch.Generator().manual_seed(page)
    order, slots = torch.randperm(pages, generator=g).tolist(), []
    for first, count in 10 * ((3, 1), (0, 1), (page - 1, 1), (5, 2 * page), (0, 3 * page), (0, 37), (7, 9), (8 % page, 41), (1, 3 * page + 2)):
        mine = [order.pop() for _ in range((first + count - 1) // page + 1)]
        slots += [mine[p // page] * page + p % page for p in range(first, first + count)]
    slots[11] = slots[60] = slots[-1] = -1
    return slots


@pytest.mark.parametrize("cached", [True, False])
@pytest.mark.parametrize("nq, nkv, d, page", [(32, 8, 64, 16), (5, 3, 128, 16), (3, 1, 16, 8), (7, 2, 96, 32), (2, 2, 256, 16), (40, 17, 48, 16)])
def test_many_tokens_are_rotated_and_cached_as_few(nq, nkv, d, page, cached, gpu):
    pages = 400
    slots = torch.tensor(_slots(page, pages), dtype=torch.int32, device=gpu)
    T = slots.numel()
    assert K.rope_tokens_wide(T, nkv, d, True) and not K.rope_tokens_wide(64, nkv, d, True) and T % 16
    g = torch.Generator().manual_seed(d)
    qkv = torch.randn((T, (nq + 2 * nkv) * d), generator=g).bfloat16().to(gpu)
    pos = torch.randint(0, 300, (T,), generator=g).to(torch.int32).to(gpu)
    cos, sin = torch.randn((300, d // 2), generator=g).to(gpu), torch.randn((300, d // 2), generator=g).to(gpu)

    def run(step):
        x = qkv.clone()
        k = K.keys_to_pages(torch.full((pages, nkv, page, d), 3.0, dtype=torch.bfloat16, device=gpu))
        v = torch.full((pages, nkv, d, page), 5.0, dtype=torch.bfloat16, device=gpu)
        for t in range(0, T, step):
            args = (k, v, slots[t:t + step].contiguous(), page) if cached else (None, None, None, 0)
            K.rope_kv_write(x[t:t + step], pos[t:t + step].contiguous(), nq, nkv, d, cos, sin, *args)
        return x, k, v
    for many, few in zip(run(T), run(64)):
        assert torch.equal(many, few)
    assert not torch.equal(run(T)[0][:, :nq * d], qkv[:, :nq * d])
