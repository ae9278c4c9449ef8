"""Partial results of decoded tokens merged and gated in one launch, against float64 over the same partial results.

Tolerance: the merged row and the gated one are each rounded to bf16's 8 significant bits, half of the last place or 2^-8 of the
value at most, and 2^-20 of the largest for the fp32 sums over up to 256 ranges."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens, heads, dim, parts", [(1, 1, 16, 2), (1, 32, 64, 32), (3, 5, 96, 33), (2, 4, 256, 7), (5, 3, 80, 256), (2, 2, 128, 65)])
@pytest.mark.parametrize("act, mul", [("sigmoid", 1.0), ("silu", 0.5), (None, 0.25)])
def test_partial_results_merged_and_gated(tokens, heads, dim, parts, act, mul, gpu):
    g = torch.Generator().manual_seed(dim + parts)
    o = torch.randn((tokens * heads, parts, dim), generator=g)
    ml = torch.stack([torch.randn((tokens * heads, parts), generator=g) * 3, torch.rand((tokens * heads, parts), generator=g) + 0.1], -1)
    ml[:, 1::3, 0] = float("-inf")                      # ranges in which a row sees no key
    o[:, 1::3], ml[:, 1::3, 1] = 0.0, 0.0
    width = heads * dim
    gate = torch.randn((tokens, width + 24), generator=g).bfloat16()
    out = torch.full((tokens, width + 16), 7.0, dtype=torch.bfloat16, device=gpu)
    x = K.AttentionPartials(o.to(gpu), ml.to(gpu), tokens, heads)
    K.attention_merge_gated(x, out, 8, None if act is None else gate.to(gpu), 16, act or "sigmoid", mul)
    w = torch.exp2(ml[..., 0].double() - ml[..., 0].double().max(-1, keepdim=True).values)
    want = ((o.double() * w[..., None]).sum(1) / (ml[..., 1].double() * w).sum(1)[:, None]).view(tokens, width) * mul
    if act is not None:
        z = gate[:, 16:16 + width].double()
        want = want * (torch.sigmoid(z) if act == "sigmoid" else z * torch.sigmoid(z))
    got = out.double().cpu()
    assert ((got[:, 8:8 + width] - want).abs() <= 2.01 * 2.0 ** -8 * want.abs() + 2.0 ** -20 * want.abs().max()).all()
    assert (got[:, :8] == 7.0).all() and (got[:, 8 + width:] == 7.0).all()
    with pytest.raises(K.KernelError):
        K.attention_merge_gated(x, out, 17, None, 0, "sigmoid", mul)
