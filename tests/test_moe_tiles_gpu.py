"""The experts' products in blocks of as many tiles of an expert as a plan says (csrc/moe_tiles.hip), against 64 bits."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu
ACT = {"silu": torch.nn.functional.silu, "relu": torch.relu, "gelu": torch.nn.functional.gelu,
       "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh"), "relu2": lambda z: torch.relu(z) ** 2}


def rnd(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).bfloat16()


# outputs below, at and past a workgroup's, K of one stage, fewer than the ring holds and more; experts nobody chose; runs of one row and of
# several blocks; lists in groups; one token an expert
@pytest.mark.parametrize("plan", range(9))
@pytest.mark.parametrize("T, E, top, H, ff, act, gated, group", [
    (1, 1, 1, 64, 64, "silu", True, 1), (37, 5, 2, 64, 72, "silu", True, 4), (700, 9, 4, 192, 200, "gelu_tanh", True, 1),
    (513, 3, 3, 128, 320, "gelu", False, 8), (300, 40, 6, 320, 64, "relu2", False, 1), (1100, 4, 1, 64, 144, "swish_clamped", True, 1)])
def test_experts_products_of_every_shape(T, E, top, H, ff, act, gated, group, plan, gpu):
    g = torch.Generator().manual_seed(T)
    idx = torch.rand((T, E), generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
    if E > 4:
        idx[idx == 3] = E                                   # (an expert nobody chose; those slots name none)
    x, wgt = rnd((T, H), 1), torch.rand((T, top), generator=g)
    up, ff_k = rnd((E, (2 if gated else 1) * ff, H), 2, H ** -0.5), (ff + 63) // 64 * 64
    down, hidden = rnd((E, H, ff_k), 3, ff ** -0.5), None
    tiles = K.moe_tiles(T * top, E, group)
    slot = torch.empty(tiles * K.MOE_TILE, dtype=torch.int32, device=gpu)
    tile_expert = torch.empty(tiles, dtype=torch.int32, device=gpu)
    K.moe_align(idx.to(gpu), E, slot, tile_expert, group)
    sl, flat, limit = slot.cpu().long(), idx.view(-1).long(), 0.9
    used = sl >= 0
    hidden = rnd((tiles * K.MOE_TILE, ff_k), 4)
    hidden[~used] = float("nan")                            # (places without a slot hold anything)
    place = torch.zeros(T * top, dtype=torch.long)
    place[sl[used]] = used.nonzero()[:, 0]
    want_act = torch.zeros(T * top, ff, dtype=torch.float64)
    want = torch.full((T * top, H), 7.0, dtype=torch.float64)
    for e in range(E):
        m = flat == e
        z = x.double().repeat_interleave(top, 0)[m] @ up[e].double().T * wgt.view(-1)[m].double()[:, None]
        if act == "swish_clamped":
            gate, u = z[:, 0::2].clamp(max=limit), z[:, 1::2].clamp(-limit, limit)
            want_act[m] = gate * torch.sigmoid(1.702 * gate) * (u + 1)
        else:
            want_act[m] = ACT[act](z[:, 0::2]) * z[:, 1::2] if gated else ACT[act](z)
        want[m] = hidden[place[m]].double() @ down[e].double().T * wgt.view(-1)[m].double()[:, None]
    got = torch.full((tiles * K.MOE_TILE, ff), 3.0, dtype=torch.bfloat16, device=gpu)
    K.moe_expert_tiles(x.to(gpu), K.moe_tiled_weight(up.to(gpu)), got, slot, tile_expert, top, plan, activation=act,
                       slot_weight=wgt.to(gpu), gated=gated, limit=limit)
    out = torch.full((T * top, H), 7.0, device=gpu)
    K.moe_expert_tiles(hidden.to(gpu), K.moe_tiled_weight(down.to(gpu)), out, slot, tile_expert, top, plan, slot_weight=wgt.to(gpu))
    # a result rounded to 16 bits: 2^-9 of it at most, and 32-bit sums of K products of numbers around 1 behind it
    got = got.cpu()
    err = (got[used].double() - want_act[sl[used]]).abs()
    assert (err <= 2.0 ** -8 * want_act[sl[used]].abs() + 2.0 ** -20 * H ** 0.5).all(), err.max()
    assert (got[~used] == 3.0).all()                        # nothing else is written
    assert ((out.cpu().double() - want).abs() <= 2.0 ** -18 * ff_k ** 0.5).all()


def test_plans_of_sizes_it_does_not_take():
    assert K.moe_tiles_plan(8192, 16, 4, 1536, 96, False) == -1         # K in stages of 64
    assert K.moe_tiles_plan(8192, 16, 4, 1544, 128, False) == -1        # whole tiles
    assert K.moe_tiles_plan(1 << 20, 16, 4, 1536, 128, False) == -1     # a list of more tiles than a wavefront's masks hold
    assert K.moe_tiles_plan(8192, 16, 4, 1536, 2048, False) >= 0 and K.moe_tiles_plan(8192, 16, 4, 2048, 768, True) >= 0
    assert K.moe_tiles_plan(8192, 4, 4, 2048, 1024, True) == -1         # its rows take as long to write as to multiply
    for slots, experts in ((40000, 64), (60000, 16), (64000, 4), (65000, 1), (30000, 300)):      # what is taken is taken over a list in groups too
        for second in (False, True):
            assert K.moe_tiles_plan(slots, experts, 1, 256, 4096, second) < 0 or K.moe_tiles(slots, experts, 8) <= 4096
    with pytest.raises(K.KernelError):
        x = torch.zeros((16, 64), dtype=torch.bfloat16, device="cuda")
        ints = torch.zeros(16, dtype=torch.int32, device="cuda")
        K.moe_expert_tiles(x, torch.zeros((1, 64, 64), dtype=torch.bfloat16, device="cuda"), x, ints, ints[:1], 1, 99, activation="silu")
