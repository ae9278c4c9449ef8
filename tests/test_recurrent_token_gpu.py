"""One token of every request through a recurrent mixer in one launch, against the launches it stands for: the same bits."""
import numpy as np
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


def ints(a):
    return torch.tensor(np.asarray(a), dtype=torch.int32, device="cuda")


def numbers(shape, g, dtype=torch.float32, scale=1.0):
    return (torch.randn(shape, generator=g) * scale).to(dtype).to("cuda")


def seats_of(entries, g):
    return ints(torch.randperm(entries + 3, generator=g)[:entries].numpy())


def same(pairs):
    for got, want in pairs:
        assert torch.equal(got, want), (int((got != want).sum()), got.numel(), float((got.float() - want.float()).abs().max()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, kv_heads, dim, vdim, taps", [(8, 4, 128, 128, 4), (2, 2, 64, 64, 4), (3, 1, 100, 40, 3), (32, 1, 20, 8, 2), (1, 1, 128, 256, 4), (6, 2, 16, 72, 4)])
@pytest.mark.parametrize("channel, act, entries", [(False, "silu", 1), (True, "sigmoid", 5)])
def test_delta_rule(heads, kv_heads, dim, vdim, taps, channel, act, entries, dtype, gpu):
    g = torch.Generator().manual_seed(heads * dim + vdim)
    C, S = 2 * kv_heads * dim + heads * vdim, heads * dim * vdim
    col0, gate_off = 16, 16 + (C + 2 * heads + 7) // 8 * 8
    y = numbers((entries, gate_off + heads * vdim), g, dtype)
    conv, norm = numbers((C, taps), g, scale=0.5), numbers((vdim,), g)
    a_log, dt_bias = numbers((heads,), g), numbers((heads,), g)
    alpha = torch.sigmoid(numbers((entries, heads * dim), g) + 2) if channel else None
    state = numbers((entries + 3, (4 + S + C * (taps - 1) + 3) // 4 * 4), g)
    starts, seats = ints(np.arange(entries + 1)), seats_of(entries, g)
    got, want = state.clone(), state.clone()
    out = torch.zeros((entries, 8 + heads * vdim), dtype=dtype, device="cuda")
    ref = out.clone()
    assert K.gated_delta_rule_token(y, col0, conv, got, 4, 4 + S, col0 + C, col0 + C + heads, None if channel else a_log, None if channel else dt_bias,
                                    alpha, 1e-6, norm, 1e-5, y, gate_off, act, out, 8, 0.7, starts, seats, heads, kv_heads, dim, vdim)
    qkv, o = torch.empty((entries, C), device="cuda"), torch.empty((entries, heads * vdim), device="cuda")
    K.causal_conv_act(y, col0, conv, qkv, want, 4 + S, starts, seats, 1)
    K.gated_delta_rule(qkv, y, col0 + C, col0 + C + heads, None if channel else a_log, None if channel else dt_bias, o, want, 4, starts, seats,
                       heads, kv_heads, dim, vdim, channel_decay=alpha)
    K.head_norm_gate(o, norm, 1e-5, y, gate_off, ref, 8, heads, vdim, act, 0.7)
    same([(out, ref), (got, want)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, dim, vdim, rank, entries", [(16, 64, 128, 16, 1), (2, 128, 256, 64, 3), (3, 20, 8, 8, 4), (5, 100, 40, 24, 2)])
def test_linear_attention(heads, dim, vdim, rank, entries, dtype, gpu):
    g = torch.Generator().manual_seed(heads * dim + vdim)
    q, k, v = 8, 8 + heads * dim, 8 + 2 * heads * dim
    gate = (v + heads * vdim + 7) // 8 * 8
    a1 = gate + heads * vdim
    y = numbers((entries, (a1 + rank + 7) // 8 * 8), g, dtype)
    a2, bias, norm = numbers((heads * dim, rank), g, dtype, 0.3), numbers((heads * dim,), g), numbers((vdim,), g)
    state = numbers((entries + 3, 4 + heads * dim * vdim), g)
    starts, seats = ints(np.arange(entries + 1)), seats_of(entries, g)
    got, want = state.clone(), state.clone()
    out = torch.zeros((entries, heads * vdim), dtype=dtype, device="cuda")
    ref = out.clone()
    assert K.gated_linear_attention_token(y, q, k, v, a1, a2, bias, 3.5, dim ** -0.5, got, 4, norm, 1e-5, gate, "silu", out, 0, 1.0, starts, seats,
                                          heads, dim, vdim)
    alpha = K.small_product_f32(y[:, a1:a1 + rank], a2, torch.empty((entries, heads * dim), device="cuda"), bias=bias, decay_tau=3.5)
    o = torch.empty((entries, heads * vdim), device="cuda")
    K.gated_linear_attention(y, q, k, v, alpha, dim ** -0.5, o, want, 4, starts, seats, heads, dim, vdim)
    K.head_norm_gate(o, norm, 1e-5, y, gate, ref, 0, heads, vdim, "silu")
    same([(out, ref), (got, want)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads, groups, n, vdim, norm_groups, taps, entries", [(32, 4, 128, 64, 4, 4, 2), (8, 8, 100, 24, 8, 3, 1), (4, 2, 16, 128, 4, 4, 5),
                                                                               (3, 3, 33, 8, 3, 2, 3), (2, 2, 128, 512, 2, 4, 1), (16, 2, 64, 16, 16, 4, 2),
                                                                               (6, 3, 128, 64, 3, 4, 2), (3, 1, 100, 64, 1, 4, 3)])
def test_state_space(heads, groups, n, vdim, norm_groups, taps, entries, dtype, gpu):
    g = torch.Generator().manual_seed(heads * n + vdim)
    inner, S = heads * vdim, heads * n * vdim
    C = inner + 2 * groups * n
    dt_off = (inner + C + 7) // 8 * 8
    y = numbers((entries, (dt_off + heads + 7) // 8 * 8), g, dtype)
    conv, cb, norm = numbers((C, taps), g, scale=0.5), numbers((C,), g), numbers((inner,), g)
    a_log, dt_bias, skip = (numbers((heads,), g) for _ in range(3))
    state = numbers((entries + 3, (S + C * (taps - 1) + 3) // 4 * 4), g)
    starts, seats = ints(np.arange(entries + 1)), seats_of(entries, g)
    got, want = state.clone(), state.clone()
    out = torch.zeros((entries, inner), dtype=dtype, device="cuda")
    ref = out.clone()
    assert K.state_space_token(y, inner, conv, cb, got, 0, S, dt_off, a_log, dt_bias, skip, norm, 1e-5, 0, out, 0, 0.5, starts, seats, heads, groups,
                               n, vdim, norm_groups)
    xbc, o = torch.empty((entries, C), dtype=dtype, device="cuda"), torch.empty((entries, inner), device="cuda")
    K.causal_conv_act(y, inner, conv, xbc, want, S, starts, seats, 1, out_bias=cb)
    K.state_space(xbc, y, dt_off, a_log, dt_bias, skip, o, want, 0, starts, seats, heads, groups, n, vdim, [1] * entries)
    K.head_norm_gate(o, norm, 1e-5, y, 0, ref, 0, norm_groups, inner // norm_groups, "silu", 0.5, gate_first=True)
    same([(out, ref), (got, want)])


def test_what_does_not_fit_is_left_alone(gpu):
    """Sizes past what a workgroup holds, and rows, states and gates at no multiple of 16 bytes: False, and nothing is written."""
    g = torch.Generator().manual_seed(0)
    starts, seats = ints([0, 1]), ints([0])

    def delta(heads=2, dim=64, vdim=64, taps=4, gate_off=0, out_off=0, state_off=0, wide=0):
        C, S = 2 * dim + heads * vdim, heads * dim * vdim
        y = numbers((1, (C + 2 * heads + heads * vdim + 15) // 8 * 8 + wide), g, torch.bfloat16)
        state = torch.ones((1, (state_off + S + C * (taps - 1) + 3) // 4 * 4), device="cuda")
        out = torch.zeros((1, heads * vdim + 8), dtype=torch.bfloat16, device="cuda")
        one = torch.ones(heads, device="cuda")
        done = K.gated_delta_rule_token(y, 0, numbers((C, taps), g), state, state_off, state_off + S, C, C + heads, one, one, None, 1e-6,
                                        numbers((vdim,), g), 1e-5, y, gate_off, "silu", out, out_off, 1.0, starts, seats, heads, 1, dim, vdim)
        assert done or (not out.any() and bool((state == 1).all()))
        return done
    assert delta()
    for other in (dict(heads=5), dict(dim=136), dict(vdim=60), dict(taps=5), dict(taps=1), dict(gate_off=4), dict(out_off=4), dict(state_off=2), dict(wide=4)):
        assert not delta(**other), other


def test_state_space_of_many_requests(gpu):
    """fp32 rows whose groups' columns take two passes stay with the three launches where workgroups are many."""
    g = torch.Generator().manual_seed(0)
    H, n, dv, taps = 8, 16, 64, 2
    inner, S, C = H * dv, H * n * dv, H * dv + 2 * n
    for dtype, entries, fits in ((torch.float32, 768, True), (torch.float32, 769, False), (torch.bfloat16, 769, True)):
        y = numbers((entries, inner + C + H), g, dtype)
        state, out = torch.zeros((entries, S + C), device="cuda"), torch.zeros((entries, inner), dtype=dtype, device="cuda")
        one = torch.ones(H, device="cuda")
        assert fits == K.state_space_token(y, inner, numbers((C, taps), g), None, state, 0, S, inner + C, one, one, one, torch.ones(inner, device="cuda"), 1e-5,
                                           0, out, 0, 1.0, ints(np.arange(entries + 1)), ints(np.arange(entries)), H, 1, n, dv, 1)
        assert bool(out.any()) == bool(state.any()) == fits


def without_a_token(run, width, state):
    """``run(state, out, starts, seats)`` over entries some of which have no token, against the others alone: their outputs and states, and
    seats without a token keep theirs, the convolution's inputs among it."""
    got, want = state.clone(), state.clone()
    out = torch.zeros((2, width), device="cuda")
    ref = out.clone()
    assert run(got, out, ints([0, 0, 1, 1, 2]), ints([3, 0, 4, 2]))
    assert run(want, ref, ints([0, 1, 2]), ints([0, 2]))
    same([(out, ref), (got, want)])
    assert torch.equal(got[[1, 3, 4]], state[[1, 3, 4]]) and not torch.equal(got[[0, 2]], state[[0, 2]])


def test_entries_without_a_token(gpu):
    """More entries than rows: an entry without a token leaves its seat's state as it is."""
    g = torch.Generator().manual_seed(1)
    heads, dim, vdim, rank = 2, 64, 64, 16
    y = numbers((2, 4 * heads * dim + 16), g)
    a2, bias, norm = numbers((heads * dim, rank), g, scale=0.3), numbers((heads * dim,), g), numbers((vdim,), g)
    offs = (0, heads * dim, 2 * heads * dim, 4 * heads * dim)
    without_a_token(lambda state, out, starts, seats: K.gated_linear_attention_token(
        y, *offs, a2, bias, 3.5, 0.125, state, 0, norm, 1e-5, 3 * heads * dim, "silu", out, 0, 1.0, starts, seats, heads, dim, vdim),
        heads * vdim, numbers((5, heads * dim * vdim), g))


def test_delta_rule_of_entries_without_a_token(gpu):
    g = torch.Generator().manual_seed(2)
    heads, dim, vdim, taps = 2, 64, 64, 4
    C, S = 2 * dim + heads * vdim, heads * dim * vdim
    y, conv, norm, one = numbers((2, C + 8 + heads * vdim), g), numbers((C, taps), g, scale=0.5), numbers((vdim,), g), torch.ones(heads, device="cuda")
    without_a_token(lambda state, out, starts, seats: K.gated_delta_rule_token(
        y, 0, conv, state, 0, S, C, C + heads, one, one, None, 1e-6, norm, 1e-5, y, C + 8, "silu", out, 0, 1.0, starts, seats, heads, 1, dim, vdim),
        heads * vdim, numbers((5, S + C * (taps - 1)), g))


def test_state_space_of_entries_without_a_token(gpu):
    g = torch.Generator().manual_seed(3)
    heads, groups, n, vdim, taps = 4, 2, 32, 64, 4
    inner, S = heads * vdim, heads * n * vdim
    C = inner + 2 * groups * n
    y, conv, norm, one = numbers((2, inner + C + 8), g), numbers((C, taps), g, scale=0.5), numbers((inner,), g), torch.ones(heads, device="cuda")
    without_a_token(lambda state, out, starts, seats: K.state_space_token(
        y, inner, conv, None, state, 0, S, inner + C, one, one, one, norm, 1e-5, 0, out, 0, 1.0, starts, seats, heads, groups, n, vdim, groups),
        inner, numbers((5, S + C * (taps - 1)), g))
