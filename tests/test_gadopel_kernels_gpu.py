"""The kernels behind the Gadopel parts, each alone against the plain functions of
``plain_gadopel``: layer norm over a 32-bit stream, gated activations (own kernel and product
epilogue), interleaved / partial / YaRN rotation with unit-norm heads and the cache write,
attention with a window that keeps first positions, sinks and a value size of its own, and
attention over low-rank rows.  Where random numbers would hide a fault - one far key among
hundreds, a key just inside or just outside a window, at a page's edge - one query and one key
are scaled so that this key's score stands out when (and only when) it is visible."""
import numpy as np
import pytest
import torch

import plain_gadopel as plain
from kv_cache_optimization_for_llm_amd.ops import kernels as K
from kv_cache_optimization_for_llm_amd.ops import latent_attention as lat_ops
from kv_cache_optimization_for_llm_amd.parts.linear import Linear
from kv_cache_optimization_for_llm_amd.parts.rotary import RotaryEncoding

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
TOL = {"float32": 2e-5, "bfloat16": 2e-2}


def rnd(shape, seed, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def close(got, want, tol, what=""):
    got, want = got.double().cpu(), want.double().cpu()
    err = (got - want).abs().max().item() / max(want.abs().max().item(), 1e-9)
    assert err <= tol, f"{what}: off by {err:.3g} of the largest value (limit {tol})"


@pytest.mark.parametrize("out_dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [72, 96, 1000])
def test_layer_norm_adds_pending_outputs_and_writes_two_copies(width, out_dtype, gpu):
    x = rnd((7, width), 1, scale=3.0) + 1.5
    d1, d2 = rnd((7, width), 2, DT[out_dtype]), rnd((7, width), 3, DT[out_dtype])
    w1, w2 = (1 + 0.1 * rnd((width,), 4)).to(DT[out_dtype]), (1 + 0.1 * rnd((width,), 5)).to(DT[out_dtype])
    xs = x.to(gpu)
    o1 = torch.empty((7, width), dtype=DT[out_dtype], device=gpu)
    o2 = torch.empty_like(o1)
    K.layernorm(xs, w1.to(gpu), 1e-5, o1, deltas=(d1.to(gpu), d2.to(gpu)), weight2=w2.to(gpu), out2=o2)
    total = x.double() + d1.double() + d2.double()
    close(xs, total, 1e-6, "the stream after the add")          # the stream itself stays 32-bit
    close(o1, plain.layer_norm(total, w1.double(), 1e-5), TOL[out_dtype], "first copy")
    close(o2, plain.layer_norm(total, w2.double(), 1e-5), TOL[out_dtype], "second copy")
    # gathered rows: nothing is written back, a row named twice is not added twice
    idx = torch.tensor([6, 0, 6], dtype=torch.int32, device=gpu)
    before = xs.clone()
    o3 = torch.empty((3, width), dtype=DT[out_dtype], device=gpu)
    K.layernorm(xs, w1.to(gpu), 1e-5, o3, deltas=(d1.to(gpu),), row_idx=idx)
    assert torch.equal(xs, before)
    tol = TOL[out_dtype]
    close(o3, plain.layer_norm((total + d1.double())[[6, 0, 6]], w1.double(), 1e-5), tol, "gathered rows")


@pytest.mark.parametrize("activation", ["relu", "gelu_tanh", "silu"])
@pytest.mark.parametrize("rows", [1, 2, 8, 40, 200])
def test_gated_activations_alone_and_in_the_product(rows, activation, gpu):
    act = {"relu": torch.relu, "silu": torch.nn.functional.silu,
           "gelu_tanh": lambda z: 0.5 * z * (1 + torch.tanh(0.7978845608028654 * (z + 0.044715 * z ** 3)))}[activation]
    inter, width = 96, 64
    x = rnd((rows, width), 1, torch.bfloat16)
    w = rnd((2 * inter, width), 2, torch.bfloat16, 0.3)
    gu = x.double() @ w.double().T
    want = act(gu[:, :inter]) * gu[:, inter:]
    for dtype in ("float32", "bfloat16"):
        out = torch.empty((rows, inter), dtype=DT[dtype], device=gpu)
        K.act_mul(gu.to(DT[dtype]).to(gpu), out, activation)
        close(out, want, TOL[dtype], f"act_mul {dtype}")
    lin = Linear(w.to(gpu), halves=2)
    if lin.fused_kernel(rows, torch.bfloat16) is not None:
        out = torch.empty((rows, inter), dtype=torch.bfloat16, device=gpu)
        lin.gated(x.to(gpu), out, activation)
        close(out, want, 2e-2, "the product's epilogue")


def cache_for(length, page_size, seed):
    """A block table that scatters the positions' pages, and the slots of positions 0..length-1."""
    blocks = (length + page_size - 1) // page_size
    perm = np.random.default_rng(seed).permutation(blocks + 3)[:blocks]
    table = torch.full((2, blocks + 2), -1, dtype=torch.int32)
    table[1, :blocks] = torch.from_numpy(perm.astype(np.int32))
    pos = np.arange(length)
    slots = torch.from_numpy((perm[pos // page_size] * page_size + pos % page_size).astype(np.int32))
    return table, slots, blocks + 3


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads, kv_heads, dim, vdim, rot, interleaved, unit", [
    (4, 2, 32, 16, 16, True, True), (3, 3, 20, 20, 12, True, True), (2, 1, 64, 64, 64, True, False),
    (6, 2, 48, 24, 32, False, True), (2, 2, 16, 40, 0, True, True)])
def test_rotation_unit_norm_and_cache_write(heads, kv_heads, dim, vdim, rot, interleaved, unit, dtype, gpu):
    T, page = 37, 8
    eps = 1e-5
    scaling = {"factor": 8.0, "original": 48, "fast": 6.0, "slow": 1.5}
    table, slots, pages = cache_for(T, page, 3)
    qkv = rnd((T, heads * dim + kv_heads * dim + kv_heads * vdim), 7, DT[dtype])
    positions = torch.arange(100, 100 + T, dtype=torch.int32)
    cos = sin = None
    if rot:
        enc = RotaryEncoding(head_dim=dim, rotary_dim=rot, max_positions=256, theta=777.0, frequencies="yarn",
                             frequency_params=scaling, magnitude=0.1 * np.log(8.0) + 1,
                             pairing="interleaved" if interleaved else "half")
        cos, sin = enc.tables(gpu)
    k_cache = torch.zeros((pages, *K.k_page_shape(kv_heads, dim)[:2], page, K.k_chunk(dim)), dtype=DT[dtype], device=gpu)
    v_cache = torch.zeros((pages, kv_heads, vdim, page), dtype=DT[dtype], device=gpu)
    dev = qkv.to(gpu)
    K.qk_encode_cache(dev, positions.to(gpu), heads, kv_heads, dim, vdim, cos, sin, interleaved,
                      eps if unit else None, k_cache, v_cache, slots.to(gpu))
    src = qkv.double()
    q = src[:, :heads * dim].view(T, heads, dim)
    k = src[:, heads * dim:(heads + kv_heads) * dim].view(T, kv_heads, dim)
    v = src[:, (heads + kv_heads) * dim:].view(T, kv_heads, vdim)
    if rot:
        freqs, mag = plain.rotary_frequencies(rot, 777.0, scaling)
        q = plain.rotate(q, positions, freqs, mag, interleaved)
        k = plain.rotate(k, positions, freqs, mag, interleaved)
    if unit:
        q, k = plain.unit_rms(q, eps), plain.unit_rms(k, eps)
    close(dev[:, :heads * dim].view(T, heads, dim), q, TOL[dtype], "queries")
    got_k = K.pages_to_keys(k_cache).reshape(pages, kv_heads, page, dim)
    sl = slots.long()
    close(got_k[sl // page, :, sl % page], k, TOL[dtype], "cached keys")
    close(v_cache[sl // page, :, :, sl % page], v, 1e-9, "cached values")


def standout(q, k, query_pos, key_pos, head, kv_head, strength=12.0):
    """Makes key ``key_pos`` the one query ``query_pos`` of ``head`` scores highest by far."""
    direction = q[query_pos, head] / q[query_pos, head].norm()
    k[key_pos, kv_head] = direction * strength
    q[query_pos, head] = direction * strength


CASES = [  # (length, window, keep_first, query position, key that stands out)
    (300, 0, 0, 299, 0), (300, 0, 0, 299, 157),                     # far keys, no window
    (300, 44, 18, 299, 256), (300, 44, 18, 299, 255),              # just inside / outside the window
    (300, 44, 18, 299, 17), (300, 44, 18, 299, 18),                # the last kept position / the first that is not
    (300, 44, 18, 45, 18), (300, 44, 18, 61, 18), (300, 44, 18, 62, 18),
    (130, 16, 16, 129, 15), (130, 16, 16, 129, 16), (130, 16, 16, 129, 113), (130, 16, 16, 129, 114),   # page edges
    (70, 64, 0, 69, 5), (70, 64, 0, 69, 6), (5, 3, 1, 4, 0), (5, 3, 1, 4, 1), (1, 0, 0, 0, 0),
]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("length, window, keep_first, qpos, kpos", CASES)
def test_attention_sees_exactly_the_visible_keys(length, window, keep_first, qpos, kpos, dtype, gpu):
    heads, kv_heads, dim, vdim, page, scale = 4, 2, 24, 40, 16, 0.3
    q, k, v = rnd((length, heads, dim), 1), rnd((length, kv_heads, dim), 2), rnd((length, kv_heads, vdim), 3)
    standout(q, k, qpos, kpos, head=2, kv_head=1)
    v[kpos, 1] = 5.0
    q, k, v = (t.to(DT[dtype]) for t in (q, k, v))
    sinks = torch.tensor([0.5, -1.0, 2.0, 0.0])
    table, slots, pages = cache_for(length, page, 11)
    k_cache = torch.zeros((pages, *K.k_page_shape(kv_heads, dim)[:2], page, K.k_chunk(dim)), dtype=DT[dtype], device=gpu)
    v_cache = torch.full((pages, kv_heads, vdim, page), float("nan"), dtype=DT[dtype], device=gpu)      # pages of others
    sl = slots.long()
    kp = K.pages_to_keys(k_cache).reshape(pages, kv_heads, page, dim)
    kp[sl // page, :, sl % page] = k.to(gpu)
    k_cache.copy_(K.keys_to_pages(kp))
    v_cache[sl // page, :, :, sl % page] = v.to(gpu)
    rows = sorted({qpos, 0, length - 1, min(length - 1, max(0, keep_first)), length // 2})
    tok_pos = torch.tensor(rows, dtype=torch.int32)
    out = torch.empty((len(rows), heads * vdim), dtype=DT[dtype], device=gpu)
    K.attention_rowwise(q[rows].reshape(len(rows), -1).contiguous().to(gpu), heads * dim, out, k_cache, v_cache,
                        table.to(gpu), torch.ones(len(rows), dtype=torch.int32, device=gpu), tok_pos.to(gpu),
                        heads, kv_heads, dim, scale, window, keep_first, sinks.to(gpu), vdim)
    qd, kd, vd = q.double(), k.double().repeat_interleave(2, dim=1), v.double().repeat_interleave(2, dim=1)
    prob = plain.softmax_rows(torch.einsum("ihd,jhd->hij", qd, kd) * scale, plain.visible(length, window, keep_first),
                              sinks.double())
    want = torch.einsum("hij,jhd->ihd", prob, vd)[rows].reshape(len(rows), -1)
    assert torch.isfinite(out).all()
    close(out, want, TOL[dtype] * 5, "attention")
    seen = plain.visible(length, window, keep_first)[qpos, kpos].item()
    got = out.view(len(rows), heads, vdim)[rows.index(qpos), 2].float().mean().item()
    assert (got > 2.5) == bool(seen), f"the key that stands out is {'visible' if seen else 'hidden'}, the output says {got:.2f}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("length, window, keep_first, qpos, kpos", CASES)
def test_latent_attention_sees_exactly_the_visible_rows(length, window, keep_first, qpos, kpos, dtype, gpu):
    heads, rank, rot, page, scale = 3, 40, 8, 16, 0.25
    kd = rank + rot
    q, rows_kv = rnd((length, heads, kd), 4), rnd((length, 1, kd), 5)
    standout(q, rows_kv, qpos, kpos, head=1, kv_head=0, strength=14.0)
    q, rows_kv = q.to(DT[dtype]), rows_kv.to(DT[dtype])
    sinks = torch.tensor([1.0, -2.0, 0.3])
    table, slots, pages = cache_for(length, page, 13)
    cache = torch.full((pages, page, kd), float("nan"), dtype=DT[dtype], device=gpu)
    cache.view(-1, kd)[slots.long()] = rows_kv[:, 0].to(gpu)
    picks = sorted({qpos, 0, length - 1, length // 2})

    class Batch:
        tok_seat = torch.ones(len(picks), dtype=torch.int32, device=gpu)
        positions = torch.tensor(picks, dtype=torch.int32, device=gpu)

    class View:
        arrays = {"latent": cache}
        block_table = table.to(gpu)
        page_size = page

    out = torch.empty((len(picks), heads, rank), dtype=DT[dtype], device=gpu)
    lat_ops.latent_attention(q[picks].contiguous().to(gpu), out, View, Batch, scale, window, keep_first, sinks.to(gpu))
    qd, kdbl = q.double(), rows_kv.double().expand(length, heads, kd)
    prob = plain.softmax_rows(torch.einsum("ihd,jhd->hij", qd, kdbl) * scale, plain.visible(length, window, keep_first),
                              sinks.double())
    want = torch.einsum("hij,jd->ihd", prob, rows_kv.double()[:, 0, :rank])[picks]
    assert torch.isfinite(out).all()
    close(out, want, TOL[dtype] * 5, "latent attention")
    seen = plain.visible(length, window, keep_first)[qpos, kpos].item()
    weight = (out[picks.index(qpos), 1].double().cpu() @ rows_kv.double()[kpos, 0, :rank]) / rows_kv.double()[kpos, 0, :rank].norm() ** 2
    assert (weight.item() > 0.5) == bool(seen)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_low_rank_entry_is_normed_rotated_and_cached(dtype, gpu):
    T, heads, dim, rot, rank, page, eps = 21, 3, 16, 8, 40, 8, 1e-5
    kd = rank + rot
    y = rnd((T, heads * (dim + rot) + kd + heads), 3, DT[dtype])
    w = (1 + 0.2 * rnd((rank,), 4)).to(DT[dtype])
    positions = torch.arange(50, 50 + T, dtype=torch.int32)
    table, slots, pages = cache_for(T, page, 5)
    enc = RotaryEncoding(head_dim=rot, max_positions=128, theta=300.0, frequencies="plain_f64")
    cos, sin = enc.tables(gpu)
    cache = torch.zeros((pages, page, kd), dtype=DT[dtype], device=gpu)
    q_lat = torch.zeros((T, heads, kd), dtype=DT[dtype], device=gpu)
    K.latent_encode_cache(y.to(gpu), heads * (dim + rot), q_lat, cache, w.to(gpu), eps, cos, sin, positions.to(gpu),
                          slots.to(gpu), heads, dim, rank)
    freqs, mag = plain.rotary_frequencies(rot, 300.0)
    yd = y.double()
    q_rot = plain.rotate(yd[:, :heads * (dim + rot)].view(T, heads, dim + rot)[..., dim:], positions, freqs, mag, False)
    entry = yd[:, heads * (dim + rot):heads * (dim + rot) + kd]
    c = plain.unit_rms(entry[:, :rank], eps) * w.double()
    k_rot = plain.rotate(entry[:, rank:], positions, freqs, mag, False)
    close(q_lat[:, :, rank:], q_rot, TOL[dtype], "rotated query parts")
    got = cache.view(-1, kd)[slots.long().to(gpu)]
    close(got[:, :rank], c, TOL[dtype], "latent")
    close(got[:, rank:], k_rot, TOL[dtype], "rotated key part")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("x_pad, out_pad", [(5, 3), (8, 4), (0, 0)])
@pytest.mark.parametrize("rows, heads, n, k", [(1, 3, 40, 16), (9, 5, 24, 8), (130, 2, 70, 96), (3, 1, 8, 200),
                                               (1, 16, 512, 128), (40, 3, 128, 512), (300, 4, 48, 64)])
def test_per_head_products_into_column_ranges(rows, heads, n, k, x_pad, out_pad, dtype, gpu):
    """(bf16 rows whose strides are multiples of 8 and whose K has an instance take the matrix
    cores, everything else the plain kernel: both against the same sums)"""
    x_wide = rnd((rows, heads, k + x_pad), 1, DT[dtype]).to(gpu)
    out_wide = torch.zeros((rows, heads, n + out_pad), dtype=DT[dtype], device=gpu)
    w = rnd((heads, n, k), 2, DT[dtype], 0.3).to(gpu)
    lat_ops.heads_product(x_wide[:, :, :k], w, out_wide[:, :, :n])
    want = torch.einsum("thk,hnk->thn", x_wide[:, :, :k].double(), w.double())
    close(out_wide[:, :, :n], want, TOL[dtype], "per-head product")
    assert (out_wide[:, :, n:] == 0).all()
    # with a gate per head, read from a column range of a wider buffer
    wide = rnd((rows, heads + 6), 3, DT[dtype]).to(gpu)
    lat_ops.heads_product(x_wide[:, :, :k], w, out_wide[:, :, :n], gates=wide[:, 2:2 + heads])
    close(out_wide[:, :, :n], want * torch.sigmoid(wide[:, 2:2 + heads].double())[:, :, None], TOL[dtype], "gated")
    got = wide[:, 2:2 + heads].clone()
    K.head_gate(got_x := torch.ones((rows, heads * 4), dtype=DT[dtype], device=gpu), wide[:, 2:2 + heads], heads)
    close(got_x.view(rows, heads, 4)[:, :, 0], torch.sigmoid(got.double()), TOL[dtype], "the gate alone")


@pytest.mark.parametrize("per_range", [0, 32, 96])
@pytest.mark.parametrize("heads, rank, rot, window, keep_first", [
    (3, 64, 32, 0, 0), (16, 64, 64, 0, 0), (5, 128, 32, 36, 10), (20, 64, 32, 33, 0), (6, 128, 64, 16, 16)])
def test_latent_attention_on_the_matrix_cores(heads, rank, rot, window, keep_first, per_range, gpu):
    """Entries of a step - two portions of prompts cut in the middle of pages and of tiles, and
    decoded tokens, one right behind a page's edge - against the plain attention over all rows;
    the keys whole and in ranges.  Pages of other requests, and the rest of a request's last page,
    hold NaN."""
    page, scale, length = 16, 0.2, 200
    kd = rank + rot
    assert K.latent_attention_mfma_supported(rank, kd, page)
    q_all = rnd((length, heads, kd), 21, torch.bfloat16)
    rows_kv = rnd((length, kd), 22, torch.bfloat16)
    sinks = rnd((heads,), 23) * 2
    table, slots, pages = cache_for(length, page, 17)
    entries = [(37, 30), (199, 1), (0, 9), (112, 1), (96, 16)]        # (first position, tokens) of one request's copies
    lat = torch.full((pages, page, kd), float("nan"), dtype=torch.bfloat16, device=gpu)
    prob = plain.softmax_rows(torch.einsum("ihd,jd->hij", q_all.double(), rows_kv.double()) * scale,
                              plain.visible(length, window, keep_first), sinks.double())
    want_all = torch.einsum("hij,jd->ihd", prob, rows_kv.double()[:, :rank])
    for start, n in entries:
        # what the request holds when this entry runs: positions up to its last token
        upto = start + n
        lat.fill_(float("nan"))
        sl = slots[:upto].long().to(gpu)
        lat.view(-1, kd)[sl] = rows_kv[:upto].to(gpu)
        q = q_all[start:upto].contiguous().to(gpu)
        ranges = 1 if per_range == 0 else -(-upto // per_range)
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)
        for item in (16, 64):                   # rows of a work item: the kernel of decoded tokens, the one of portions
            tiles = (n * heads + item - 1) // item
            out = torch.empty((n, heads, rank), dtype=torch.bfloat16, device=gpu)
            K.latent_attention_mfma(q, out, lat, table.to(gpu), i32([0] * tiles), i32([item * t for t in range(tiles)]),
                                    i32([1]), i32([0, n]), i32([start]), scale, window, keep_first, sinks.to(gpu),
                                    ranges, per_range, item)
            assert torch.isfinite(out.float()).all(), f"entry {start}+{n}, items of {item}"
            close(out, want_all[start:upto], 3e-2, f"entry {start}+{n}, items of {item}")


@pytest.mark.parametrize("row_tiles", [1, 2])
@pytest.mark.parametrize("per_range", [0, 64])
@pytest.mark.parametrize("heads, kv_heads, dim, vdim, window, keep_first", [
    (4, 1, 64, 64, 44, 18), (8, 2, 32, 64, 33, 17), (6, 3, 64, 32, 0, 0), (32, 2, 64, 64, 16, 16), (2, 2, 128, 128, 50, 0)])
def test_windowed_attention_on_the_matrix_cores(heads, kv_heads, dim, vdim, window, keep_first, per_range, row_tiles, gpu):
    """The matrix-core kernel that takes a window with kept first positions, sinks and a value
    size of its own: portions of prompts and decoded tokens against the plain attention."""
    page, scale, length = 16, 0.2, 200
    assert K.attention_rows_mfma_supported(dim, vdim, page)
    group = heads // kv_heads
    q_all = rnd((length, heads, dim), 31, torch.bfloat16)
    k_all, v_all = rnd((length, kv_heads, dim), 32, torch.bfloat16), rnd((length, kv_heads, vdim), 33, torch.bfloat16)
    sinks = rnd((heads,), 34) * 2
    table, slots, pages = cache_for(length, page, 19)
    prob = plain.softmax_rows(torch.einsum("ihd,jhd->hij", q_all.double(), k_all.double().repeat_interleave(group, dim=1)) * scale,
                              plain.visible(length, window, keep_first), sinks.double())
    want_all = torch.einsum("hij,jhd->ihd", prob, v_all.double().repeat_interleave(group, dim=1))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=gpu)
    for start, n in [(37, 30), (199, 1), (0, 9), (112, 1), (96, 16)]:
        upto = start + n
        kp = torch.full((pages, kv_heads, page, dim), float("nan"), dtype=torch.bfloat16, device=gpu)
        v_cache = torch.full((pages, kv_heads, vdim, page), float("nan"), dtype=torch.bfloat16, device=gpu)
        sl = slots[:upto].long().to(gpu)
        kp[sl // page, :, sl % page] = k_all[:upto].to(gpu)
        v_cache[sl // page, :, :, sl % page] = v_all[:upto].to(gpu)
        k_cache = K.keys_to_pages(kp)
        q = q_all[start:upto].reshape(n, heads * dim).contiguous().to(gpu)
        per_item = 16 * row_tiles
        tiles = (n * group + per_item - 1) // per_item
        out = torch.empty((n, heads * vdim), dtype=torch.bfloat16, device=gpu)
        ranges = 1 if per_range == 0 else -(-upto // per_range)
        K.attention_rows_mfma(q, heads * dim, out, k_cache, v_cache, table.to(gpu), i32([0] * tiles),
                              i32([per_item * t for t in range(tiles)]), i32([1]), i32([0, n]), i32([start]), heads, kv_heads,
                              dim, scale, window, keep_first, sinks.to(gpu), vdim, ranges, per_range, row_tiles)
        assert torch.isfinite(out.float()).all(), f"entry {start}+{n}"
        close(out.view(n, heads, vdim), want_all[start:upto], 3e-2, f"entry {start}+{n}")


@pytest.mark.parametrize("x_dtype, out_dtype", [("float32", "float32"), ("float32", "bfloat16"), ("bfloat16", "bfloat16")])
@pytest.mark.parametrize("width, offset", [(8, 0), (2048, 0), (2056, 0), (4096, 0), (8192, 0), (8200, 0), (2048, 1)])
def test_layer_norm_rows_in_registers(width, offset, x_dtype, out_dtype, gpu):
    """Widths around what a thread holds once, twice and four times, and operands that do not start at 16 bytes."""
    def put(t):
        flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=gpu)
        return flat[offset:].view(t.shape).copy_(t)
    x, d1 = (rnd((5, width), 1, scale=3.0) + 1.5).to(DT[x_dtype]), rnd((5, width), 2, DT[out_dtype])
    d2, w1, w2 = rnd((5, width), 3), 1 + 0.1 * rnd((width,), 4), 1 + 0.1 * rnd((width,), 5)
    for rms in (False, True):
        for scale in (1.0, 0.7):
            xs, o1, o2 = put(x), put(torch.zeros((5, width), dtype=DT[out_dtype])), put(torch.zeros((5, width), dtype=DT[out_dtype]))
            K.layernorm(xs, put(w1), 1e-5, o1, deltas=(put(d1), put(d2)), weight2=put(w2), out2=o2, rms=rms, delta_scale=scale)
            total = x.double() + scale * (d1.double() + d2.double())
            close(xs, total, 1e-6 if x_dtype == "float32" else 5e-3, "the stream after the add")
            held = xs.double().cpu()
            centred = held if rms else held - held.mean(-1, keepdim=True)
            n = centred / torch.sqrt((centred ** 2).mean(-1, keepdim=True) + 1e-5)
            close(o1, n * w1.double(), TOL[out_dtype], "first copy")
            close(o2, n * w2.double(), TOL[out_dtype], "second copy")


@pytest.mark.parametrize("dim, rot", [(8, 0), (8, 8), (16, 16), (32, 16), (64, 32), (64, 64), (128, 96), (512, 512)])
@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("norm", [None, "unit", "weights", "weights first"])
@pytest.mark.parametrize("with_bias, offset", [(False, 0), (True, 0), (True, 1)])
def test_heads_of_a_power_of_two_in_registers(dim, rot, interleaved, norm, with_bias, offset, gpu):
    """Every form together with and without the others; a bias at an odd address takes the general kernel."""
    heads, kv_heads, vdim, T, page, eps = 5, 3, 24, 11, 8, 1e-2
    width = (heads + kv_heads) * dim + kv_heads * vdim
    qkv, bias = rnd((T, width), 7, torch.bfloat16), rnd((width,), 8, torch.bfloat16)
    wq, wk = 1 + 0.2 * rnd((dim,), 9), 1 + 0.2 * rnd((dim,), 10)
    table, slots, pages = cache_for(T, page, 3)
    slots[4] = -1
    angle = rnd((T, max(1, rot // 2)), 11, scale=2.0)
    cos, sin = (torch.cos(angle), torch.sin(angle)) if rot else (None, None)
    k_cache = torch.zeros((pages, *K.k_page_shape(kv_heads, dim)[:2], page, K.k_chunk(dim)), dtype=torch.bfloat16, device=gpu)
    v_cache = torch.zeros((pages, kv_heads, vdim, page), dtype=torch.bfloat16, device=gpu)
    buf = torch.zeros(width + offset, dtype=torch.bfloat16, device=gpu)
    buf[offset:] = bias.to(gpu)
    got, weighted = qkv.to(gpu), norm is not None and "weights" in norm
    K.qk_encode_cache(got, torch.arange(T, dtype=torch.int32, device=gpu), heads, kv_heads, dim, vdim, None if cos is None else cos.to(gpu),
                      None if sin is None else sin.to(gpu), interleaved, None if norm is None else eps, k_cache, v_cache, slots.to(gpu),
                      bias=buf[offset:] if with_bias else None, q_weight=wq.to(gpu) if weighted else None,
                      k_weight=wk.to(gpu) if weighted else None, norm_first=norm == "weights first")
    full = qkv.double() + (bias.double() if with_bias else 0.0)
    first = torch.arange(0, rot, 2) if interleaved else torch.arange(rot // 2)
    second = first + 1 if interleaved else first + rot // 2

    def encode(x, w):
        def unit(z):
            return z / torch.sqrt((z ** 2).mean(-1, keepdim=True) + eps) * (w.double() if weighted else 1.0)
        x = unit(x) if norm == "weights first" else x.clone()
        if rot:
            c, s, u, v = cos.double()[:, None], sin.double()[:, None], x[..., first].clone(), x[..., second].clone()
            x[..., first], x[..., second] = u * c - v * s, v * c + u * s
        return unit(x) if norm in ("unit", "weights") else x
    close(got[:, :heads * dim].view(T, heads, dim), encode(full[:, :heads * dim].view(T, heads, dim), wq), TOL["bfloat16"], "queries")
    written = slots >= 0
    sl = slots.long()[written]
    keys = K.pages_to_keys(k_cache).reshape(pages, kv_heads, page, dim)
    want = encode(full[:, heads * dim:(heads + kv_heads) * dim].view(T, kv_heads, dim), wk)[written]
    close(keys[sl // page, :, sl % page], want, TOL["bfloat16"], "cached keys")
    close(v_cache[sl // page, :, :, sl % page], full[:, (heads + kv_heads) * dim:].view(T, kv_heads, vdim)[written], 4e-3, "cached values")
