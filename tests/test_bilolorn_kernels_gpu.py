"""The kernels behind the Bilolorn parts, each alone against plain formulas: the step between branches with
norms on both sides, the query latent beside the cache write, per-head products with a gate per element and a
rotation in the same launch, experts by token id, the squared relu, the scaled embedding gather with its second
copy, and the mixer as a whole with one key that stands out."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import plain_bilolorn as plain
from kv_cache_optimization_for_llm_amd.engine.graphs import context_bucket
from kv_cache_optimization_for_llm_amd.ops import kernels as K
from kv_cache_optimization_for_llm_amd.ops import latent_attention as lat_ops
from kv_cache_optimization_for_llm_amd.parts.base import MixerContext, PendingNorm
from kv_cache_optimization_for_llm_amd.parts.mlp import PlainMLP
from kv_cache_optimization_for_llm_amd.parts.moe import RoutedExperts
from kv_cache_optimization_for_llm_amd.parts.norm import LayerNorm
from kv_cache_optimization_for_llm_amd.parts.rotary import RotaryEncoding
from kv_cache_optimization_for_llm_amd.parts.stream_ops import AddFirst

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
TOL = {"float32": 2e-5, "bfloat16": 2e-2}


def rnd(shape, seed, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def close(got, want, tol, what=""):
    got, want = got.double().cpu(), want.double().cpu()
    assert got.shape == want.shape
    err = (got - want).abs().max().item() / max(want.abs().max().item(), 1e-9)
    assert err <= tol, f"{what}: off by {err:.3g} of the largest value (limit {tol})"


# ---------------------------------------------------------------- the step between branches
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [30, 72, 1000, 1024, 1028, 2048, 2052, 4096, 5000, 8192, 9000])
def test_a_branch_output_enters_under_its_norm_and_the_row_is_normed_again(width, dtype, gpu):
    T = 5
    x, y, first = rnd((T, width), 1, scale=3.0) + 0.5, rnd((T, width), 2, DT[dtype], 2.0) - 0.75, rnd((T, width), 3)
    post = [(1 + 0.3 * rnd((width,), 4)).to(DT[dtype]), rnd((width,), 5, DT[dtype], 0.3)]
    pre = [(1 + 0.3 * rnd((width,), 6)).to(DT[dtype]), rnd((width,), 7, DT[dtype], 0.3)]

    def step(stream, y=None, addend=None, read=True, row_idx=None, bias=True, center=True):
        dev = stream.to(gpu)
        rows = T if row_idx is None else len(row_idx)
        out = torch.empty((rows, width), dtype=DT[dtype], device=gpu) if read else None
        K.sandwich_step(dev, y=None if y is None else y.to(gpu),
                        post=None if y is None else (post[0].to(gpu), post[1].to(gpu) if bias else None, 0.03, center),
                        addend=None if addend is None else addend.to(gpu),
                        pre=(pre[0].to(gpu), pre[1].to(gpu) if bias else None, 0.2, center) if read else None, out=out,
                        row_idx=None if row_idx is None else torch.tensor(row_idx, dtype=torch.int32, device=gpu))
        return dev, out

    def norm(v, w, b, eps, center=True):
        b = torch.zeros(width, dtype=torch.float64) if b is None else b.double()
        return plain.layer_norm(v, w.double(), b, eps) if center else plain.rms_norm(v, w.double(), eps) + b
    entered = x.double() + norm(y.double(), *post, 0.03)
    for addend in (None, first):
        total = entered + (0 if addend is None else addend.double())
        dev, out = step(x, y, addend)
        close(dev, total, 1e-6, "the stream stays 32-bit")
        close(out, norm(total, *pre, 0.2), TOL[dtype], "the read-out")
    dev, out = step(x)                                              # nothing pending: only read
    assert torch.equal(dev.cpu(), x)
    close(out, norm(x.double(), *pre, 0.2), TOL[dtype], "read-out alone")
    dev, _ = step(x, y, first, read=False)                          # only enter
    close(dev, entered + first.double(), 1e-6, "entering alone")
    dev, out = step(x, None, first)
    close(out, norm(x.double() + first.double(), *pre, 0.2), TOL[dtype], "the addend alone")
    dev, out = step(x, y, None, row_idx=[4, 0, 4])                  # gathered rows: nothing is written back
    assert torch.equal(dev.cpu(), x)
    close(out, norm(entered, *pre, 0.2)[[4, 0, 4]], TOL[dtype], "gathered rows")
    dev, out = step(x, y, None, bias=False, center=False)           # RMS norms without a bias
    total = x.double() + norm(y.double(), post[0], None, 0.03, False)
    close(dev, total, 1e-6, "RMS form, stream")
    close(out, norm(total, pre[0], None, 0.2, False), TOL[dtype], "RMS form, read-out")


def test_a_row_does_not_depend_on_the_other_rows_of_the_step(gpu):
    x, y = rnd((300, 256), 1).to(gpu), rnd((300, 256), 2, torch.bfloat16).to(gpu)
    w, b = (1 + rnd((256,), 3, scale=0.1)).bfloat16().to(gpu), rnd((256,), 4, torch.bfloat16).to(gpu)

    def run(lo, hi):
        s, out = x[lo:hi].clone(), torch.empty((hi - lo, 256), dtype=torch.bfloat16, device=gpu)
        K.sandwich_step(s, y=y[lo:hi].contiguous(), post=(w, b, 1e-5, True), pre=(b, w, 1e-5, True), out=out)
        return s, out
    for a, c in zip(run(0, 300), run(123, 124)):
        assert torch.equal(a[123:124], c)


def test_the_step_refuses_what_does_not_fit(gpu):
    x, w = torch.zeros((2, 8), device=gpu), torch.ones(8, device=gpu)
    with pytest.raises(K.KernelError):
        K.sandwich_step(x, post=(w, None, 0.0, True))               # a norm without an output
    with pytest.raises(K.KernelError):
        K.sandwich_step(x, y=torch.zeros((2, 4), device=gpu))
    with pytest.raises(K.KernelError):
        K.sandwich_step(x, pre=(w[:4].contiguous(), None, 0.0, True), out=x.clone())
    with pytest.raises(K.KernelError):
        K.sandwich_step(x.bfloat16(), pre=(w, None, 0.0, True), out=x.clone())
    with pytest.raises(K.KernelError):
        K.sandwich_step(x)


def test_the_embedding_output_is_added_with_or_behind_a_pending_output(gpu):
    op = AddFirst()
    h, y, first = rnd((4, 40), 1), rnd((4, 40), 2), rnd((4, 40), 3)
    norm = LayerNorm("n.", width=40, eps=1e-3, weight_name="w", bias_name="b")
    norm.load({"n.w": rnd((40,), 4).to(gpu), "n.b": rnd((40,), 5).to(gpu)})
    dev, delta = op.defer(h.to(gpu), PendingNorm(y.to(gpu), norm), first.to(gpu))
    assert torch.equal(dev.cpu(), h) and delta.norm is norm           # left to whoever reads the stream next
    out = norm.forward(dev, delta=delta)
    total = h.double() + plain.layer_norm(y.double(), norm.weight.cpu().double(), norm.bias.cpu().double(), 1e-3) + first.double()
    close(dev, total, 1e-6)
    close(out, plain.layer_norm(total, norm.weight.cpu().double(), norm.bias.cpu().double(), 1e-3), 1e-5)
    for pending in (None, y.to(gpu), (y.to(gpu), y.to(gpu))):         # other arrangements' outputs
        n = 0 if pending is None else (2 if isinstance(pending, tuple) else 1)
        dev, delta = op.defer(h.to(gpu), pending, first.to(gpu))
        assert delta is None
        close(dev, h.double() + n * y.double() + first.double(), 1e-6)


@pytest.mark.parametrize("table_dtype, out_dtype", [("bfloat16", "float32"), ("float32", "float32"), ("bfloat16", "bfloat16")])
def test_embedding_rows_times_a_constant_and_once_more(table_dtype, out_dtype, gpu):
    table = rnd((50, 24), 1, DT[table_dtype])
    ids = torch.tensor([3, 49, 0, -2, 3], dtype=torch.int32, device=gpu)
    feedback = torch.tensor([7, 11], dtype=torch.int32, device=gpu)
    out = torch.empty((5, 24), dtype=DT[out_dtype], device=gpu)
    copy = torch.empty_like(out)
    K.embed_gather(table.to(gpu), ids, out, feedback, 1.3, copy)
    close(out, table.double()[[3, 49, 0, 11, 3]] * 1.3, TOL[out_dtype] if out_dtype == "bfloat16" else 1e-6)
    assert torch.equal(out, copy)


# ---------------------------------------------------------------- latent attention
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("q_rank, rank, rot", [(24, 40, 8), (1, 16, 2), (300, 64, 32), (77, 129, 6)])
def test_query_latent_norm_beside_the_cache_write(q_rank, rank, rot, dtype, gpu):
    T, page, gates, eps = 19, 16, 13, 0.05
    y = rnd((T, q_rank + rank + rot + gates), 1, DT[dtype])
    qw, kw = (1 + rnd((q_rank,), 2, scale=0.3)).to(DT[dtype]), (1 + rnd((rank,), 3, scale=0.3)).to(DT[dtype])
    cos, sin = RotaryEncoding(head_dim=rot, max_positions=64, theta=90.0, frequencies="plain_f64", pairing="interleaved").tables(gpu)
    slots = torch.from_numpy(np.random.default_rng(1).permutation(48)[:T].astype(np.int32))
    cache = torch.zeros((3, page, rank + rot), dtype=DT[dtype], device=gpu)
    c_q = torch.empty((T, q_rank), dtype=DT[dtype], device=gpu)
    K.latent_encode_cache(y.to(gpu), q_rank, None, cache, kw.to(gpu), eps, cos, sin, torch.arange(T, dtype=torch.int32, device=gpu),
                          slots.to(gpu), 4, 12, rank, interleaved=True, c_q=c_q, q_norm_weight=qw.to(gpu))
    src = y.double()
    close(c_q, plain.rms_norm(src[:, :q_rank], qw.double(), eps), TOL[dtype], "query latent")
    got = cache.view(48, rank + rot)[slots.long().to(gpu)]
    c = plain.rms_norm(src[:, q_rank:q_rank + rank], kw.double(), eps)
    close(got[:, :rank], c, TOL[dtype], "latent")
    close(got[:, rank:], plain.rotate_pairs(src[:, q_rank + rank:q_rank + rank + rot], 90.0), TOL[dtype], "rotated part")
    # without a cache (a layer call that only reads) the query latent is still made
    again = torch.empty_like(c_q)
    K.latent_encode_cache(y.to(gpu), q_rank, None, None, kw.to(gpu), eps, cos, sin, torch.arange(T, dtype=torch.int32, device=gpu),
                          None, 4, 12, rank, interleaved=True, c_q=again, q_norm_weight=qw.to(gpu))
    assert torch.equal(again, c_q)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads, n, k", [(3, 20, 40), (1, 64, 32), (5, 48, 160), (20, 33, 64), (2, 200, 256), (4, 31, 320), (7, 4, 96)])
@pytest.mark.parametrize("rows", [1, 2, 17, 70, 300])
def test_per_head_products_with_a_gate_per_element(heads, n, k, rows, dtype, gpu):
    x, w = rnd((rows, heads, k), 1, DT[dtype]), rnd((heads, n, k), 2, DT[dtype], k ** -0.5)
    wide = rnd((rows, heads * n + 11), 3, DT[dtype], 2.0)           # the gates are columns of a wider buffer
    out = torch.empty((rows, heads * n), dtype=DT[dtype], device=gpu)
    gates = wide.to(gpu)[:, 11:]
    K.heads_matmul(x.to(gpu), w.to(gpu), out.view(rows, heads, n), gates.unflatten(1, (heads, n)))
    want = torch.einsum("thk,hnk->thn", x.double(), w.double()) * torch.sigmoid(wide[:, 11:].double()).view(rows, heads, n)
    close(out.view(rows, heads, n), want, TOL[dtype], "gate per element")
    K.heads_matmul(x.to(gpu), w.to(gpu), out.view(rows, heads, n), wide.to(gpu)[:, 3:3 + heads])
    want = torch.einsum("thk,hnk->thn", x.double(), w.double()) * torch.sigmoid(wide[:, 3:3 + heads].double())[:, :, None]
    close(out.view(rows, heads, n), want, TOL[dtype], "gate per head")


@pytest.mark.parametrize("heads, n, k, rot", [(36, 264, 96, 0), (36, 260, 32, 0), (40, 130, 64, 6), (130, 128, 160, 4)])
def test_per_head_products_of_many_rows_and_heads(heads, n, k, rot, gpu):
    """Enough work for the larger of the two tiles: rows and outputs that end inside one, outputs whose rows are
    not aligned for 16 bytes, a rotation in the same launch, and rows cut from a wider buffer."""
    rows = 517
    x, w = rnd((rows, heads, k + 8), 1, torch.bfloat16), rnd((heads, n, k), 2, torch.bfloat16, k ** -0.5)
    out = torch.full((rows + 1, heads, n + rot), float("nan"), dtype=torch.bfloat16, device=gpu)
    dev, turn = x.to(gpu), None
    if rot:
        cos, sin = RotaryEncoding(head_dim=rot, max_positions=600, theta=60.0, frequencies="plain_f64", pairing="interleaved").tables(gpu)
        turn = (dev[:, :, k:k + rot], out[:rows, :, n:], cos, sin, torch.arange(rows, dtype=torch.int32, device=gpu), True)
    lat_ops.heads_product(dev[:, :, :k], w.to(gpu), out[:rows, :, :n], rotate=turn)
    want = torch.matmul(x[..., :k].double().transpose(0, 1).contiguous(), w.double().transpose(1, 2).contiguous()).transpose(0, 1)
    close(out[:rows, :, :n], want, TOL["bfloat16"], "product")
    if rot:
        close(out[:rows, :, n:], plain.rotate_pairs(x[..., k:k + rot].double(), 60.0), TOL["bfloat16"], "rotation")
    assert out[rows].isnan().all()                                  # nothing behind the last row


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("interleaved", [True, False])
@pytest.mark.parametrize("rows, heads, plain_dim, rot, rank", [(1, 3, 12, 8, 40), (1, 1, 32, 2, 16), (37, 5, 64, 32, 96),
                                                               (300, 2, 32, 64, 128), (70, 17, 20, 6, 33), (2, 4, 128, 64, 256)])
def test_queries_are_rotated_in_the_expansions_launch(rows, heads, plain_dim, rot, rank, interleaved, dtype, gpu):
    q = rnd((rows, heads, plain_dim + rot), 1, DT[dtype])
    w = rnd((heads, rank, plain_dim), 2, DT[dtype], plain_dim ** -0.5)
    pos = torch.from_numpy(np.random.default_rng(2).integers(0, 500, rows).astype(np.int32))
    enc = RotaryEncoding(head_dim=rot, max_positions=512, theta=60.0, frequencies="plain_f64",
                         pairing="interleaved" if interleaved else "half")
    cos, sin = enc.tables(gpu)
    dev = q.to(gpu)
    q_lat = torch.full((rows, heads, rank + rot), float("nan"), dtype=DT[dtype], device=gpu)
    lat_ops.heads_product(dev[:, :, :plain_dim], w.to(gpu), q_lat[:, :, :rank],
                          rotate=(dev[:, :, plain_dim:], q_lat[:, :, rank:], cos, sin, pos.to(gpu), interleaved))
    close(q_lat[:, :, :rank], torch.einsum("thd,hrd->thr", q[..., :plain_dim].double(), w.double()), TOL[dtype], "expansion")
    table = torch.outer(pos.double(), torch.tensor([60.0 ** (-2 * i / rot) for i in range(rot // 2)], dtype=torch.float64))
    co, si = torch.cos(table)[:, None], torch.sin(table)[:, None]
    r = q[..., plain_dim:].double()
    u, v = (r[..., 0::2], r[..., 1::2]) if interleaved else (r[..., :rot // 2], r[..., rot // 2:])
    a, b = u * co - v * si, v * co + u * si
    want = torch.stack([a, b], -1).flatten(-2) if interleaved else torch.cat([a, b], -1)
    close(q_lat[:, :, rank:], want, TOL[dtype], "rotation")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads, rank, rot", [(5, 40, 8), (16, 64, 64), (33, 96, 32), (3, 192, 32), (8, 512, 64)])
def test_a_far_key_that_stands_out_and_a_sink_over_low_rank_rows(heads, rank, rot, dtype, gpu):
    """One query head and one cached row are scaled so that this key carries nearly all the weight: the very
    first key, keys on both sides of a page's border, and the query's own position - and a sink that outweighs
    every key.  Prompt rows and decoded rows; keys in one range and in many."""
    T, page, scale = 700, 16, 0.2
    key_dim = rank + rot
    pages = (T + page - 1) // page
    perm = torch.from_numpy(np.random.default_rng(3).permutation(pages + 2)[:pages].astype(np.int32))
    rows = rnd((T, key_dim), 1, DT[dtype])
    table = torch.full((2, pages + 1), -1, dtype=torch.int32)
    table[1, :pages] = perm
    fast = dtype == "bfloat16" and lat_ops.mfma_supported(rank, key_dim, page)
    sinks = torch.linspace(-2.0, 3.0, heads)
    sinks[heads - 1] = 60.0
    for key in (0, 15, 16, 335, 336, 699):
        r = rows.clone()
        r[key] = r[key] * 3
        cache = torch.zeros(((pages + 2) * page, key_dim), dtype=DT[dtype])
        pos = torch.arange(T)
        cache[perm.long()[pos // page] * page + pos % page] = r
        cache = cache.view(pages + 2, page, key_dim).to(gpu)
        for q_pos in ((699,), tuple(range(690, 700))):
            n = len(q_pos)
            q = rnd((n, heads, key_dim), 5, DT[dtype], 0.3)
            q[:, 0] = (r[key].float() * 4 / r[key].float().norm() ** 2 / scale * 3).to(DT[dtype])
            out = torch.full((n, heads, rank), float("nan"), dtype=DT[dtype], device=gpu)
            seat = torch.ones(n, dtype=torch.int32, device=gpu)
            p = torch.tensor(q_pos, dtype=torch.int32, device=gpu)
            s = torch.einsum("ihk,jk->hij", q.double(), r.double()) * scale
            s = s.masked_fill(torch.arange(T)[None, None, :] > torch.tensor(q_pos)[None, :, None], float("-inf"))
            full = torch.softmax(torch.cat([s, sinks.double()[:, None, None].expand(heads, n, 1)], -1), -1)
            want = torch.einsum("hij,jk->ihk", full[..., :-1], r.double()[:, :rank])
            assert full[0, -1, key] > 0.9 and full[heads - 1, -1, -1] > 0.99
            if not fast:
                K.latent_attention_rowwise(q.to(gpu), out, cache, table.to(gpu), seat, p, scale, 0, 0, sinks.to(gpu))
                close(out, want, TOL[dtype], f"key {key}")
                continue
            i32 = dict(dtype=torch.int32, device=gpu)
            for item_rows in (16, 64):
                items = (n * heads + item_rows - 1) // item_rows
                entry = torch.zeros(items, dtype=torch.int32, device=gpu)
                row0 = (item_rows * torch.arange(items)).to(torch.int32).to(gpu)
                for splits, per in ((1, 0), (2, 352), (6, 128), (22, 32)):
                    out.fill_(float("nan"))
                    K.latent_attention_mfma(q.to(gpu), out, cache, table.to(gpu), entry, row0, torch.tensor([1], **i32),
                                            torch.tensor([0, n], **i32), torch.tensor([q_pos[0]], **i32), scale, 0, 0, sinks.to(gpu),
                                            splits, per, item_rows)
                    close(out, want, TOL[dtype], f"key {key}, items of {item_rows} rows, {splits} ranges")


@pytest.mark.parametrize("heads, rank, rot, page", [(5, 64, 32, 16), (16, 128, 32, 32), (4, 512, 64, 16), (3, 96, 32, 48), (33, 192, 32, 16),
                                                    (8, 256, 64, 16), (6, 384, 64, 16), (7, 160, 32, 64)])
@pytest.mark.parametrize("window, keep_first", [(0, 0), (50, 0), (37, 5), (1, 3)])
def test_rows_of_several_entries_in_items_of_both_sizes(heads, rank, rot, page, window, keep_first, gpu):
    """Prompt portions and decoded tokens of several requests in one call, pages that hold garbage (NaN) behind
    every request's newest token and where a window has let pages go, keys in one range and in several."""
    key_dim, scale = rank + rot, 0.15
    starts, lens = [0, 75, 130, 9], [40, 1, 23, 2]
    seats, blocks = [2, 0, 3, 1], 12
    pool = sum((s + n + page - 1) // page for s, n in zip(starts, lens)) + 2
    perm = torch.from_numpy(np.random.default_rng(heads).permutation(pool).astype(np.int32))
    cache = torch.full((pool, page, key_dim), float("nan"), dtype=torch.bfloat16)
    table = torch.full((4, blocks), -1, dtype=torch.int32)
    rows, at = [], 0
    for s, n, seat in zip(starts, lens, seats):
        r = rnd((s + n, key_dim), 10 + s, torch.bfloat16)
        rows.append(r)
        need = (s + n + page - 1) // page
        for b in range(need):
            # a page that lies wholly behind the window of the entry's first token, and past the kept positions, is gone
            if window > 0 and (b + 1) * page <= s - window + 1 and b * page >= keep_first:
                continue
            table[seat, b] = perm[at + b]
            part = r[b * page:(b + 1) * page]
            cache[perm[at + b], :part.shape[0]] = part
        at += need
    q_start = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(q_start[-1])
    q = rnd((T, heads, key_dim), 3, torch.bfloat16, 0.4)
    sinks = torch.linspace(-1, 2, heads)
    want = torch.empty((T, heads, rank), dtype=torch.float64)
    for e, (s, n) in enumerate(zip(starts, lens)):
        k = rows[e].double()
        sc = torch.einsum("ihk,jk->hij", q[q_start[e]:q_start[e + 1]].double(), k) * scale
        i, j = torch.arange(s, s + n)[:, None], torch.arange(s + n)[None, :]
        seen = (j <= i) & ((i - j < window) | (j < keep_first) if window > 0 else torch.ones_like(j <= i))
        sc = sc.masked_fill(~seen[None], float("-inf"))
        p = torch.softmax(torch.cat([sc, sinks.double()[:, None, None].expand(heads, n, 1)], -1), -1)[..., :-1]
        want[q_start[e]:q_start[e + 1]] = torch.einsum("hij,jk->ihk", p, k[:, :rank])
    dev, i32 = cache.to(gpu), dict(dtype=torch.int32, device=gpu)

    def items(rows_per_item, entries):
        ent = [e for e in entries for _ in range(0, lens[e] * heads, rows_per_item)]
        row0 = [r for e in entries for r in range(0, lens[e] * heads, rows_per_item)]
        return torch.tensor(ent, **i32), torch.tensor(row0, **i32), rows_per_item
    few = [e for e in range(4) if lens[e] <= 2]
    many = [e for e in range(4) if e not in few]
    for first, more in ((items(16, range(4)), ()), (items(64, range(4)), ()), (items(64, many), (items(16, few),))):
        for splits, per in ((1, 0), (3, 64), (5, 32)):            # (the longest request has 153 keys)
            out = torch.full((T, heads, rank), float("nan"), dtype=torch.bfloat16, device=gpu)
            K.latent_attention_mfma(q.to(gpu), out, dev, table.to(gpu), first[0], first[1], torch.tensor(seats, **i32),
                                    torch.from_numpy(q_start).to(gpu), torch.tensor(starts, **i32), scale, window, keep_first,
                                    sinks.to(gpu), splits, per, first[2], more)
            close(out, want, 2e-2, f"items of {first[2]} rows, {splits} ranges of {per}")


# ---------------------------------------------------------------- feed-forwards
@pytest.mark.parametrize("interleaved, gate, sink", [(True, "element", True), (False, "head", False), (True, None, True)])
@pytest.mark.parametrize("heads, rank, page, entries", [(1, 32, 16, [(0, 1)]), (3, 96, 16, [(0, 63), (5, 64), (200, 65)]), (16, 512, 16, [(0, 300), (700, 129)]), (40, 32, 16, [(3, 900)]),
                                                        (3, 64, 16, [(5, 1200)]), (4, 96, 16, [(900, 300), (1021, 257), (0, 64)]), (6, 32, 16, [(1030, 256), (17, 1)]),
                                                        (4, 512, 48, [(31, 257), (0, 33), (96, 128), (1, 1)])])
def test_prompts_over_expanded_keys_and_values(heads, rank, page, entries, interleaved, gate, sink, gpu):
    """Entries (first position, tokens) whose tokens and contexts end inside, at and behind tiles of 64 tokens, blocks of 64 keys, their
    halves and tiles of 128 positions, on pages in no order, a context bound larger than any of them; 16 tokens a wavefront or (contexts
    above 1,024, at least 256 tokens, no more workgroups than the chip takes at once) 32."""
    d, rot, dv, T = 128, 64, 128, sum(n for _, n in entries)
    context = max(s + n for s, n in entries) + 37
    blocks = -(-context // page)
    g = torch.Generator().manual_seed(heads + rank)
    table = torch.randperm(len(entries) * blocks, generator=g).view(len(entries), blocks).to(torch.int32)
    seats = torch.randperm(len(entries), generator=g).to(torch.int32)
    cache = torch.full((len(entries) * blocks, page, rank + rot), float("nan"), dtype=torch.bfloat16)      # what nobody wrote
    rows = {}
    for e, (start, n) in enumerate(entries):
        rows[e] = rnd((start + n, rank + rot), 10 + e, torch.bfloat16)
        for p in range(start + n):
            cache[int(table[seats[e], p // page]), p % page] = rows[e][p]
    q = rnd((T, heads, d + rot), 1, torch.bfloat16)
    up_k, up_v = rnd((heads * d, rank), 2, torch.bfloat16, rank ** -0.5), rnd((heads * dv, rank), 3, torch.bfloat16, rank ** -0.5)
    position = RotaryEncoding(head_dim=rot, max_positions=2048, theta=10000.0, frequencies="plain_f64", pairing="interleaved" if interleaved else "half")
    cos, sin = position.tables(gpu)
    sinks = rnd((heads,), 4, scale=2.0) if sink else None
    gates = None if gate is None else rnd((T, heads, dv) if gate == "element" else (T, heads), 5, torch.bfloat16)
    first = torch.tensor(np.cumsum([0] + [n for _, n in entries]), dtype=torch.int32)
    out = torch.full((T, heads * dv), float("nan"), dtype=torch.bfloat16, device=gpu)
    w = K.moe_tiled_weight(torch.cat([up_k, up_v])[None].to(gpu))[0]
    K.latent_prompt(q.to(gpu), cache.to(gpu), w, out, table.to(gpu), seats.to(gpu), first.to(gpu),
                    torch.tensor([s for s, _ in entries], dtype=torch.int32, device=gpu), cos, sin, interleaved, 192 ** -0.5, context,
                    max(n for _, n in entries), None if sinks is None else sinks.to(gpu), None if gates is None else gates.to(gpu))
    c64, s64 = cos.double().cpu(), sin.double().cpu()
    for e, (start, n) in enumerate(entries):
        at, lat = slice(int(first[e]), int(first[e]) + n), rows[e].double()
        k = torch.cat([(lat[:, :rank] @ up_k.double().T).view(-1, heads, d), lat[:, None, rank:].expand(-1, heads, -1)], -1)
        v = (lat[:, :rank] @ up_v.double().T).view(-1, heads, dv)
        x, pos = q[at].double(), torch.arange(start, start + n)
        c, s = c64[pos][:, None], s64[pos][:, None]
        a, b = (x[..., d::2], x[..., d + 1::2]) if interleaved else (x[..., d:d + rot // 2], x[..., d + rot // 2:])
        turned = torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2) if interleaved else torch.cat([a * c - b * s, b * c + a * s], -1)
        x = torch.cat([x[..., :d], turned], -1)
        score = torch.einsum("thd,khd->htk", x, k) * 192 ** -0.5
        score = score.masked_fill(torch.arange(start + n)[None, None, :] > pos[None, :, None], float("-inf"))
        if sinks is not None:
            score = torch.cat([score, sinks.double()[:, None, None].expand(-1, n, 1)], -1)
        p = torch.softmax(score, -1)[..., :start + n]
        want = torch.einsum("htk,khd->thd", p, v)
        if gates is not None:
            z = torch.sigmoid(gates[at].double())
            want = want * (z if gate == "element" else z[..., None])
        got = out[at].double().cpu().view(n, heads, dv)
        # keys, values, rotated queries, probabilities and results are rounded to bf16 (2^-9 each, relative): their squares add up
        assert (got - want).norm() <= 2.0 ** -9 * 5 ** 0.5 * 1.5 * want.norm(), e


@pytest.mark.parametrize("heads, start, n", [(2, 0, 100), (2, 5, 100), (3, 39, 64), (40, 3, 900), (2, 0, 1100), (3, 1029, 260), (2, 1039, 300), (2, 1045, 256)])
def test_a_prompts_later_positions_leave_earlier_tokens_alone(heads, start, n, gpu):
    """Positions that are no numbers: tokens that, with the 16 that they go with, see none of the 32 keys beside theirs have the bits that
    they have without, with 16 tokens a wavefront and with 32."""
    d, rot, rank, page = 128, 64, 32, 16
    context, T = start + n + 9, n
    blocks = -(-context // page)
    q = rnd((T, heads, d + rot), 1, torch.bfloat16).to(gpu)
    up = K.moe_tiled_weight(torch.cat([rnd((heads * d, rank), 2, torch.bfloat16, rank ** -0.5), rnd((heads * d, rank), 3, torch.bfloat16, rank ** -0.5)])[None].to(gpu))[0]
    cos, sin = RotaryEncoding(head_dim=rot, max_positions=2048, theta=10000.0, frequencies="plain_f64", pairing="half").tables(gpu)
    rows = rnd((blocks * page, rank + rot), 4, torch.bfloat16)

    def run(cache):
        out = torch.empty((T, heads * d), dtype=torch.bfloat16, device=gpu)
        one = lambda *v: torch.tensor(v, dtype=torch.int32, device=gpu)
        return K.latent_prompt(q, cache.view(blocks, page, rank + rot).to(gpu), up, out, torch.arange(blocks, dtype=torch.int32, device=gpu)[None],
                               one(0), one(0, n), one(start), cos, sin, False, 192 ** -0.5, context, n).cpu()
    want = run(rows)
    assert want.isfinite().all()
    newest = start + torch.clamp(torch.arange(n) // 16 * 16 + 15, max=n - 1)       # of a token's 16
    for bad in sorted({start, start + n - 1, start + n // 2, start + 17, start + 33, max(start, min(64, start + n - 1))}):
        spoilt = rows.clone()
        spoilt[bad] = float("nan") if bad % 2 else float("inf")
        got = run(spoilt)
        apart = newest < bad // 32 * 32
        assert torch.equal(got[apart], want[apart]), bad
        assert not got[bad - start:].isfinite().any(dim=1).any(), bad


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows, width, ff", [(1, 64, 96), (3, 30, 25), (40, 128, 200), (300, 64, 512)])
def test_squared_relu_feed_forward(rows, width, ff, dtype, gpu):
    x = rnd((rows, width), 1, DT[dtype])
    w = {"p.up": rnd((ff, width), 2, DT[dtype], width ** -0.5), "p.down": rnd((width, ff), 3, DT[dtype], ff ** -0.5)}
    part = PlainMLP("p.", hidden_size=width, intermediate_size=ff, activation="relu2")
    part.load({k: v.to(gpu) for k, v in w.items()})
    want = plain.squared_relu_mlp(x.double(), {k: v.double() for k, v in w.items()}, "p.")
    close(part.forward(x.to(gpu), None), want, TOL[dtype])
    z = rnd((rows, ff), 4, DT[dtype])
    out = torch.empty_like(z, device=gpu)
    K.bias_act(z.to(gpu), out, "relu2")
    close(out, torch.clamp(z.double(), min=0) ** 2, 1e-6 if dtype == "float32" else 5e-3)
    bias = rnd((ff,), 5)
    K.bias_act(z.to(gpu), out, "relu2", bias.to(gpu))
    close(out, torch.clamp(z.double() + bias.double(), min=0) ** 2, 1e-6 if dtype == "float32" else 5e-3)


def test_squared_relu_as_a_gate_and_in_a_products_epilogue(gpu):
    from kv_cache_optimization_for_llm_amd.parts.linear import Linear
    for rows in (1, 8, 100):
        x, w = rnd((rows, 64), 1, torch.bfloat16), rnd((192, 64), 2, torch.bfloat16, 0.2)
        gu = x.double() @ w.double().T
        want = torch.clamp(gu[:, :96], min=0) ** 2 * gu[:, 96:]
        out = torch.empty((rows, 96), dtype=torch.bfloat16, device=gpu)
        K.act_mul(gu.bfloat16().to(gpu), out, "relu2")
        close(out, want, 2e-2)
        lin = Linear(w.to(gpu), halves=2)
        if lin.fused_kernel(rows, torch.bfloat16) is not None:
            lin.gated(x.to(gpu), out, "relu2")
            close(out, want, 2e-2, "epilogue")


@pytest.mark.parametrize("group", [1, 4, 8])
@pytest.mark.parametrize("rows, experts, top", [(1, 1, 1), (5, 3, 2), (40, 24, 5), (900, 7, 7), (700, 300, 3), (2049, 16, 4), (6000, 5, 3)])
def test_experts_by_token_id_and_their_sorted_tiles(rows, experts, top, group, gpu):
    vocab = 97
    g = torch.Generator().manual_seed(rows)
    table = torch.rand((vocab, experts), generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
    ids = torch.randint(0, vocab, (rows,), generator=g).to(torch.int32)
    feedback = torch.tensor([5, 96], dtype=torch.int32)
    real = ids.clone().long()
    if rows > 2:
        ids[1], ids[2], real[1], real[2] = -1, -2, 5, 96              # ids that are still on the device
    idx = torch.full((rows, top), -9, dtype=torch.int32, device=gpu)
    wgt = torch.empty((rows, top), dtype=torch.float32, device=gpu)
    tiles = K.moe_tiles(rows * top, experts, group)
    slot = torch.empty(tiles * K.MOE_TILE, dtype=torch.int32, device=gpu)
    tile_expert = torch.empty(tiles, dtype=torch.int32, device=gpu)
    K.moe_table_align(table.to(gpu), ids.to(gpu), idx, wgt, experts, slot, tile_expert, feedback.to(gpu), group)
    assert torch.equal(idx.cpu(), table[real])
    assert torch.allclose(wgt.cpu(), torch.full((rows, top), 1.0 / top))
    slot, tile_expert = slot.cpu().view(tiles, K.MOE_TILE), tile_expert.cpu()
    used = slot[slot >= 0]
    assert sorted(used.tolist()) == list(range(rows * top))           # every slot once
    flat = idx.cpu().view(-1)
    for t in range(tiles):
        for s in slot[t][slot[t] >= 0].tolist():
            assert flat[s] == tile_expert[t]
    assert ((tile_expert >= 0) == (slot >= 0).any(-1)).all()
    groups = tile_expert.view(-1, group)                              # a group belongs to one expert, from its first tile on
    assert ((groups == groups[:, :1]) | (groups < 0)).all()
    # the same list from choices that are there already
    again, again_expert = torch.empty_like(slot, device=gpu).view(-1), torch.empty_like(tile_expert, device=gpu)
    K.moe_align(idx, experts, again, again_expert, group)
    assert torch.equal(again_expert.cpu(), tile_expert)
    for t in range(tiles):
        assert sorted(again.cpu().view(tiles, -1)[t].tolist()) == sorted(slot[t].tolist()) or tile_expert[t] >= 0


@pytest.mark.parametrize("group", [1, 4, 8])
@pytest.mark.parametrize("rows, width, ff, experts, top, gated", [(7, 64, 96, 5, 2, True), (300, 64, 96, 5, 2, True), (90, 96, 160, 3, 3, False), (700, 128, 36, 9, 4, True),
                                                                  (513, 32, 64, 2, 1, True), (1500, 288, 200, 8, 3, False)])
def test_experts_products_in_tiles_and_in_groups_of_tiles(rows, width, ff, experts, top, gated, group, gpu):
    """Both products alone: outputs that are no multiples of the kernel's 128, inner sizes of one step of 32
    and of odd numbers of them, experts without a token, runs that end inside a group."""
    g = torch.Generator().manual_seed(rows)
    idx = torch.rand((rows, experts), generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
    if experts > 4:
        idx[idx == 3] = experts                                       # (an expert nobody chose; those slots name none)
    x = rnd((rows, width), 1, torch.bfloat16)
    up = rnd((experts, (2 if gated else 1) * ff, width), 2, torch.bfloat16, width ** -0.5)
    ff_pad = (ff + 31) // 32 * 32
    down = torch.zeros((experts, width, ff_pad), dtype=torch.bfloat16)
    down[:, :, :ff] = rnd((experts, width, ff), 3, torch.bfloat16, ff ** -0.5)
    wgt = torch.rand((rows, top), generator=g)
    tiles = K.moe_tiles(rows * top, experts, group)
    slot = torch.empty(tiles * K.MOE_TILE, dtype=torch.int32, device=gpu)
    tile_expert = torch.empty(tiles, dtype=torch.int32, device=gpu)
    K.moe_align(idx.to(gpu), experts, slot, tile_expert, group)
    flat, xd = idx.view(-1).long(), x.double().repeat_interleave(top, 0)
    want_act, want = torch.zeros(rows * top, ff, dtype=torch.float64), torch.zeros(rows * top, width, dtype=torch.float64)
    for e in range(experts):
        m = flat == e
        z = xd[m] @ up[e].double().T
        h = torch.nn.functional.silu(z[:, 0::2]) * z[:, 1::2] if gated else torch.clamp(z, min=0) ** 2
        want_act[m] = h
        want[m] = h @ down[e, :, :ff].double().T * wgt.view(-1)[m].double()[:, None]
    sl = slot.cpu().long()
    used = sl >= 0
    # the matrices row by row, and - where outputs come in whole tiles - in operand order
    for tiled in (False, True)[:2 if up.shape[1] % 16 == 0 else 1]:
        lay = K.moe_tiled_weight if tiled else (lambda w: w)
        act = torch.full((tiles * K.MOE_TILE, ff), float("nan"), dtype=torch.bfloat16, device=gpu)
        K.moe_expert_rows(x.to(gpu), lay(up.to(gpu)), act, slot, tile_expert, top, activation="silu" if gated else "relu2", gated=gated,
                          group=group, tiled=tiled)
        wide = torch.zeros((tiles * K.MOE_TILE, ff_pad), dtype=torch.bfloat16, device=gpu)
        wide[:, :ff] = act
        out = torch.zeros((rows * top, width), dtype=torch.float32, device=gpu)
        K.moe_expert_rows(wide, lay(down.to(gpu)), out, slot, tile_expert, top, slot_weight=wgt.to(gpu), group=group, tiled=tiled)
        close(act.cpu()[used], want_act[sl[used]], 2e-2, "first product")
        close(out, want, 3e-2, "second product")


@pytest.mark.parametrize("rows, width, ff, experts, top, gated", [(7, 96, 36, 5, 2, True), (700, 128, 132, 9, 4, True), (513, 256, 256, 2, 1, False),
                                                                  (1500, 544, 264, 8, 3, False)])
def test_experts_products_are_the_same_against_128_and_256_outputs_a_workgroup(rows, width, ff, experts, top, gated, gpu, monkeypatch):
    """Bit for bit: an output's products are added up in the same order.  Outputs below, at and behind multiples of 128 and 256."""
    g = torch.Generator().manual_seed(rows)
    idx = torch.rand((rows, experts), generator=g).argsort(-1)[:, :top].to(torch.int32).contiguous()
    x, ff_pad = rnd((rows, width), 1, torch.bfloat16), (ff + 31) // 32 * 32
    up = rnd((experts, (2 if gated else 1) * ff, width), 2, torch.bfloat16, width ** -0.5)
    down = rnd((experts, width, ff_pad), 3, torch.bfloat16, ff ** -0.5)
    wgt = torch.rand((rows, top), generator=g).to(gpu)
    tiles = K.moe_tiles(rows * top, experts, 8)
    slot = torch.empty(tiles * K.MOE_TILE, dtype=torch.int32, device=gpu)
    tile_expert = torch.empty(tiles, dtype=torch.int32, device=gpu)
    K.moe_align(idx.to(gpu), experts, slot, tile_expert, 8)
    hidden = rnd((tiles * K.MOE_TILE, ff_pad), 4, torch.bfloat16).to(gpu)
    for tiled in (False, True)[:2 if up.shape[1] % 16 == 0 else 1]:
        lay = K.moe_tiled_weight if tiled else (lambda w: w)
        got = []
        for wide in (False, True):
            monkeypatch.setattr(K, "moe_wide", lambda *sizes: wide)
            act = torch.zeros((tiles * K.MOE_TILE, ff), dtype=torch.bfloat16, device=gpu)
            K.moe_expert_rows(x.to(gpu), lay(up.to(gpu)), act, slot, tile_expert, top, activation="silu" if gated else "relu2", gated=gated,
                              group=8, tiled=tiled)
            out = torch.full((rows * top, width), float("nan"), dtype=torch.float32, device=gpu)
            K.moe_expert_rows(hidden, lay(down.to(gpu)), out, slot, tile_expert, top, slot_weight=wgt, group=8, tiled=tiled)
            got.append((act[slot >= 0].cpu(), out.cpu()))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]) and got[0][0].any() and got[0][1].isfinite().all()


@pytest.mark.parametrize("x_at, w_at", [(1, 0), (0, 1), (4, 2)])
@pytest.mark.parametrize("group", [4, 8])
def test_products_of_many_rows_take_operands_at_any_address(group, x_at, w_at, gpu):
    """Experts' products and products per head whose operands start at no multiple of 16 bytes go through registers, not straight to
    LDS: the same numbers but for the order of the sums, the results rounded to bf16 (2^-9 of a result, each)."""
    def at(t, offset):
        flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=gpu)
        flat[offset:].copy_(t.reshape(-1))
        return flat[offset:].view(t.shape)
    rows, width, ff, experts, top = 700, 96, 136, 3, 2
    x, up = rnd((rows, width), 1, torch.bfloat16).to(gpu), rnd((experts, ff, width), 2, torch.bfloat16, width ** -0.5).to(gpu)
    idx = torch.rand((rows, experts), generator=torch.Generator().manual_seed(group)).argsort(-1)[:, :top].to(torch.int32).contiguous()
    tiles = K.moe_tiles(rows * top, experts, group)
    slot = torch.empty(tiles * K.MOE_TILE, dtype=torch.int32, device=gpu)
    tile_expert = torch.empty(tiles, dtype=torch.int32, device=gpu)
    K.moe_align(idx.to(gpu), experts, slot, tile_expert, group)
    got = []
    for dx, dw in ((0, 0), (x_at, w_at)):
        act = torch.zeros((tiles * K.MOE_TILE, ff), dtype=torch.bfloat16, device=gpu)
        K.moe_expert_rows(at(x, dx), at(up, dw), act, slot, tile_expert, top, activation="relu2", group=group)
        heads = torch.zeros((rows, 3, ff), dtype=torch.bfloat16, device=gpu)
        K.heads_matmul(at(x, dx).view(rows, 3, 32), at(rnd((3, ff, 32), 3, torch.bfloat16, 0.2), dw), heads)
        got.append((act.double().cpu(), heads.double().cpu()))
    for a, b in zip(*got):
        assert a.any() and (a - b).norm() <= 2.0 ** -8 * a.norm()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows, width, ff, experts, top, shared", [(1, 64, 32, 6, 2, 48), (33, 40, 20, 3, 1, 0), (300, 128, 96, 9, 4, 64)])
def test_table_experts_with_and_without_the_expert_every_token_uses(rows, width, ff, experts, top, shared, dtype, gpu):
    part = RoutedExperts("p.", hidden_size=width, intermediate_size=ff, experts=experts, top=top, activation="silu", gated=True,
                         correction=False, router="table", table_rows=53, shared_intermediate=shared)
    from kv_cache_optimization_for_llm_amd.weights.random_init import random_state_dict
    state = random_state_dict(part.tensor_specs(), 4, DT[dtype], 1.0)
    part.load({k: v.to(gpu) for k, v in state.items()})
    x = rnd((rows, width), 1, DT[dtype])
    ids = torch.randint(0, 53, (rows,), generator=torch.Generator().manual_seed(1)).to(torch.int32)

    class Batch:
        token_ids, feedback = ids.to(gpu), None
    got = part.forward(x.to(gpu), MixerContext(batch=Batch()))
    w = {k: (v.double() if v.is_floating_point() else v) for k, v in state.items()}
    mlp = {"router": {"top": top}, **({"shared": {"ff": shared}} if shared else {})}
    close(got, plain.table_experts(x.double(), ids, w, "p.", mlp), TOL[dtype])


def test_which_steps_expand_keys_and_values(gpu):
    def step(shortest, context, entries=1):
        return SimpleNamespace(min_q_len=shortest, max_context=context, num_entries=entries)
    rule = lambda batch, heads=16, rot=64, rank=512, window=0, dtype=torch.bfloat16: \
        lat_ops.expands(batch, heads, 128, rot, 128, rank, window, dtype)
    assert rule(step(64, 1024)) and rule(step(64, 64), heads=1024)
    assert not rule(step(63, 63)) and not rule(step(64, 1025)) and not rule(step(64, 64), heads=1025)
    assert not rule(step(2048, 2048, 64)) and not rule(step(64, 64), window=32) and not rule(step(64, 64), dtype=torch.float32)
    assert not rule(step(64, 64), rot=32) and not rule(step(64, 64), rank=48)
    # a captured step's contexts are rounded up: what it was captured for and every step it stands for take the same path
    for shortest, context in ((100, 1500), (100, 1601), (64, 1), (256, 4096), (300, 4097), (1024, 8191), (4096, 40000)):
        assert rule(step(shortest, context)) == rule(step(shortest, context_bucket(context)))
