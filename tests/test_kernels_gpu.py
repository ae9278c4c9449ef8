"""Each HIP kernel alone against a plain PyTorch fp32 reference, at sizes other than the engine's."""
import math

import numpy as np
import pytest
import torch

import plain_llama as plain
from kv_cache_optimization_for_llm_amd.ops import kernels as K
from kv_cache_optimization_for_llm_amd.ops.attention import choose_splits

pytestmark = pytest.mark.gpu
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def rnd(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


def close(got, want, dtype, what, tol32=2e-6, tol16=1e-2):
    got, want = got.float().cpu(), want.float().cpu()
    tol = tol32 if dtype == torch.float32 else tol16
    err = (got - want).abs().max().item() / max(want.abs().max().item(), 1e-6)
    assert err <= tol, f"{what}: relative error {err:.3g} > {tol}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("table_dtype", ["float32", "bfloat16"])
def test_embed_gather(dtype, table_dtype, gpu):
    table = rnd(77, 50, dtype=DT[table_dtype])
    ids = torch.tensor([3, 76, 0, 3, 41], dtype=torch.int32)
    out = torch.empty(5, 50, dtype=DT[dtype], device=gpu)
    K.embed_gather(table.to(gpu), ids.to(gpu), out)
    want = table.float()[ids.long()].to(DT[dtype])
    assert torch.equal(out.cpu(), want)


def test_logits_without_a_finite_value_are_reported_and_lookups_stay_inside_the_table(gpu):
    """A row of logits that are all NaN or all -inf names no token.  The sampler says so with -1,
    greedy and sampled rows alike (the host ends the request with an error), and a lookup of
    whatever a kernel left in the feedback buffer stays inside the table: the token of such a row
    is looked up on the device by the next step, which may be queued before the host has seen
    the -1, and a row past the table's end is a memory fault, not an error message."""
    vocab = 333
    lg = torch.randn(5, vocab)
    lg[0] = float("nan")
    lg[1] = float("-inf")
    lg[3] = float("nan")
    lg[4, 7:] = float("nan")                               # some finite logits: a token can be named
    lg = lg.to(gpu)
    out = torch.full((5,), -7, dtype=torch.int32, device=gpu)
    K.sample(lg, out, chunks=4)
    assert out.cpu().tolist() == [-1, -1, int(lg[2].argmax()), -1, int(lg[4, :7].argmax())]
    inv_t = torch.tensor([1.0, 1.25, 0.0, 2.0, 1.0], device=gpu)
    zeros = torch.zeros(5, dtype=torch.int32, device=gpu)
    host = torch.full((5,), -7, dtype=torch.int32).pin_memory()
    K.sample(lg, out, chunks=4, inv_temperature=inv_t, seed=5, rng_key=zeros, rng_step=zeros, host_tokens=host)
    torch.cuda.synchronize()
    got = out.cpu().tolist()
    assert got[:4] == [-1, -1, int(lg[2].argmax()), -1] and 0 <= got[4] < 7 and host.tolist() == got
    # more chunks than the vocabulary fills (the last ones are empty): the same answers
    K.sample(lg, out, chunks=128, inv_temperature=inv_t, seed=5, rng_key=zeros, rng_step=zeros)
    assert out.cpu().tolist()[:4] == got[:4]
    table = rnd(vocab, 64, dtype=torch.bfloat16)
    feedback = torch.tensor([vocab, -9, 1 << 30, 5], dtype=torch.int32)
    ids = torch.tensor([-1, -2, -3, -4], dtype=torch.int32)
    emb = torch.empty(4, 64, dtype=torch.bfloat16, device=gpu)
    K.embed_gather(table.to(gpu), ids.to(gpu), emb, feedback.to(gpu))
    assert torch.equal(emb.cpu(), table[[vocab - 1, 0, vocab - 1, 5]])
    hidden, scaled = torch.empty_like(emb), torch.empty_like(emb)
    sumsq = torch.empty((4, 1), device=gpu)
    K.embed_gather_prep(table.to(gpu), ids.to(gpu), hidden, scaled, sumsq, torch.ones(64).to(gpu), feedback.to(gpu))
    assert torch.equal(hidden.cpu(), table[[vocab - 1, 0, vocab - 1, 5]])


@pytest.mark.parametrize("width", [8, 520, 2048, 4104])
@pytest.mark.parametrize("weight_dtype", ["float32", "bfloat16"])
def test_embed_gather_that_prepares_the_first_norm(width, weight_dtype, gpu):
    """hidden = table[ids] (ids from the feedback buffer too), scaled = round(hidden * w), the sum of
    squares per row; finished, it is the norm of the gathered rows."""
    table = rnd(91, width, dtype=torch.bfloat16)
    w = (1 + 0.1 * rnd(width, seed=2)).to(DT[weight_dtype])
    ids = torch.tensor([3, -1, 90, 0, -2, 3], dtype=torch.int32)
    feedback = torch.tensor([55, 7], dtype=torch.int32)
    real = torch.tensor([3, 55, 90, 0, 7, 3])
    hidden = torch.full((6, width), float("nan"), dtype=torch.bfloat16, device=gpu)
    scaled, sumsq = torch.empty_like(hidden), torch.full((6, 1), float("nan"), device=gpu)
    K.embed_gather_prep(table.to(gpu), ids.to(gpu), hidden, scaled, sumsq, w.to(gpu), feedback.to(gpu))
    want = table[real]
    assert torch.equal(hidden.cpu(), want)
    assert torch.equal(scaled.cpu(), (want.float() * w.float()).to(torch.bfloat16))
    assert torch.allclose(sumsq.cpu()[:, 0], (want.float() ** 2).sum(-1), rtol=1e-5)
    eps = 2e-6
    fin = torch.empty_like(hidden)
    K.normed_rows_finish(scaled, sumsq, width, eps, fin)
    close(fin, plain.rms_norm(want.float(), w.float(), eps), torch.bfloat16, "gather + norm", tol16=1.2e-2)
    with pytest.raises(K.KernelError):
        K.embed_gather_prep(table.float().to(gpu), ids.to(gpu), hidden, scaled, sumsq, w.to(gpu), feedback.to(gpu))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [50, 64, 520, 1000, 2048, 2050, 4096, 4104])
def test_rmsnorm_plain_fused_and_gathered(dtype, width, gpu):
    dt = DT[dtype]
    x, d, w = rnd(9, width, dtype=dt), rnd(9, width, dtype=dt, seed=1), (1 + 0.1 * rnd(width, seed=2)).to(dt)
    eps = 3e-6
    out = torch.empty(9, width, dtype=dt, device=gpu)
    K.rmsnorm(x.to(gpu), w.to(gpu), eps, out)
    close(out, plain.rms_norm(x.float(), w.float(), eps), dt, "rmsnorm", tol16=5e-3)
    # fused residual add: hidden becomes round(x + d), the norm is of that
    h = x.clone().to(gpu)
    K.rmsnorm(h, w.to(gpu), eps, out, delta=d.to(gpu))
    s = (x.float() + d.float()).to(dt)
    assert torch.equal(h.cpu(), s)
    close(out, plain.rms_norm(s.float(), w.float(), eps), dt, "add+rmsnorm", tol16=5e-3)
    # gathered rows (a row may be named twice), with and without the add; hidden is untouched
    rows = torch.tensor([8, 2, 2], dtype=torch.int32)
    h = x.clone().to(gpu)
    o3 = torch.empty(3, width, dtype=dt, device=gpu)
    K.rmsnorm(h, w.to(gpu), eps, o3, delta=d.to(gpu), row_idx=rows.to(gpu))
    assert torch.equal(h.cpu(), x)
    close(o3, plain.rms_norm(s.float()[rows.long()], w.float(), eps), dt, "gather+add+rmsnorm", tol16=5e-3)
    # a weight stored in 32-bit is used in 32-bit
    K.rmsnorm(x.to(gpu), w.float().to(gpu), eps, out)
    close(out, plain.rms_norm(x.float(), w.float(), eps), dt, "rmsnorm fp32 weight", tol16=5e-3)
    # many rows (a prompt portion): the same three forms
    R = 515
    X, D = rnd(R, width, dtype=dt, seed=5), rnd(R, width, dtype=dt, seed=6)
    O = torch.full((R, width), float("nan"), dtype=dt, device=gpu)
    H = X.clone().to(gpu)
    K.rmsnorm(H, w.to(gpu), eps, O)
    close(O, plain.rms_norm(X.float(), w.float(), eps), dt, "rmsnorm, many rows", tol16=5e-3)
    assert torch.equal(H.cpu(), X)
    K.rmsnorm(H, w.to(gpu), eps, O, delta=D.to(gpu))
    S = (X.float() + D.float()).to(dt)
    assert torch.equal(H.cpu(), S)
    close(O, plain.rms_norm(S.float(), w.float(), eps), dt, "add+rmsnorm, many rows", tol16=5e-3)
    idx = torch.arange(R - 1, -1, -1, dtype=torch.int32)
    idx[7] = idx[8]
    H = X.clone().to(gpu)
    K.rmsnorm(H, w.float().to(gpu), eps, O, delta=D.to(gpu), row_idx=idx.to(gpu))
    assert torch.equal(H.cpu(), X)
    close(O, plain.rms_norm(S.float()[idx.long()], w.float(), eps), dt, "gather+add+rmsnorm, many rows", tol16=5e-3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_silu_mul_residual_and_cast(dtype, gpu):
    dt = DT[dtype]
    gu = rnd(7, 2 * 250, dtype=dt, scale=3.0)
    out = torch.empty(7, 250, dtype=dt, device=gpu)
    K.silu_mul(gu.to(gpu), out)
    g, u = gu.float()[:, :250], gu.float()[:, 250:]
    close(out, g * (1 / (1 + torch.exp(-g))) * u, dt, "silu_mul", tol16=5e-3)
    h, d = rnd(5, 33, dtype=dt), rnd(5, 33, dtype=dt, seed=4)
    hg = h.clone().to(gpu)
    K.residual_add(hg, d.to(gpu))
    assert torch.equal(hg.cpu(), (h.float() + d.float()).to(dt))
    x = rnd(1000, dtype=torch.float32)
    b = torch.empty(1000, dtype=torch.bfloat16, device=gpu)
    K.cast(x.to(gpu), b)
    assert torch.equal(b.cpu(), x.to(torch.bfloat16))          # round to nearest even, as torch does
    f = torch.empty(1000, dtype=torch.float32, device=gpu)
    K.cast(b, f)
    assert torch.equal(f.cpu(), x.to(torch.bfloat16).float())


@pytest.mark.parametrize("m, n, k", [(1, 7, 5), (33, 130, 70), (64, 64, 64), (100, 389, 120), (3, 16, 2050)])
def test_gemm_f32_is_true_fp32_and_row_independent(m, n, k, gpu):
    a, w = rnd(m, k), rnd(n, k, seed=1)
    out = torch.empty(m, n, device=gpu)
    K.gemm_nt_f32(a.to(gpu), w.to(gpu), out)
    want = (a.double() @ w.double().t()).float()
    assert (out.cpu() - want).abs().max() <= 2e-6 * k ** 0.5 * max(1.0, want.abs().max().item())
    # a row's result does not depend on the other rows in the batch (bitwise)
    one = torch.empty(1, n, device=gpu)
    K.gemm_nt_f32(a[m - 1:m].to(gpu), w.to(gpu), one)
    assert torch.equal(one[0], out[m - 1])


@pytest.mark.parametrize("k", [1, 15, 64, 100, 1040, 2048, 2050, 5000])
@pytest.mark.parametrize("n", [16, 130, 4161])
def test_gemm_f32_rows_are_the_same_bits_in_every_kernel(n, k, gpu):
    """One row alone, 16, 17, 32 rows (the few-rows kernel), 33, 64, 65 and 600 rows (both tiles): the same bits."""
    a, w = rnd(600, k).to(gpu), rnd(n, k, seed=1).to(gpu)
    rows = {}
    for m in (1, 16, 17, 32, 33, 64, 65, 600):
        rows[m] = K.gemm_nt_f32(a[:m], w, torch.full((m, n), float("nan"), device=gpu))
    for m, got in rows.items():
        assert torch.equal(got, rows[600][:m]), m
    last = K.gemm_nt_f32(a[599:], w, torch.empty(1, n, device=gpu))
    assert torch.equal(last[0], rows[600][599])
    want = a.double() @ w.double().t()
    # K products and additions of relative error 2^-24 each, by their root: rms errors add up in squares
    assert (rows[600] - want).double().pow(2).mean().sqrt() <= 2.0 ** -24 * max(4.0, (2.0 * k) ** 0.5) * (a.double().pow(2) @ w.double().pow(2).t()).sqrt().mean()
    # a view whose rows do not start at multiples of 16 bytes
    flat = torch.zeros(65 * k + 1, device=gpu)
    flat[1:] = a[:65].reshape(-1)
    odd = K.gemm_nt_f32(flat[1:].view(65, k), w, torch.empty(65, n, device=gpu))
    assert torch.equal(odd, rows[65])


@pytest.mark.parametrize("n, k", [(7167, 40), (7168, 32), (14335, 48), (14336, 31), (20000, 96)])
def test_gemm_f32_rows_are_the_same_bits_where_the_kernel_changes(n, k, gpu):
    """16, 17, 32, 33, 64 and 65 rows of about as many outputs as send few rows to the tiles; sums of one to three parts."""
    a, w = rnd(65, k).to(gpu), rnd(n, k, seed=1).to(gpu)
    got = {m: K.gemm_nt_f32(a[:m], w, torch.full((m, n), float("nan"), device=gpu)) for m in (1, 16, 17, 32, 33, 64, 65)}
    for m, rows in got.items():
        assert torch.equal(rows, got[65][:m]), m
    close(got[65], a.double() @ w.double().t(), torch.float32, "gemm_nt_f32")


@pytest.mark.parametrize("m, n", [(20, 16), (66, 70)])
def test_gemm_f32_rows_of_more_than_8_mib(m, n, gpu):
    """Rows that a tile's 32-bit offsets do not reach: in parts of 16 bytes or one by one, alone or among others, the same bits."""
    k = (1 << 21) + 4
    g = torch.Generator(device=gpu).manual_seed(m)
    flat = torch.empty(m * k + 1, device=gpu)
    a, w = torch.randn((m, k), generator=g, device=gpu), torch.randn((n, k), generator=g, device=gpu)
    flat[1:].view(m, k).copy_(a)
    got = K.gemm_nt_f32(a, w, torch.empty(m, n, device=gpu))
    assert torch.equal(K.gemm_nt_f32(flat[1:].view(m, k), w, torch.empty(m, n, device=gpu)), got)
    assert torch.equal(K.gemm_nt_f32(a[-1:], w, torch.empty(1, n, device=gpu))[0], got[-1])
    want = sum(a[:, i:i + 65536].double() @ w[:, i:i + 65536].double().t() for i in range(0, k, 65536))
    # as above: K products and additions of relative error 2^-24 each, by their root
    assert (got - want).pow(2).mean().sqrt() <= 2.0 ** -24 * (2.0 * k) ** 0.5 * k ** 0.5


@pytest.mark.parametrize("m, n, k", [(48, 3072, 1024), (49, 3072, 1024), (33, 3072, 1020), (20, 8192, 6144), (21, 8192, 6144), (20, 8196, 6144), (40, 4096, 6144),
                                     (41, 4096, 6144), (40, 4100, 6144)])
def test_gemm_f32_either_side_of_where_few_rows_end(m, n, k, gpu):
    """By outputs, rows and K: the bits of a row alone, whichever kernel the rows go to."""
    a, w = rnd(m, k).to(gpu), rnd(n, k, seed=1).to(gpu)
    got = K.gemm_nt_f32(a, w, torch.full((m, n), 7.0, device=gpu))
    for row in (0, m // 2, m - 1):
        assert torch.equal(K.gemm_nt_f32(a[row:row + 1].contiguous(), w, torch.empty(1, n, device=gpu))[0], got[row]), row


@pytest.mark.parametrize("m, n", [(65, 68), (100, 3000), (130, 4500), (190, 10000), (517, 2048), (402, 3072), (517, 3072), (250, 16384), (129, 8196)])
@pytest.mark.parametrize("k", [4, 36, 96, 2052])
def test_gemm_f32_every_height_of_a_tile(m, n, k, gpu):
    """Tiles of 16 to 128 rows, remainders of rows, outputs and columns: the bits of a row alone, and nothing of a neighbouring row (whose
    first elements lie behind a row's last ones)."""
    a, w = rnd(m, k).to(gpu), rnd(n, k, seed=1).to(gpu)
    a[m // 2 + 1], w[n // 3 + 1] = float("nan"), float("inf")
    got = K.gemm_nt_f32(a, w, torch.full((m, n), 7.0, device=gpu))
    for row in (0, m // 2, m - 1):
        one = K.gemm_nt_f32(a[row:row + 1].contiguous(), w, torch.empty(1, n, device=gpu))
        assert torch.equal(one[0].nan_to_num(nan=5.0), got[row].nan_to_num(nan=5.0)), row
    rows, outputs = [i for i in range(m) if i != m // 2 + 1], [i for i in range(n) if i != n // 3 + 1]
    want = a[rows].double() @ w[outputs].double().t()
    # as above: K products and additions of relative error 2^-24 each
    bound = 2.0 ** -24 * max(4.0, (2.0 * k) ** 0.5) * (a[rows].double().pow(2) @ w[outputs].double().pow(2).t()).sqrt().mean()
    assert (got[rows][:, outputs] - want).double().pow(2).mean().sqrt() <= bound
    assert got[m // 2 + 1, outputs].isnan().all()


def rope_reference(x, pos, inv, heads, d, rot):
    cos, sin = plain.rope_cos_sin(pos, inv)
    x = x.view(len(pos), heads, d).clone()
    x[..., :rot] = plain.apply_rope(x[..., :rot], cos, sin)
    return x


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("nq, nkv, d, rot, page", [(4, 2, 16, 16, 16), (6, 1, 24, 24, 8), (3, 3, 48, 32, 4)])
def test_rope_and_cache_write(dtype, nq, nkv, d, rot, page, gpu):
    dt = DT[dtype]
    T, pages = 11, 20
    qkv = rnd(T, (nq + 2 * nkv) * d, dtype=dt)
    pos = [0, 1, 2, 50, 51, 7, 300, 8, 9, 10, 11]
    slots = torch.tensor([5, 17, 3, -1, 40, 41, 42, 8, 9, 70, 71], dtype=torch.int32) % (pages * page)
    slots[3] = -1
    inv = plain.rope_inv_freq(rot, 20000.0, dict(rope_type="llama3", factor=4.0, low_freq_factor=1.0,
                                                 high_freq_factor=2.0, original_max_position_embeddings=64))
    cos, sin = plain.rope_cos_sin(range(400), inv)
    k_cache = K.keys_to_pages(torch.zeros(pages, nkv, page, d, dtype=dt, device=gpu))
    v_cache = torch.zeros(pages, nkv, d, page, dtype=dt, device=gpu)
    x = qkv.clone().to(gpu)
    K.rope_kv_write(x, torch.tensor(pos, dtype=torch.int32, device=gpu), nq, nkv, d,
                    torch.from_numpy(cos).to(gpu), torch.from_numpy(sin).to(gpu), k_cache, v_cache,
                    slots.to(gpu), page)
    f = qkv.float()
    q_want = rope_reference(f[:, :nq * d], pos, inv, nq, d, rot)
    k_want = rope_reference(f[:, nq * d:(nq + nkv) * d], pos, inv, nkv, d, rot)
    v_want = f[:, (nq + nkv) * d:].view(T, nkv, d)
    close(x[:, :nq * d].view(T, nq, d), q_want, dt, "rope q", tol16=5e-3)
    assert torch.equal(x[:, nq * d:].cpu(), qkv[:, nq * d:])       # K and V columns are not touched
    kc, vc = K.pages_to_keys(k_cache).float().cpu(), v_cache.float().cpu()
    for t in range(T):
        s = int(slots[t])
        if s < 0:
            continue
        close(kc[s // page, :, s % page, :], k_want[t], dt, f"cached k of token {t}", tol16=5e-3)
        assert torch.equal(vc[s // page, :, :, s % page], v_want[t].to(dt).float())
    written = {int(s) for s in slots if s >= 0}
    for s in range(pages * page):
        if s not in written:
            assert kc[s // page, :, s % page, :].abs().max() == 0 and vc[s // page, :, :, s % page].abs().max() == 0


def attention_case(dtype, nq, nkv, d, page, window, entries, seed, gpu, stale=0.0):
    """entries: [(start_pos, q_len)].  Builds a cache with random pages, runs both kernels.
    ``stale``: what every position holds that no entry has written (the rest of a request's last
    page, pages nobody owns)."""
    dt = DT[dtype]
    g = torch.Generator().manual_seed(seed)
    E = len(entries)
    max_blocks = max((s + n + page - 1) // page for s, n in entries) + 1
    n_pages = E * max_blocks + 3
    perm = torch.randperm(n_pages, generator=g)
    table = torch.full((E + 2, max_blocks), -1, dtype=torch.int32)
    seats = [E + 1 - i for i in range(E)]                    # seats differ from entry numbers
    kc = torch.full((n_pages, nkv, page, d), stale)
    vc = torch.full((n_pages, nkv, d, page), stale)
    if stale != 0.0:
        vc[..., 1::2] = float("inf")        # NaN and infinities side by side
        kc[:, :, 1::2, :] = float("-inf")
    keys, vals, qs = [], [], []
    used = 0
    for e, (s, n) in enumerate(entries):
        ctx = s + n
        k, v = torch.randn(ctx, nkv, d, generator=g), torch.randn(ctx, nkv, d, generator=g)
        k, v = k.to(dt).float(), v.to(dt).float()
        nb = (ctx + page - 1) // page
        table[seats[e], :nb] = perm[used:used + nb].to(torch.int32)
        used += nb
        for p in range(ctx):
            pg = int(table[seats[e], p // page])
            kc[pg, :, p % page, :] = k[p]
            vc[pg, :, :, p % page] = v[p]
        keys.append(k)
        vals.append(v)
        qs.append((torch.randn(n, nq, d, generator=g) * 1.5).to(dt).float())
    scale = 1.0 / math.sqrt(d)
    want = []
    for e, (s, n) in enumerate(entries):
        full_q = torch.zeros(s + n, nq, d)
        full_q[s:] = qs[e]
        want.append(plain.causal_gqa_attention(full_q, keys[e], vals[e], scale, window)[s:])
    want = torch.cat(want).reshape(-1, nq * d)
    T = want.shape[0]
    stride = (nq + 2 * nkv) * d
    qkv = torch.zeros(T, stride)
    qkv[:, :nq * d] = torch.cat(qs).reshape(T, nq * d)
    lens = [n for _, n in entries]
    q_start = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    tok_seat = np.repeat(np.asarray(seats, dtype=np.int32), lens)
    tok_pos = np.concatenate([np.arange(s, s + n, dtype=np.int32) for s, n in entries])
    dev = dict(qkv=qkv.to(dt).to(gpu), kc=K.keys_to_pages(kc.to(dt)).to(gpu), vc=vc.to(dt).to(gpu), table=table.to(gpu),
               tok_seat=torch.from_numpy(tok_seat).to(gpu), tok_pos=torch.from_numpy(tok_pos).to(gpu),
               entry_seat=torch.tensor(seats, dtype=torch.int32, device=gpu),
               q_start=torch.from_numpy(q_start).to(gpu),
               start_pos=torch.tensor([s for s, _ in entries], dtype=torch.int32, device=gpu))
    return dev, want, T, stride, scale, lens


ENTRIES = [(0, 1), (0, 37), (63, 1), (64, 2), (100, 29), (255, 1), (17, 70)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("nq, nkv, d, page, window", [(4, 2, 16, 16, 0), (6, 1, 24, 8, 0), (3, 3, 48, 4, 0),
                                                      (8, 2, 64, 16, 45), (5, 5, 128, 32, 0)])
def test_attention_rowwise(dtype, nq, nkv, d, page, window, gpu):
    dev, want, T, stride, scale, _ = attention_case(dtype, nq, nkv, d, page, window, ENTRIES, 7, gpu)
    out = torch.empty(T, nq * d, dtype=DT[dtype], device=gpu)
    K.attention_rowwise(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], dev["tok_seat"],
                        dev["tok_pos"], nq, nkv, d, scale, window)
    close(out, want, DT[dtype], "attention_rowwise", tol32=3e-6, tol16=8e-3)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("page", [16, 6])               # (pages of 6: keys of a page are not read by fours)
@pytest.mark.parametrize("nq, nkv, d", [(32, 4, 32), (36, 12, 16), (20, 10, 20), (28, 4, 64)])
def test_attention_rowwise_is_the_same_bits_however_many_heads_go_together(dtype, page, nq, nkv, d, gpu):
    """The launches lie on every side of the rule's lines (3,072 / 6,144 / 12,288 rows of a head)."""
    dev, want, T, stride, scale, _ = attention_case(dtype, nq, nkv, d, page, 0, ENTRIES, 7, gpu)
    outs = []
    for rows in (0, 3072, 6144, 12288):
        times = max(1, -(-rows // (T * nq)))
        out = torch.full((T * times, nq * d), float("nan"), dtype=DT[dtype], device=gpu)
        q, seat, pos = dev["qkv"].repeat(times, 1), dev["tok_seat"].repeat(times), dev["tok_pos"].repeat(times)
        for a in range(0, T * times, T * times if rows else 16):
            some = slice(a, a + (T * times if rows else 16))
            K.attention_rowwise(q[some], stride, out[some], dev["kc"], dev["vc"], dev["table"], seat[some], pos[some], nq, nkv, d,
                                scale, 0)
        outs += [o.cpu() for o in out.split(T)]
    close(outs[0], want, DT[dtype], "attention_rowwise", tol32=3e-6, tol16=8e-3)
    assert all(torch.equal(o, outs[0]) for o in outs[1:])


def items_for(lens, group, gpu, row_tiles=1):
    ent, row0 = [], []
    for e, n in enumerate(lens):
        for r in range(0, n * group, 16 * row_tiles):
            ent.append(e)
            row0.append(r)
    return (torch.tensor(ent, dtype=torch.int32, device=gpu), torch.tensor(row0, dtype=torch.int32, device=gpu))


def chunked_oracle(chunk, entries, *case):
    """Chunks of so many positions: the window oracle row by row."""
    whole = [attention_case("bfloat16", *case, w, entries, 11, "cpu")[1] for w in range(1, chunk + 1)]
    pos = np.concatenate([np.arange(s, s + n) for s, n in entries])
    return torch.stack([whole[p % chunk][t] for t, p in enumerate(pos)])


@pytest.mark.parametrize("tiles", [1, 2])
@pytest.mark.parametrize("window", [9, -40])
def test_keys_that_begin_in_the_second_tile_of_a_block(window, tiles, gpu):
    """The tile in front of them is read from their first page: stale places behind the last key there stay out."""
    entries = [(17, 270), (255, 33), (1000, 17), (276, 5), (283, 1)]
    dev, want, T, stride, scale, lens = attention_case("bfloat16", 8, 2, 64, 16, max(window, 0), entries, 11, gpu, stale=float("nan"))
    if window < 0:
        want = chunked_oracle(-window, entries, 8, 2, 64, 16)
    ent, row0 = items_for(lens, 4, gpu, tiles)
    out = torch.full((T, 8 * 64), float("nan"), dtype=torch.bfloat16, device=gpu)
    K.attention_mfma(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], ent, row0, dev["entry_seat"], dev["q_start"],
                     dev["start_pos"], 8, 2, 64, scale, window, 1, 0, tiles)
    close(out, want, torch.bfloat16, f"attention_mfma tiles={tiles}", tol16=8e-3)


@pytest.mark.parametrize("waves", [2, 4])
@pytest.mark.parametrize("nq, nkv, d, page, window", [
    (4, 2, 16, 16, 0), (3, 3, 32, 4, 0), (8, 2, 64, 16, 45), (32, 8, 64, 16, 0), (32, 8, 64, 16, -40), (5, 1, 80, 8, 0),
    (24, 8, 128, 16, 0), (24, 8, 128, 16, 33), (6, 2, 96, 32, 0), (14, 2, 112, 16, 0)])
def test_prompt_items_in_equal_shares(nq, nkv, d, page, window, waves, gpu):
    """Entries from one key (three shares without a key) to several blocks a share; stale places hold NaN and infinities."""
    entries = [(0, 1), (0, 37), (63, 1), (100, 29), (255, 33), (17, 270), (1000, 17)]
    dev, want, T, stride, scale, lens = attention_case("bfloat16", nq, nkv, d, page, max(window, 0), entries, 11, gpu, stale=float("nan"))
    if window < 0:
        want = chunked_oracle(-window, entries, nq, nkv, d, page)
    ent, row0 = items_for(lens, nq // nkv, gpu, 2)
    out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    K.attention_mfma(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], ent, row0, dev["entry_seat"], dev["q_start"],
                     dev["start_pos"], nq, nkv, d, scale, window, waves, 0, 2, False, waves=waves)
    close(out, want, torch.bfloat16, f"attention_mfma waves={waves}", tol16=8e-3)
    with pytest.raises(K.KernelError):          # (equal shares are for the wavefronts of one workgroup)
        K.attention_mfma(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], ent, row0, dev["entry_seat"], dev["q_start"],
                         dev["start_pos"], nq, nkv, d, scale, window, 2 * waves, 0, 2, False, waves=waves)


@pytest.mark.parametrize("nq, nkv, d, page, window", [
    (4, 2, 16, 16, 0), (6, 2, 48, 8, 0), (3, 3, 32, 4, 0), (8, 2, 64, 16, 45), (32, 8, 64, 16, 0),
    (5, 1, 80, 16, 0), (24, 8, 128, 16, 0), (4, 4, 96, 32, 33), (2, 1, 256, 16, 0), (14, 2, 112, 16, 0)])
@pytest.mark.parametrize("splits, wide, pair", [(1, False, False), (3, False, False), (1, True, False),
                                                (2, True, False), (1, True, True), (2, False, True)])
def test_attention_mfma(nq, nkv, d, page, window, splits, wide, pair, gpu):
    assert K.attention_mfma_supported(d, page)
    dev, want, T, stride, scale, lens = attention_case("bfloat16", nq, nkv, d, page, window, ENTRIES, 11, gpu)
    tiles = K.attention_mfma_row_tiles(d, wide)
    assert tiles == (1 if not wide or d > 128 else 2)
    ent, row0 = items_for(lens, nq // nkv, gpu, tiles)
    out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    per = 0
    if splits > 1:
        per = (max(s + n for s, n in ENTRIES) + splits - 1) // splits
        per = (per + 31) // 32 * 32
    K.attention_mfma(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], ent, row0,
                     dev["entry_seat"], dev["q_start"], dev["start_pos"], nq, nkv, d, scale, window,
                     splits, per, tiles, pair)
    close(out, want, torch.bfloat16, f"attention_mfma splits={splits} tiles={tiles} pair={pair}", tol16=8e-3)
    # the same with one record per item instead of the lookups through the entry: bitwise equal
    e = ent.cpu().long()
    qs, sp, seat = dev["q_start"].cpu(), dev["start_pos"].cpu(), dev["entry_seat"].cpu()
    meta = torch.zeros((e.shape[0], 8), dtype=torch.int32)
    meta[:, 0], meta[:, 1], meta[:, 2], meta[:, 3], meta[:, 4] = qs[e], qs[e + 1] - qs[e], sp[e], seat[e], row0.cpu()
    out2 = torch.full_like(out, float("nan"))
    K.attention_mfma(dev["qkv"], stride, out2, dev["kc"], dev["vc"], dev["table"], ent, row0,
                     dev["entry_seat"], dev["q_start"], dev["start_pos"], nq, nkv, d, scale, window,
                     splits, per, tiles, pair, meta.to(gpu))
    assert torch.equal(out2, out)
    # keys and values loaded through the caches instead of past them: the same bits
    out4 = torch.full_like(out, float("nan"))
    K.attention_mfma(dev["qkv"], stride, out4, dev["kc"], dev["vc"], dev["table"], ent, row0,
                     dev["entry_seat"], dev["q_start"], dev["start_pos"], nq, nkv, d, scale, window,
                     splits, per, tiles, pair, keep_cached=True)
    assert torch.equal(out4, out)
    # a launch over some of the entries only (the others belong to another launch of the same
    # step): their rows are right, every other row keeps what it held, split merge included
    keep = (ent.cpu() % 2 == 0)
    sub = keep.nonzero().flatten().to(gpu)
    out3 = torch.full_like(out, 7.0)
    K.attention_mfma(dev["qkv"], stride, out3, dev["kc"], dev["vc"], dev["table"], ent[sub], row0[sub],
                     dev["entry_seat"], dev["q_start"], dev["start_pos"], nq, nkv, d, scale, window,
                     splits, per, tiles, False, meta.to(gpu)[sub] if pair else None, covers_all_rows=False)
    for e in range(len(lens)):
        rows = slice(int(qs[e]), int(qs[e + 1]))
        if e % 2 == 0:
            assert torch.equal(out3[rows], out[rows])
        else:
            assert (out3[rows] == 7.0).all()


@pytest.mark.parametrize("nq, nkv, d, page, window", [(4, 2, 16, 16, 0), (32, 8, 64, 16, 0), (8, 2, 64, 16, 45),
                                                      (6, 2, 48, 8, 0), (4, 4, 96, 32, 33), (24, 8, 128, 16, 0)])
def test_attention_never_sees_what_a_page_held_before(nq, nkv, d, page, window, gpu):
    """A page handed to a request still holds its previous owner's keys and values behind the
    request's newest token, and pages it does not own hold anything at all: here NaN and
    infinities.  Those positions have probability zero, and zero times a non-finite value must not
    reach the output (the matrix-core kernels multiply whole 32-key blocks, masked keys included)."""
    dev, want, T, stride, scale, lens = attention_case("bfloat16", nq, nkv, d, page, window, ENTRIES, 13, gpu,
                                                       stale=float("nan"))
    assert not torch.isfinite(dev["kc"].float()).all() and not torch.isfinite(dev["vc"].float()).all()
    out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    K.attention_rowwise(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], dev["tok_seat"],
                        dev["tok_pos"], nq, nkv, d, scale, window)
    close(out, want, torch.bfloat16, "attention_rowwise over stale pages", tol16=8e-3)
    for splits, wide, pair in ((1, False, False), (3, False, False), (1, True, True), (2, True, False)):
        tiles = K.attention_mfma_row_tiles(d, wide)
        ent, row0 = items_for(lens, nq // nkv, gpu, tiles)
        per = ((max(s + n for s, n in ENTRIES) + splits - 1) // splits + 31) // 32 * 32 if splits > 1 else 0
        out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
        K.attention_mfma(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], ent, row0,
                         dev["entry_seat"], dev["q_start"], dev["start_pos"], nq, nkv, d, scale, window,
                         splits, per, tiles, pair)
        assert torch.isfinite(out.float()).all(), f"splits={splits} tiles={tiles}: a stale value reached the output"
        close(out, want, torch.bfloat16, f"attention_mfma over stale pages splits={splits} tiles={tiles}", tol16=8e-3)
    if K.attention_lds_supported(d, page):
        dev, want, T, stride, scale, lens = attention_case("bfloat16", nq, nkv, d, page, window, LONG_ENTRIES, 17, gpu,
                                                           stale=float("nan"))
        group = nq // nkv
        qs, sp, seat = dev["q_start"].cpu(), dev["start_pos"].cpu(), dev["entry_seat"].cpu()
        rows = [(int(qs[e]), n, int(sp[e]), int(seat[e]), r0, 0, 0, 0)
                for e, n in enumerate(lens) for r0 in range(0, n * group, 128)]
        meta = torch.tensor(rows, dtype=torch.int32, device=gpu)
        for splits in (1, 3):
            per = ((max(s + n for s, n in LONG_ENTRIES) + splits - 1) // splits + 31) // 32 * 32 if splits > 1 else 0
            out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
            K.attention_lds(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], meta, nq, nkv, d, scale,
                            window, False, splits, per)
            assert torch.isfinite(out.float()).all(), f"workgroup kernel, splits={splits}: a stale value reached the output"
            close(out, want, torch.bfloat16, f"attention_lds over stale pages splits={splits}", tol16=8e-3)


@pytest.mark.parametrize("nq, nkv, d, window", [(32, 8, 64, 0), (24, 8, 128, 0), (8, 2, 64, 45), (16, 1, 64, 0), (4, 4, 128, 0)])
@pytest.mark.parametrize("splits, waves", [(1, 1), (3, 1), (8, 1), (2, 2), (4, 4), (8, 4), (8, 2), (12, 4)])
@pytest.mark.parametrize("rotate", [True, False])
def test_decode_attention_that_rotates_and_caches_inside(nq, nkv, d, window, splits, waves, rotate, gpu):
    """Decoded tokens straight from the joined projection: the attention kernel rotates Q and the
    new K, caches K and V and attends.  Same output and same cache contents as the rotation kernel
    followed by the attention kernel; positions at every place of a page and of a 32-key block,
    position 0 included; a token without a cache slot is attended to but not stored; without a
    slot mapping (a layer call that only reads another's cache) nothing is stored and the key
    comes from the cache.  With ``waves`` > 1 so many key ranges go to the wavefronts of one
    workgroup, which adds their results up itself (all of them: no merge launch), in both kernels."""
    assert K.attention_mfma_rope_supported(d, 16, nq // nkv) and not K.attention_mfma_rope_supported(48, 16, 2)
    assert not K.attention_mfma_rope_supported(64, 8, 2) and not K.attention_mfma_rope_supported(64, 16, 32)
    page = 16
    positions = [0, 1, 15, 16, 17, 31, 32, 33, 47, 63, 64, 100, 255, 256, 300, 511, 5]
    T = len(positions)
    g = torch.Generator().manual_seed(d + nq + splits)
    max_blocks = max(positions) // page + 2
    n_pages = T * max_blocks + 3
    perm = torch.randperm(n_pages, generator=g).to(torch.int32)
    table = perm[:T * max_blocks].view(T, max_blocks).contiguous()
    kc = (torch.randn(n_pages, nkv, page, d, generator=g)).to(torch.bfloat16)
    vc = (torch.randn(n_pages, nkv, d, page, generator=g)).to(torch.bfloat16)
    qkv = (torch.randn(T, (nq + 2 * nkv) * d, generator=g) * 1.5).to(torch.bfloat16)
    pos_t = torch.tensor(positions, dtype=torch.int32)
    slots = torch.tensor([int(table[t, p // page]) * page + p % page for t, p in enumerate(positions)], dtype=torch.int32)
    inv = plain.rope_inv_freq(d, 500000.0, None)
    cos, sin = (torch.from_numpy(a).to(gpu) for a in plain.rope_cos_sin(range(600), inv))
    if not rotate:
        cos = sin = None
    meta = torch.zeros((T, 8), dtype=torch.int32)
    meta[:, 0], meta[:, 1], meta[:, 2], meta[:, 3] = torch.arange(T), 1, pos_t, torch.arange(T)
    order = torch.argsort(-pos_t.long(), stable=True)                 # most keys first, as the engine orders items
    meta = meta[order].contiguous().to(gpu)
    scale = 1.0 / math.sqrt(d)
    per = ((max(positions) + 1 + splits - 1) // splits + 31) // 32 * 32 if splits > 1 else 0
    ent = order.to(torch.int32).to(gpu)
    zeros = torch.zeros(T, dtype=torch.int32, device=gpu)
    seat = torch.arange(T, dtype=torch.int32, device=gpu)
    qs = torch.arange(T + 1, dtype=torch.int32, device=gpu)

    def separate(slot_map, waves=1):
        k, v, x = K.keys_to_pages(kc).to(gpu), vc.clone().to(gpu), qkv.clone().to(gpu)
        K.rope_kv_write(x, pos_t.to(gpu), nq, nkv, d, cos, sin, k, v, slot_map.to(gpu), page)
        out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
        K.attention_mfma(x, x.shape[1], out, k, v, table.to(gpu), ent, zeros, seat, qs, pos_t.to(gpu), nq, nkv, d,
                         scale, window, splits, per, 1, False, meta, waves=waves)
        return out, k, v

    def fused(slot_map, k=None, v=None):
        k = K.keys_to_pages(kc).to(gpu) if k is None else k
        v = vc.clone().to(gpu) if v is None else v
        out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
        K.attention_mfma_rope(qkv.to(gpu), out, k, v, table.to(gpu), meta, nq, nkv, d, scale, cos, sin,
                              None if slot_map is None else slot_map.to(gpu), window, splits, per, waves=waves)
        return out, k, v

    want, k_want, v_want = separate(slots)
    if waves > 1:
        shared, _, _ = separate(slots, waves)
        assert torch.isfinite(shared.float()).all()
        close(shared, want, torch.bfloat16, f"{waves} wavefronts of a workgroup on one item", tol16=4e-3)
        with pytest.raises(K.KernelError):
            separate(slots, 3)
    got, k_got, v_got = fused(slots)
    assert torch.equal(k_got, k_want) and torch.equal(v_got, v_want), "the cache holds other keys or values"
    assert torch.isfinite(got.float()).all()
    close(got, want, torch.bfloat16, "rotation and cache write inside the attention kernel", tol16=4e-3)
    assert (got.float() - want.float()).abs().max() <= 2 ** -6 * want.float().abs().max()
    # a token without a slot: attended to (from registers), not stored
    some = slots.clone()
    some[3] = some[11] = -1
    got2, k2, v2 = fused(some)
    assert torch.equal(got2, got)
    kw, vw = K.pages_to_keys(k_want).clone(), v_want.clone()
    for t in (3, 11):
        pg, off = int(slots[t]) // page, int(slots[t]) % page
        kw[pg, :, off, :] = kc[pg, :, off, :].to(gpu)
        vw[pg, :, :, off] = vc[pg, :, :, off].to(gpu)
    assert torch.equal(K.pages_to_keys(k2), kw) and torch.equal(v2, vw)
    # no slot mapping: the cache (which already holds the tokens' keys) is only read
    got3, k3, v3 = fused(None, k_want.clone(), v_want.clone())
    assert torch.equal(k3, k_want) and torch.equal(v3, v_want)
    close(got3, want, torch.bfloat16, "rotation inside, keys from the cache", tol16=4e-3)


LONG_ENTRIES = [(0, 300), (40, 1), (200, 131), (5, 64), (0, 33)]


@pytest.mark.parametrize("nq, nkv, d, window", [(4, 2, 32, 0), (32, 8, 64, 0), (8, 2, 64, 70), (6, 2, 96, 0),
                                                (24, 8, 128, 0), (5, 1, 64, 0), (3, 3, 128, 150)])
@pytest.mark.parametrize("pair, splits", [(False, 1), (True, 1), (False, 3), (True, 2), (False, 11)])
def test_attention_with_keys_shared_through_lds(nq, nkv, d, window, pair, splits, gpu):
    """The workgroup kernel for prompt portions (128 query rows share each key block): long and
    short entries, entries that start deep in their request, groups that do not divide 128,
    windows, and work items taken in pairs."""
    assert K.attention_lds_supported(d, 16) and not K.attention_lds_supported(d, 8)
    assert not K.attention_lds_supported(48, 16)
    dev, want, T, stride, scale, lens = attention_case("bfloat16", nq, nkv, d, 16, window, LONG_ENTRIES, 3, gpu)
    group = nq // nkv
    qs, sp, seat = dev["q_start"].cpu(), dev["start_pos"].cpu(), dev["entry_seat"].cpu()
    rows = []
    for e, n in enumerate(lens):
        for r0 in range(0, n * group, 128):
            rows.append((int(qs[e]), n, int(sp[e]), int(seat[e]), r0, 0, 0, 0))
    rows.sort(key=lambda m: -(m[2] + (min(m[4] + 128, m[1] * group) - 1) // group))     # most keys first
    meta = torch.tensor(rows, dtype=torch.int32, device=gpu)
    out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    per = 0
    if splits > 1:      # key ranges cut anywhere in blocks of 32: some are empty for the short entries
        per = ((max(s + n for s, n in LONG_ENTRIES) + splits - 1) // splits + 31) // 32 * 32
    K.attention_lds(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], meta, nq, nkv, d, scale, window, pair,
                    splits, per)
    close(out, want, torch.bfloat16, f"attention_lds pair={pair} splits={splits}", tol16=8e-3)
    if splits > 1:
        # merged over the items' rows alone: rows of other launches are left as they are
        some = meta[meta[:, 0] == int(qs[2])]
        out2 = torch.full((T, nq * d), 7.0, dtype=torch.bfloat16, device=gpu)
        K.attention_lds(dev["qkv"], stride, out2, dev["kc"], dev["vc"], dev["table"], some, nq, nkv, d, scale,
                        window, False, splits, per, covers_all_rows=False)
        lo, hi = int(qs[2]), int(qs[3])
        assert torch.equal(out2[lo:hi], out[lo:hi]) or (out2[lo:hi].float() - out[lo:hi].float()).abs().max() < 1e-2
        assert bool((out2[:lo] == 7.0).all()) and bool((out2[hi:] == 7.0).all())


@pytest.mark.parametrize("slope", [0.0, 0.35, -0.35, 3.0])
def test_attention_with_scores_that_keep_rising_or_falling(slope, gpu):
    """The kernel re-bases its running softmax only when a row's maximum has moved far; scores
    that climb a little with every key (many small moves), fall, or jump must all give the plain
    softmax.  Keys are made so that q.k grows by ``slope`` per position."""
    nq, nkv, d, page, ctx = 4, 2, 64, 16, 600
    g = torch.Generator().manual_seed(5)
    q = torch.zeros(1, nq, d)
    q[..., 0] = 8.0                                    # scale 1/8: the score is k[..., 0]
    q[..., 1:] = torch.randn(nq, d - 1, generator=g) * 0.05
    k = torch.randn(ctx, nkv, d, generator=g) * 0.05
    k[..., 0] = (torch.arange(ctx, dtype=torch.float32) * slope)[:, None]
    v = torch.randn(ctx, nkv, d, generator=g)
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    want = torch.zeros(1, nq, d, dtype=torch.float64)
    for h in range(nq):
        kh = h // (nq // nkv)
        p = torch.softmax((k[:, kh].double() @ q[0, h].double()) / 8.0, dim=0)
        want[0, h] = p @ v[:, kh].double()
    pages = (ctx + page - 1) // page
    kc = torch.zeros(pages, nkv, page, d, dtype=torch.bfloat16)
    vc = torch.zeros(pages, nkv, d, page, dtype=torch.bfloat16)
    for t in range(ctx):
        kc[t // page, :, t % page, :] = k[t]
        vc[t // page, :, :, t % page] = v[t]
    kc = K.keys_to_pages(kc)
    table = torch.arange(pages, dtype=torch.int32).view(1, pages).to(gpu)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=gpu)
    for splits, per in ((1, 0), (4, 160)):
        out = torch.full((1, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
        K.attention_mfma(q.view(1, nq * d).to(gpu), nq * d, out, kc.to(gpu), vc.to(gpu), table, i32(0), i32(0),
                         i32(0), i32(0, 1), i32(ctx - 1), nq, nkv, d, 1 / 8.0, 0, splits, per, 1)
        close(out.view(1, nq, d), want, torch.bfloat16, f"slope {slope} splits {splits}", tol16=1e-2)


def test_attention_finds_one_far_key_among_hundreds(gpu):
    """One key far back is made to dominate the softmax; a kernel that skips it (a page's edge, a
    split's edge, a wrong mask) returns the average of the others instead of that key's value."""
    nq, nkv, d, page = 4, 1, 64, 16
    ctx = 700
    for far in (0, 15, 16, 31, 32, 255, 256, 511, 698):
        for dtype in ("float32", "bfloat16"):
            dt = DT[dtype]
            g = torch.Generator().manual_seed(far)
            k = torch.randn(ctx, nkv, d, generator=g) * 0.1
            v = torch.randn(ctx, nkv, d, generator=g)
            q = torch.randn(1, nq, d, generator=g) * 0.1
            k[far, 0] = 0
            k[far, 0, 5] = 12.0
            q[0, :, 5] = 12.0                               # score of `far` is 144 / 8 = 18 above the rest
            pages = (ctx + page - 1) // page
            kc = torch.zeros(pages, nkv, page, d)
            vc = torch.zeros(pages, nkv, d, page)
            for p in range(ctx):
                kc[p // page, :, p % page] = k[p]
                vc[p // page, :, :, p % page] = v[p]
            kc = K.keys_to_pages(kc)
            table = torch.arange(pages, dtype=torch.int32)[None].to(gpu)
            qkv = torch.zeros(1, (nq + 2) * d)
            qkv[0, :nq * d] = q.reshape(-1)
            full_q = torch.zeros(ctx, nq, d)
            full_q[-1] = q[0].to(dt).float()
            want = plain.causal_gqa_attention(full_q, k.to(dt).float(), v.to(dt).float(), 1 / 8.0)[-1:].reshape(1, -1)
            assert (want[0, :d] - v[far, 0]).abs().max() < 0.2      # the far key really dominates
            args = (qkv.to(dt).to(gpu), (nq + 2) * d)
            seat = torch.zeros(1, dtype=torch.int32, device=gpu)
            pos = torch.tensor([ctx - 1], dtype=torch.int32, device=gpu)
            out = torch.empty(1, nq * d, dtype=dt, device=gpu)
            K.attention_rowwise(*args, out, kc.to(dt).to(gpu), vc.to(dt).to(gpu), table, seat, pos, nq, nkv, d, 1 / 8.0)
            close(out, want, dt, f"rowwise far={far}", tol32=3e-6, tol16=8e-3)
            if dtype == "bfloat16":
                for splits in (1, 4, 7):
                    per = ((ctx + splits - 1) // splits + 31) // 32 * 32
                    out2 = torch.empty_like(out)
                    K.attention_mfma(*args, out2, kc.to(dt).to(gpu), vc.to(dt).to(gpu), table,
                                     torch.zeros(1, dtype=torch.int32, device=gpu),
                                     torch.zeros(1, dtype=torch.int32, device=gpu), seat,
                                     torch.tensor([0, 1], dtype=torch.int32, device=gpu),
                                     pos.clone(), nq, nkv, d, 1 / 8.0, 0, splits, per if splits > 1 else 0)
                    close(out2, want, dt, f"mfma far={far} splits={splits}", tol16=8e-3)


@pytest.mark.parametrize("nkv, ctx", [(1, 65536), (2, 65536), (4, 131072), (1, 131072)])
def test_attention_of_one_decoded_token_over_a_very_long_context(nkv, ctx, gpu):
    """Few kv heads, one request, a context of 65,536 or 131,072 keys: the split policy wants more
    key ranges than the kernels take and must stop at their limit.  One key at a range's edge is
    made to dominate, so a range that is dropped or counted twice shows."""
    nq, d, page = 2 * nkv, 64, 16
    splits, per = choose_splits(1, nkv, ctx, decoding=True)
    assert K.attention_max_splits() == 256 and splits * per >= ctx
    # 512 wavefronts are wanted at least: with one or two kv heads more splits than the kernels take
    assert splits == (256 if nkv <= 2 else 128)
    far = per * 101 - 1                                   # the last key of range 100
    g = torch.Generator().manual_seed(ctx + nkv)
    k = torch.randn(ctx, nkv, d, generator=g) * 0.1
    v = torch.randn(ctx, nkv, d, generator=g)
    q = torch.randn(nq, d, generator=g) * 0.1
    k[far] = 0
    k[far, :, 3] = 12.0
    q[:, 3] = 12.0
    k, v, q = (t.to(torch.bfloat16) for t in (k, v, q))
    pages = ctx // page
    perm = torch.randperm(pages, generator=g)
    kc = torch.empty(pages, nkv, page, d, dtype=torch.bfloat16)
    vc = torch.empty(pages, nkv, d, page, dtype=torch.bfloat16)
    kc[perm] = k.view(pages, page, nkv, d).permute(0, 2, 1, 3)
    vc[perm] = v.view(pages, page, nkv, d).permute(0, 2, 3, 1)
    kc = K.keys_to_pages(kc)
    # the last row of plain causal attention, written out for one query (the plain function
    # computes every row: 131,072 squared is too much)
    want = torch.empty(nq, d)
    for h in range(nq):
        kh = h // (nq // nkv)
        scores = (k[:, kh].float() @ q[h].float()) / 8.0
        p = torch.softmax(scores.double(), 0).float()
        want[h] = p @ v[:, kh].float()
    assert (want[0] - v[far, 0].float()).abs().max() < 0.3          # that key really dominates
    qkv = torch.zeros(1, (nq + 2 * nkv) * d, dtype=torch.bfloat16)
    qkv[0, :nq * d] = q.reshape(-1)
    out = torch.empty(1, nq * d, dtype=torch.bfloat16, device=gpu)
    zero = torch.zeros(1, dtype=torch.int32, device=gpu)
    K.attention_mfma(qkv.to(gpu), qkv.shape[1], out, kc.to(gpu), vc.to(gpu), perm.to(torch.int32)[None].to(gpu),
                     zero, zero, zero, torch.tensor([0, 1], dtype=torch.int32, device=gpu),
                     torch.tensor([ctx - 1], dtype=torch.int32, device=gpu), nq, nkv, d, 1 / 8.0, 0, splits, per)
    close(out, want.reshape(1, -1), torch.bfloat16, f"{nkv} kv heads, {ctx} keys, {splits} splits", tol16=8e-3)
    with pytest.raises(K.KernelError):                    # and the kernel itself refuses more
        K.attention_mfma(qkv.to(gpu), qkv.shape[1], out, kc.to(gpu), vc.to(gpu), perm.to(torch.int32)[None].to(gpu),
                         zero, zero, zero, torch.tensor([0, 1], dtype=torch.int32, device=gpu),
                         torch.tensor([ctx - 1], dtype=torch.int32, device=gpu), nq, nkv, d, 1 / 8.0, 0, 512, 256)


@pytest.mark.parametrize("items, ctx", [(5, 5000), (12, 2500), (20, 4200), (36, 8300), (7, 8192), (3, 9000)])
def test_several_decoded_tokens_over_long_contexts_with_the_ranges_the_policy_picks(items, ctx, gpu):
    """3 to 63 requests with thousands of keys each (8 kv heads, heads of 64): the policy gives
    every (request, kv head) pair one to ten workgroups of four neighbouring key ranges, some
    ranges of the shorter requests hold no key, and more than one workgroup a pair goes through
    the merge kernel.  Contexts differ per request; in each, one key at a place of its own is made
    to dominate one head, so a range that is dropped, counted twice or given to the wrong request
    shows.  Against every request's last row of plain attention."""
    from kv_cache_optimization_for_llm_amd.ops.attention import choose_decode_ranges
    nq, nkv, d, page = 16, 8, 64, 16
    g = torch.Generator().manual_seed(items * 7 + ctx)
    lens = [ctx] + [int(x) for x in torch.randint(ctx // 3, ctx + 1, (items - 1,), generator=g)]
    bucket = 1 << (ctx - 1).bit_length()
    splits, per, waves = choose_decode_ranges(items, nkv, bucket, d)
    assert waves == 4 and splits % 4 == 0 and splits >= 8, "the shapes of this test are the ones that share workgroups"
    pages_each = [(n + page - 1) // page for n in lens]
    total = sum(pages_each)
    perm = torch.randperm(total, generator=g)
    kc = torch.zeros(total, nkv, page, d, dtype=torch.bfloat16)
    vc = torch.zeros(total, nkv, d, page, dtype=torch.bfloat16)
    table = torch.zeros(items, max(pages_each), dtype=torch.int32)
    qkv = torch.zeros(items, (nq + 2 * nkv) * d, dtype=torch.bfloat16)
    want = torch.empty(items, nq * d)
    at = 0
    for i, n in enumerate(lens):
        k = torch.randn(n, nkv, d, generator=g) * 0.1
        v = torch.randn(n, nkv, d, generator=g)
        q = torch.randn(nq, d, generator=g) * 0.1
        far = (n * (i + 1) // (items + 1)) // per * per           # the first key of some range, another one per request
        k[far] = 0
        k[far, i % nkv, 5] = 12.0
        q[(i % nkv) * 2, 5] = 12.0
        k, v, q = (t.to(torch.bfloat16) for t in (k, v, q))
        mine = perm[at:at + pages_each[i]]
        at += pages_each[i]
        pad = pages_each[i] * page - n
        kp = torch.cat([k, torch.zeros(pad, nkv, d, dtype=torch.bfloat16)]).view(-1, page, nkv, d)
        vp = torch.cat([v, torch.zeros(pad, nkv, d, dtype=torch.bfloat16)]).view(-1, page, nkv, d)
        kc[mine] = kp.permute(0, 2, 1, 3)
        vc[mine] = vp.permute(0, 2, 3, 1)
        table[i, :pages_each[i]] = mine.to(torch.int32)
        qkv[i, :nq * d] = q.reshape(-1)
        kf, vf = k.float().to(gpu), v.float().to(gpu)
        for h in range(nq):
            kh = h // (nq // nkv)
            p = torch.softmax((kf[:, kh] @ q[h].float().to(gpu) / 8.0).double(), 0).float()
            want[i, h * d:(h + 1) * d] = (p @ vf[:, kh]).cpu()
        h = (i % nkv) * 2
        assert (want[i, h * d:(h + 1) * d] - v[far, i % nkv].float()).abs().max() < 0.3       # that key dominates its head
    out = torch.empty(items, nq * d, dtype=torch.bfloat16, device=gpu)
    idx = torch.arange(items, dtype=torch.int32, device=gpu)
    K.attention_mfma(qkv.to(gpu), qkv.shape[1], out, K.keys_to_pages(kc).to(gpu), vc.to(gpu), table.to(gpu),
                     idx, torch.zeros(items, dtype=torch.int32, device=gpu), idx,
                     torch.arange(items + 1, dtype=torch.int32, device=gpu),
                     torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=gpu), nq, nkv, d, 1 / 8.0, 0,
                     splits, per, waves=waves)
    close(out, want, torch.bfloat16, f"{items} requests of up to {ctx} keys in {splits} ranges of {per}", tol16=8e-3)


def test_choose_splits():
    assert choose_splits(4096, 8, 2048) == (1, 0)                 # a big prompt fills the GPU by itself
    s, per = choose_splits(1, 8, 8192)
    assert s > 16 and per % 32 == 0 and s * per >= 8192 and (s - 1) * per < 8192
    assert choose_splits(1, 8, 100) == (1, 0)                     # too short to split
    # decoded tokens: not split at all when they alone give three wavefronts per two compute units,
    # else until there are four per unit, in ranges of at least 64 keys (128 in long contexts)
    assert choose_splits(64, 8, 1024, decoding=True) == (1, 0) == choose_splits(48, 8, 8192, decoding=True)
    assert choose_splits(32, 8, 1024, decoding=True) == (4, 256)
    assert choose_splits(1, 8, 1024, decoding=True) == (16, 64)
    assert choose_splits(1, 8, 8192, decoding=True) == (64, 128)
    assert choose_splits(1, 8, 32768, decoding=True) == (64, 512)      # never more ranges than the merge walks cheaply
    assert choose_splits(2, 8, 32768, decoding=True) == (64, 512)
    assert choose_splits(8, 8, 8192, decoding=True) == (16, 512)


@pytest.mark.parametrize("vocab", [1000, 1001, 128256])
def test_sampler_against_flat_cdf(vocab, gpu):
    """The reference's own check (python/sampling_reference.py:98-108): the chunked two-level walk
    picks the token of the flat CDF for the same draw; plus greedy ties and the penalty."""
    rng = np.random.default_rng(0)
    logits = rng.normal(0.0, 2.0, vocab).astype(np.float32)
    logits[rng.choice(vocab, 20, replace=False)] += 12.0
    rows = 96
    lg = torch.from_numpy(np.tile(logits, (rows, 1))).to(gpu)
    out = torch.empty(rows, dtype=torch.int32, device=gpu)
    temps = [0.7, 1.0, 1.5]
    inv_t = torch.tensor([1.0 / temps[i % 3] for i in range(rows)], device=gpu)
    key = torch.full((rows,), 7, dtype=torch.int32, device=gpu)
    step = torch.arange(rows, dtype=torch.int32, device=gpu)
    # 1,001 tokens in 128 chunks of 8: the last two chunks are empty
    chunks = {1000: 4, 1001: 128, 128256: 128}[vocab]
    K.sample(lg, out, chunks=chunks, inv_temperature=inv_t, seed=1234, rng_key=key, rng_step=step)
    got = out.cpu().numpy()
    bad = 0
    for i in range(rows):
        u = plain.counter_uniform(1234, 7, i)
        w = np.exp((logits.astype(np.float64) - logits.max()) / temps[i % 3])
        cdf = np.cumsum(w)
        want = plain.sample_temperature(logits, temps[i % 3], u)
        if got[i] != want:
            # fp32 partial sums may move a draw that lands within rounding of a boundary
            lo = cdf[got[i] - 1] if got[i] > 0 else 0.0
            assert lo - 1e-4 * cdf[-1] <= u * cdf[-1] <= cdf[got[i]] + 1e-4 * cdf[-1], f"row {i}"
            bad += 1
    assert bad <= 2
    # greedy: lowest id among equal maxima; rows with inv_temperature 0 stay greedy in a mixed batch
    tie = torch.zeros(3, vocab, device=gpu)
    tie[0, [vocab - 1, 500, 777]] = 5.0
    tie[1, 0] = -1.0
    tie[2, vocab - 1] = 1.0
    o3 = torch.empty(3, dtype=torch.int32, device=gpu)
    K.sample(tie, o3, chunks=16)
    assert o3.cpu().tolist() == [500, 1, vocab - 1]
    K.sample(tie, o3, chunks=16, inv_temperature=torch.tensor([0.0, 0.0, 0.0], device=gpu),
             rng_key=key[:3].clone(), rng_step=step[:3].clone())
    assert o3.cpu().tolist() == [500, 1, vocab - 1]
    # repetition penalty on marked tokens only, two-sided
    pl = torch.zeros(2, vocab, device=gpu)
    pl[:, 10], pl[:, 20] = 2.0, 1.9
    pl[1, :] = -3.0
    pl[1, 30], pl[1, 40] = -1.0, -1.1
    mask = torch.zeros(4, vocab, dtype=torch.uint8, device=gpu)
    K.mark_tokens(mask, torch.tensor([2, 3], dtype=torch.int32, device=gpu),
                  torch.tensor([10, 30], dtype=torch.int32, device=gpu))
    o2 = torch.empty(2, dtype=torch.int32, device=gpu)
    K.sample(pl, o2, chunks=8, penalty_mask=mask, row_seat=torch.tensor([2, 3], dtype=torch.int32, device=gpu), penalty=1.15)
    assert o2.cpu().tolist() == [20, 40]                  # 2/1.15 < 1.9 ; -1*1.15 < -1.1
    K.sample(pl, o2, chunks=8, penalty_mask=mask, row_seat=torch.tensor([-1, 0], dtype=torch.int32, device=gpu), penalty=1.15)
    assert o2.cpu().tolist() == [10, 30]                  # seat -1: no penalty; seat 0: nothing marked
    # the launch that chooses a token marks it in the request's mask row (seat -1: nowhere); the
    # mask it reads may be the mask it marks
    K.sample(pl, o2, chunks=8, penalty_mask=mask, row_seat=torch.tensor([2, 3], dtype=torch.int32, device=gpu),
             penalty=1.15, mark_mask=mask, mark_seat=torch.tensor([1, -1], dtype=torch.int32, device=gpu))
    assert o2.cpu().tolist() == [20, 40]
    marked = mask.nonzero().cpu().tolist()
    assert marked == [[1, 20], [2, 10], [3, 30]]


@pytest.mark.parametrize("chunks", [1, 3, 64])
@pytest.mark.parametrize("vocab", [1, 63, 4095, 4096, 4097, 10002, 32000])
def test_sampler_at_the_edges_of_what_a_workgroup_holds(vocab, chunks, gpu):
    """Chunks of more, as many and fewer tokens than a workgroup holds in registers, rows that do not start at multiples
    of 16 bytes, empty last chunks, masked, infinite and NaN logits: the flat CDF's token, or (rounding) one whose
    cumulative weight is within 1e-5 of the target."""
    rows, g = 12, torch.Generator().manual_seed(vocab + chunks)
    lg = torch.randn(rows, vocab, generator=g) * 3
    lg[3] = float("-inf")
    lg[3, vocab // 2] = 1.0
    lg[4, ::2] = float("nan")
    lg[5] = 0.25                                                    # all equal
    mask = (torch.rand(rows, vocab, generator=g) < 0.3).to(torch.uint8)
    inv_t = torch.tensor([0.0, 1.25, 0.5, 2.0, 1.0, 1.0, 0.0, 1.0, 4.0, 1.0, 0.0, 1.0])
    seat = torch.tensor([r if r % 3 else -1 for r in range(rows)], dtype=torch.int32)
    key, step = torch.arange(rows, dtype=torch.int32) * 8, torch.arange(rows, dtype=torch.int32) + 5
    out = torch.empty(rows, dtype=torch.int32, device=gpu)
    K.sample(lg.to(gpu), out, chunks=chunks, inv_temperature=inv_t.to(gpu), seed=77, rng_key=key.to(gpu), rng_step=step.to(gpu),
             penalty_mask=mask.to(gpu), row_seat=seat.to(gpu), penalty=1.15)
    for r in range(rows):
        l, got = lg[r].double().numpy().copy(), int(out[r])
        if seat[r] >= 0:
            l = plain.penalised(l, np.nonzero(mask[r].numpy())[0], 1.15)
        l[np.isnan(l)] = -np.inf
        if not (l > -np.inf).any():
            assert got == -1, r
        elif inv_t[r] == 0:
            assert got == int(np.argmax(l.astype(np.float32))), r
        else:
            w = np.exp((l - l.max()) * float(inv_t[r]))
            cdf, u = np.cumsum(w) / w.sum(), plain.counter_uniform(77, int(key[r]), int(step[r]))
            assert w[got] > 0 and (cdf[got - 1] if got else 0.0) - 1e-5 <= u <= cdf[got] + 1e-5, r


@pytest.mark.parametrize("chunks", [1, 2])
@pytest.mark.parametrize("vocab", [1279, 1280, 1281, 2560, 2561])
def test_sampler_at_the_edges_of_what_a_wavefront_holds(vocab, chunks, gpu):
    test_sampler_at_the_edges_of_what_a_workgroup_holds(vocab, chunks, gpu)


@pytest.mark.parametrize("vocab", [128256, 32003, 160001])
def test_a_row_draws_the_same_token_alone_and_among_others(vocab, gpu):
    """Flat rows: a token's share of the cumulative weights is a hundred roundings wide, so that of some hundred draws several lie
    where another order of the sums would choose the neighbour."""
    from kv_cache_optimization_for_llm_amd.sampling.sampler import Sampler, SampleRow
    rows = 100
    lg = (torch.rand(rows, vocab, generator=torch.Generator().manual_seed(vocab)) * 1e-3).to(gpu)
    sampler = Sampler(vocab, rows, gpu, seed=5)
    for step in range(4):
        which = [SampleRow(r, 0.8, rng_key=8 * r, rng_step=step) for r in range(rows)]
        alone = [int(sampler.sample(lg[r:r + 1], which[r:r + 1])[0]) for r in range(rows)]
        for n in (2, 17, 33, 64, rows):
            assert [int(t) for t in sampler.sample(lg[:n].contiguous(), which[:n])] == alone[:n], n


@pytest.mark.parametrize("how", ["more rows", "dropped"])
def test_row_arguments_stay_until_their_copy_has_left_them(how, gpu):
    """Samplings queued behind a long step: their staging is neither filled again nor handed out as somebody else's pinned
    memory when the next sampling has more rows, or when the sampler is dropped."""
    from kv_cache_optimization_for_llm_amd.sampling.sampler import Sampler, SampleRow
    vocab, rows = 5000, 70
    lg = (torch.randn(rows, vocab, generator=torch.Generator().manual_seed(3)) * 2).to(gpu)
    which = [SampleRow(r, 0.9, rng_key=8 * r, rng_step=9) for r in range(rows)]
    want = Sampler(vocab, rows, gpu, seed=5).sample(lg, which)
    sampler, busy = Sampler(vocab, rows, gpu, seed=5), torch.randn(4096, 4096, device=gpu)
    assert (sampler.sample(lg[:64].contiguous(), which[:64]) == want[:64]).all()
    few = lg[:64].contiguous()
    torch.cuda.synchronize()
    for _ in range(100):
        busy = busy @ busy * 1e-3
    pending = [(sampler.sample_async(few, which[:64]), 64) for _ in range(3)]
    if how == "more rows":
        pending += [(sampler.sample_async(lg[:n].contiguous(), which[:n]), n) for n in (65, 66, rows)]
    del sampler
    others = [torch.full((5, 64), -1, dtype=torch.int32).pin_memory() for _ in range(8)]
    for tokens, n in pending:
        assert (tokens.wait() == want[:n]).all()
    del others


@pytest.mark.parametrize("penalty", [1.0, 1.3])
def test_rows_with_the_launch_and_rows_in_a_copy(penalty, gpu):
    """As many rows as a launch's arguments take, one more, and all of them behind a long step: every row draws what it draws
    alone, and with a penalty leaves the same mask."""
    from kv_cache_optimization_for_llm_amd.sampling.sampler import Sampler, SampleRow
    vocab, most = 2500, K.sample_rows_by_value()
    rows = 3 * most
    lg = (torch.randn(rows, vocab, generator=torch.Generator().manual_seed(4)) * 2).to(gpu)
    which = [SampleRow(r, (0.0, 0.9, 0.7)[r % 3], rng_key=8 * r, rng_step=9, apply_penalty=r % 2 == 0) for r in range(rows)]

    def fresh():
        s = Sampler(vocab, rows, gpu, seed=5, repetition_penalty=penalty)
        s.mark(list(range(rows)), lg.argmax(1).tolist())
        return s
    one = fresh()
    want = [int(one.sample(lg[r:r + 1], which[r:r + 1])[0]) for r in range(rows)]
    busy = torch.randn(4096, 4096, device=gpu)
    for n in (most, most + 1, rows):
        sampler, part = fresh(), lg[:n].contiguous()
        torch.cuda.synchronize()
        for _ in range(50):
            busy = busy @ busy * 1e-3
        pending = sampler.sample_async(part, which[:n])
        if penalty == 1.0:                  # (a mask's marks would change the second one's draws)
            others = [sampler.sample_async(part, which[:n]) for _ in range(2)]
            assert all(o.wait().tolist() == want[:n] for o in others), n
        else:
            torch.cuda.synchronize()
            assert torch.equal(sampler.mask[:n], one.mask[:n])
        assert pending.wait().tolist() == want[:n], n


def test_sampler_takes_keys_and_steps_of_any_integer_type(gpu):
    from kv_cache_optimization_for_llm_amd.sampling.sampler import Sampler, SampleRow
    lg = torch.randn(1, 4000, generator=torch.Generator().manual_seed(1)).to(gpu)
    sampler = Sampler(4000, 1, gpu, seed=5)
    want = int(sampler.sample(lg, [SampleRow(0, 1.0, rng_key=(1 << 32) - 16, rng_step=70000)])[0])
    for key, step in ((-16, 70000), (np.int32(-16), np.int32(70000)), (np.int64(-16), np.uint32(70000)), (np.uint32((1 << 32) - 16), np.int64(70000))):
        assert int(sampler.sample(lg, [SampleRow(0, 1.0, rng_key=key, rng_step=step)])[0]) == want


def test_sampler_distribution_and_boundaries(gpu):
    """python/sampling_reference.py:110-134: top-8 frequencies within 5 % over 40 000 draws."""
    vocab = 5000
    rng = np.random.default_rng(1)
    logits = rng.normal(0.0, 2.0, vocab).astype(np.float32)
    logits[rng.choice(vocab, 20, replace=False)] += 12.0
    probs = np.exp(logits.astype(np.float64) - logits.max())
    probs /= probs.sum()
    draws = 40000
    lg = torch.from_numpy(logits)[None].expand(draws, vocab).contiguous().to(gpu)
    out = torch.empty(draws, dtype=torch.int32, device=gpu)
    K.sample(lg, out, chunks=16, inv_temperature=torch.ones(draws, device=gpu), seed=99,
             rng_key=torch.full((draws,), 3, dtype=torch.int32, device=gpu),
             rng_step=torch.arange(draws, dtype=torch.int32, device=gpu))
    got = out.cpu().numpy()
    assert got.min() >= 0 and got.max() < vocab
    counts = np.bincount(got, minlength=vocab)
    for t in np.argsort(probs)[-8:]:
        assert abs(counts[t] / draws - probs[t]) / probs[t] < 0.05


def test_sampler_writes_the_tokens_to_pinned_host_memory_too(gpu):
    """The kernel that chooses the tokens leaves them in the host's pinned buffer as well: the same
    values as in the device vector once the stream has passed the launch; memory that is not
    pinned is refused before anything is launched."""
    g = torch.Generator().manual_seed(11)
    logits = torch.randn(5, 1001, generator=g).to(gpu)
    out = torch.full((5,), -1, dtype=torch.int32, device=gpu)
    host = torch.full((8,), -7, dtype=torch.int32).pin_memory()
    K.sample(logits, out, chunks=16, host_tokens=host)
    torch.cuda.synchronize()
    assert torch.equal(host[:5], out.cpu()) and torch.equal(out.cpu().long(), logits.cpu().argmax(-1))
    assert (host[5:] == -7).all()
    with pytest.raises(K.KernelError):
        K.sample(logits, out, chunks=16, host_tokens=torch.zeros(8, dtype=torch.int32))


def test_which_host_memory_a_kernel_may_write(gpu):
    assert K.host_memory_is_mapped(torch.zeros(8, dtype=torch.int32).pin_memory())
    assert not K.host_memory_is_mapped(torch.zeros(8, dtype=torch.int32))
    assert not K.host_memory_is_mapped(torch.zeros(8, dtype=torch.int32, device=gpu))


def test_the_read_probes_take_their_ranges_and_refuse_bad_ones(gpu):
    """The probes of the measurement programs store nothing; what can be checked is that they run
    over odd sizes, alone and together, and that a bad range is refused before any launch."""
    sink = torch.zeros(4, dtype=torch.int32, device=gpu)
    own = torch.zeros(5 * 4096 + 48, dtype=torch.uint8, device=gpu)
    shared = torch.zeros(3 * 1024 + 16, dtype=torch.uint8, device=gpu)
    K.stream_read(own, 7, sink)
    K.stream_reread(shared, 5, 3, sink)
    K.stream_mixed(own, shared, 5, sink)
    K.stream_mixed(own, None, 5, sink)
    K.stream_mixed(None, shared, 5, sink)
    torch.cuda.synchronize()
    assert int(sink.abs().sum()) == 0
    with pytest.raises(K.KernelError):
        K.stream_mixed(None, None, 5, sink)
    with pytest.raises(K.KernelError):
        K.stream_mixed(own, shared, 0, sink)


@pytest.mark.parametrize("heads, kv_heads, d, tokens", [(32, 8, 64, 512), (32, 8, 64, 513), (40, 16, 64, 700), (3, 1, 128, 600)])
def test_a_heads_encoding_does_not_depend_on_the_tokens_beside_it(heads, kv_heads, d, tokens, gpu):
    """Either side of where a token's heads go to one workgroup instead of one a turn: rows, keys and values of a token alone."""
    width, pages = (heads + 2 * kv_heads) * d, -(-tokens // 16)
    y = rnd(tokens, width).to(torch.bfloat16).to(gpu)
    pos = torch.arange(tokens, dtype=torch.int32, device=gpu)
    angle = torch.rand((tokens, d // 2), generator=torch.Generator().manual_seed(3)).to(gpu) * 6
    cos, sin = angle.cos(), angle.sin()

    def run(at):
        k = torch.full((pages, kv_heads, d // 8, 16, 8), 7.0, dtype=torch.bfloat16, device=gpu)
        v = torch.full((pages, kv_heads, d, 16), 7.0, dtype=torch.bfloat16, device=gpu)
        rows = y[at].clone()
        K.qk_encode_cache(rows, pos[at], heads, kv_heads, d, d, cos, sin, False, 1e-6, k, v, pos[at])
        return rows, k, v
    rows, k, v = run(slice(0, tokens))
    for t in (0, 17, tokens - 1):
        one, k1, v1 = run(slice(t, t + 1))
        assert torch.equal(one[0], rows[t]), t
        assert torch.equal(k1[t // 16, :, :, t % 16], k[t // 16, :, :, t % 16]) and torch.equal(v1[t // 16, ..., t % 16], v[t // 16, ..., t % 16]), t


@pytest.mark.parametrize("heads, kv_heads, d, tokens", [(16, 4, 64, 1024), (16, 4, 64, 1025), (32, 8, 64, 1025), (3, 1, 32, 1030)])
def test_a_maps_encoding_does_not_depend_on_the_tokens_beside_it(heads, kv_heads, d, tokens, gpu):
    width, pages, dv = 2 * (heads + kv_heads) * d + kv_heads * 2 * d, -(-tokens // 16), 2 * d
    y = rnd(tokens, width).to(torch.bfloat16).to(gpu)
    pos = torch.arange(tokens, dtype=torch.int32, device=gpu)
    angle = torch.rand((tokens, d // 2), generator=torch.Generator().manual_seed(3)).to(gpu) * 6
    cos, sin = angle.cos(), angle.sin()

    def run(at):
        k = torch.full((pages, kv_heads, 2 * d // 8, 16, 8), 7.0, dtype=torch.bfloat16, device=gpu)
        v = torch.full((pages, kv_heads, dv, 16), 7.0, dtype=torch.bfloat16, device=gpu)
        rows = y[at].contiguous()
        q = torch.full((rows.shape[0], 4 * heads * d), 7.0, dtype=torch.bfloat16, device=gpu)
        K.maps_encode_cache(rows, q, pos[at], heads, kv_heads, d, dv, cos, sin, True, k, v, pos[at])
        return q, k, v
    q, k, v = run(slice(0, tokens))
    for t in (0, 17, tokens - 1):
        one, k1, v1 = run(slice(t, t + 1))
        assert torch.equal(one[0], q[t]), t
        assert torch.equal(k1[t // 16, :, :, t % 16], k[t // 16, :, :, t % 16]) and torch.equal(v1[t // 16, ..., t % 16], v[t // 16, ..., t % 16]), t
