"""The few-rows matrix-core product against a plain fp32 product, at sizes other than the engine's."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu


def rnd(*shape, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("m", [1, 8, 16, 17, 33, 64])
@pytest.mark.parametrize("n, k", [(16, 32), (100, 96), (389, 128), (2048, 2048), (3072, 1024), (48, 8192)])
def test_skinny_product_bf16_and_fp32_outputs(m, n, k, gpu):
    assert K.gemm_skinny_supported(m, n, k)
    x, w = rnd(m, k), rnd(n, k, scale=0.05, seed=1)
    want = x.double() @ w.double().t()
    for dt, tol in ((torch.float32, 1e-5), (torch.bfloat16, 6e-3)):
        out = torch.full((m, n), float("nan"), dtype=dt, device=gpu)
        K.gemm_skinny(x.to(gpu), K.TiledWeight(w.to(gpu)), out)
        err = (out.double().cpu() - want).abs().max() / want.abs().max()
        assert err <= tol, f"{dt}: {err:.3g}"
    # a token's result does not depend on the batch it is in (bitwise)
    one = torch.empty((1, n), dtype=torch.float32, device=gpu)
    full = torch.empty((m, n), dtype=torch.float32, device=gpu)
    K.gemm_skinny(x.to(gpu), K.TiledWeight(w.to(gpu)), full)
    K.gemm_skinny(x[m - 1:].contiguous().to(gpu), K.TiledWeight(w.to(gpu)), one)
    assert torch.equal(one[0], full[m - 1])


@pytest.mark.parametrize("m", [3, 17, 32, 47, 64])
@pytest.mark.parametrize("n, k", [(33000, 96), (66010, 160), (40000, 1024)])
def test_skinny_product_of_vocabulary_sized_matrices(m, n, k, gpu):
    """Several tiles per wave; above 16 rows the waves of a workgroup share X through LDS (K
    ranges that end in half a chunk included)."""
    x, w = rnd(m, k), rnd(n, k, scale=0.05, seed=3)
    want = x.double() @ w.double().t()
    tiled = K.TiledWeight(w.to(gpu))
    out = torch.full((m, n), float("nan"), dtype=torch.float32, device=gpu)
    K.gemm_skinny(x.to(gpu), tiled, out)
    err = (out.double().cpu() - want).abs().max() / want.abs().max()
    assert err <= 1e-5, f"{err:.3g}"
    # a token's result in a batch of its own: the same bits up to 16 rows; above, the workgroups
    # that share X through LDS walk K from different starts, which reorders the fp32 sum
    one = torch.empty((1, n), dtype=torch.float32, device=gpu)
    K.gemm_skinny(x[m - 1:].contiguous().to(gpu), tiled, one)
    if m <= 16:
        assert torch.equal(one[0], out[m - 1])
    else:
        assert float((one[0] - out[m - 1]).abs().max()) <= 2e-6 * float(want.abs().max())


@pytest.mark.parametrize("m", [1, 5, 16, 40, 64])
@pytest.mark.parametrize("inter, k", [(16, 64), (250, 96), (8192, 2048), (56, 160), (14336, 512)])
def test_skinny_product_with_swiglu_epilogue(m, inter, k, gpu):
    x, w = rnd(m, k), rnd(2 * inter, k, scale=0.2, seed=2)
    g = x.double() @ w[:inter].double().t()
    u = x.double() @ w[inter:].double().t()
    want = g * (1 / (1 + torch.exp(-g))) * u
    out = torch.full((m, inter), float("nan"), dtype=torch.bfloat16, device=gpu)
    K.gemm_skinny(x.to(gpu), K.TiledWeight(w.to(gpu), halves=2), out, swiglu=True)
    err = (out.double().cpu() - want).abs().max() / want.abs().max()
    assert err <= 6e-3, f"{err:.3g}"


def test_skinny_product_refuses_what_it_cannot_do(gpu):
    assert not K.gemm_skinny_supported(65, 16, 32) and not K.gemm_skinny_supported(4, 16, 40)
    x, w = rnd(4, 40).to(gpu), rnd(16, 40).to(gpu)
    with pytest.raises(K.KernelError):
        K.TiledWeight(w)                                   # K is not a multiple of 32
    with pytest.raises(K.KernelError):
        K.gemm_skinny(x, w, torch.empty((4, 16), dtype=torch.bfloat16, device=gpu))
    tw = K.TiledWeight(rnd(50, 64).to(gpu))                # 50 rows are padded to 64
    # [tile][step of 32][quarter of the step][row][8]: rows 2..15 of the last tile are the padding
    assert tw.data.shape == (4, 2, 4, 16, 8) and tw.data[3, :, :, 2:].abs().max() == 0


def rms(h, w, eps):
    return h * torch.rsqrt((h * h).mean(-1, keepdim=True) + eps) * w


@pytest.mark.parametrize("m", [1, 8, 33, 64])
@pytest.mark.parametrize("n, k", [(2048, 2048), (96, 160), (389, 64), (512, 8192)])
def test_product_adds_into_the_stream_and_prepares_the_next_norm(m, n, k, gpu):
    """EPI_RESID: hidden += x W^T (rounded), scaled = round(hidden * w_next), partial sums of
    hidden^2; a following product that takes (scaled, sumsq) equals norm-then-product."""
    x, w = rnd(m, k), rnd(n, k, scale=0.05, seed=1)
    h0 = rnd(m, n, seed=2)
    w_next = (1 + 0.1 * torch.randn(n, generator=torch.Generator().manual_seed(3)))
    eps = 2e-6
    for wn in (w_next.to(torch.bfloat16), w_next.float()):            # norm weight stored in bf16 or fp32
        hidden = h0.clone().to(gpu)
        scaled = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
        parts = K.gemm_skinny_sumsq_parts(n)
        assert parts in ((n + 15) // 16, 2 * ((n + 15) // 16))      # twice as many where tiles are halved
        sumsq = torch.full((m, parts), float("nan"), device=gpu)
        K.gemm_skinny(x.to(gpu), K.TiledWeight(w.to(gpu)), None, hidden=hidden, next_weight=wn.to(gpu), scaled_out=scaled,
                      sumsq_out=sumsq)
        want_h = (h0.float() + (x.double() @ w.double().t()).float()).to(torch.bfloat16)
        diff = (hidden.cpu().float() - want_h.float()).abs().max() / want_h.float().abs().max()
        assert diff <= 8e-3                                            # one bf16 ulp where a sum sits on a tie
        hf = hidden.cpu().float()
        assert torch.allclose(sumsq.cpu().sum(-1), (hf * hf).sum(-1), rtol=1e-5)
        assert torch.equal(scaled.cpu(), (hf * wn.float()).to(torch.bfloat16))
        # finishing the norm alone
        fin = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
        K.normed_rows_finish(scaled, sumsq, n, eps, fin)
        want_norm = rms(hf, wn.float(), eps)
        assert (fin.cpu().float() - want_norm).abs().max() <= 1.2e-2 * want_norm.abs().max()
        rows = torch.tensor([m - 1, 0, m - 1], dtype=torch.int32, device=gpu)
        fin3 = torch.empty((3, n), dtype=torch.bfloat16, device=gpu)
        K.normed_rows_finish(scaled, sumsq, n, eps, fin3, rows)
        assert torch.equal(fin3.cpu(), fin.cpu()[rows.cpu().long()])
        # a following product finishes the norm in its epilogue (needs its K = n to be a multiple of 32)
        if n % 32 == 0:
            w2 = rnd(80, n, scale=0.05, seed=4)
            out = torch.empty((m, 80), dtype=torch.float32, device=gpu)
            K.gemm_skinny(scaled, K.TiledWeight(w2.to(gpu)), out, sumsq=sumsq, norm_width=n, eps=eps)
            want = want_norm.double() @ w2.double().t()
            assert (out.cpu().double() - want).abs().max() <= 6e-3 * want.abs().max()
            act = torch.empty((m, 40), dtype=torch.bfloat16, device=gpu)
            K.gemm_skinny(scaled, K.TiledWeight(w2.to(gpu), halves=2), act, swiglu=True, sumsq=sumsq, norm_width=n, eps=eps)
            g, u = want[:, :40], want[:, 40:]
            want_act = g * (1 / (1 + torch.exp(-g))) * u
            assert (act.cpu().double() - want_act).abs().max() <= 1e-2 * want_act.abs().max()


def test_wide_matrices_give_a_wave_several_tiles(gpu):
    """N >= 32768 and >= 65536 switch to 2 and 4 n-tiles per wave (the vocabulary-sized product)."""
    for n in (32768 + 48, 65536 + 16, 128256):
        x, w = rnd(5, 64), rnd(n, 64, scale=0.1, seed=n)
        out = torch.full((5, n), float("nan"), dtype=torch.float32, device=gpu)
        K.gemm_skinny(x.to(gpu), K.TiledWeight(w.to(gpu)), out)
        want = x.double() @ w.double().t()
        assert (out.cpu().double() - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("m", [1, 7, 16, 17, 35, 64])
@pytest.mark.parametrize("nq, nkv, d, page, k", [(4, 2, 32, 16, 64), (6, 1, 96, 8, 160), (3, 3, 64, 4, 2048),
                                                 (32, 8, 64, 16, 2048)])
@pytest.mark.parametrize("rotate, normed", [(True, False), (True, True), (False, False)])
def test_qkv_product_rotates_and_writes_the_cache(m, nq, nkv, d, page, k, rotate, normed, gpu):
    """The fused projection equals product -> round -> rotate-half rotation -> cache write done
    one after the other in fp32 (the cache is checked slot by slot, untouched slots stay zero)."""
    import plain_llama as plain
    n = (nq + 2 * nkv) * d
    x, w = rnd(m, k), rnd(n, k, scale=0.05, seed=1)
    pos = [(37 * i + 3) % 300 for i in range(m)]
    pages = (m + page - 1) // page + 3
    perm = torch.randperm(pages * page, generator=torch.Generator().manual_seed(m))[:m].to(torch.int32)
    slots = perm.clone()
    if m > 2:
        slots[2] = -1
    inv = plain.rope_inv_freq(d, 20000.0, dict(rope_type="llama3", factor=4.0, low_freq_factor=1.0,
                                               high_freq_factor=2.0, original_max_position_embeddings=64))
    cos, sin = plain.rope_cos_sin(range(300), inv)
    y = x.double() @ w.double().t()
    extra = {}
    xin = x
    if normed:
        # x is an unfinished norm input: (scaled, partial sums of squares of the stream)
        parts = 5
        sumsq = torch.rand(m, parts, generator=torch.Generator().manual_seed(9)) * 40 + 1
        eps, width = 3e-6, 100
        y = y * torch.rsqrt(sumsq.double().sum(-1, keepdim=True) / width + eps)
        extra = dict(sumsq=sumsq.to(gpu), norm_width=width, eps=eps)
    y = y.float().to(torch.bfloat16).float()                            # what a separate product leaves
    q_want = y[:, :nq * d].view(m, nq, d).clone()
    k_want = y[:, nq * d:(nq + nkv) * d].view(m, nkv, d).clone()
    v_want = y[:, (nq + nkv) * d:].view(m, nkv, d)
    if rotate:
        c, s = plain.rope_cos_sin(pos, inv)
        q_want = plain.apply_rope(q_want, c, s)
        k_want = plain.apply_rope(k_want, c, s)
    k_cache = K.keys_to_pages(torch.zeros(pages, nkv, page, d, dtype=torch.bfloat16, device=gpu))
    v_cache = torch.zeros(pages, nkv, d, page, dtype=torch.bfloat16, device=gpu)
    q = torch.full((m, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    assert K.gemm_skinny_qkv_rope_supported(m, k, d)
    K.gemm_skinny_qkv_rope(xin.to(gpu), K.TiledWeight(w.to(gpu)), q, nq, nkv, d,
                           torch.tensor(pos, dtype=torch.int32, device=gpu),
                           torch.from_numpy(cos).to(gpu) if rotate else None,
                           torch.from_numpy(sin).to(gpu) if rotate else None,
                           k_cache, v_cache, slots.to(gpu), page, **extra)
    scale = y.abs().max()
    assert (q.float().cpu().view(m, nq, d) - q_want).abs().max() <= 1e-2 * scale
    kc, vc = K.pages_to_keys(k_cache).float().cpu(), v_cache.float().cpu()
    for t in range(m):
        sl = int(slots[t])
        if sl < 0:
            continue
        assert (kc[sl // page, :, sl % page, :] - k_want[t]).abs().max() <= 1e-2 * scale, f"k of row {t}"
        assert (vc[sl // page, :, :, sl % page] - v_want[t]).abs().max() <= 1e-2 * scale, f"v of row {t}"
    written = {int(sl) for sl in slots if sl >= 0}
    for sl in range(pages * page):
        if sl not in written:
            assert kc[sl // page, :, sl % page, :].abs().max() == 0 and vc[sl // page, :, :, sl % page].abs().max() == 0
    # without a cache only Q is produced
    q2 = torch.empty_like(q)
    K.gemm_skinny_qkv_rope(xin.to(gpu), K.TiledWeight(w.to(gpu)), q2, nq, nkv, d,
                           torch.tensor(pos, dtype=torch.int32, device=gpu),
                           torch.from_numpy(cos).to(gpu) if rotate else None,
                           torch.from_numpy(sin).to(gpu) if rotate else None, None, None, None, 0, **extra)
    assert torch.equal(q2, q)


def test_qkv_product_refuses_head_sizes_it_cannot_pair(gpu):
    assert not K.gemm_skinny_qkv_rope_supported(4, 64, 48) and not K.gemm_skinny_qkv_rope_supported(4, 64, 16)
    w = K.TiledWeight(rnd(4 * 48, 64).to(gpu))
    with pytest.raises(K.KernelError):
        K.gemm_skinny_qkv_rope(rnd(4, 64).to(gpu), w, torch.empty((4, 96), dtype=torch.bfloat16, device=gpu), 2, 1, 48,
                               torch.zeros(4, dtype=torch.int32, device=gpu), None, None, None, None, None, 0)


@pytest.mark.parametrize("m", [1, 33, 64, 200, 2048])
@pytest.mark.parametrize("n, k", [(2048, 2048), (3072, 1024), (389, 96), (100, 40), (8192, 256)])
def test_vendor_product_bf16_and_fp32_results(m, n, k, gpu):
    """The library product called directly (descriptors and algorithm kept per shape): against a
    plain product, twice per shape (the second call takes the kept plan), bf16 and fp32 results.
    A shape the library has no algorithm for returns False and launches nothing."""
    x, w = rnd(m, k), rnd(n, k, scale=0.05, seed=4)
    want = x.double() @ w.double().t()
    for dt, tol in ((torch.bfloat16, 6e-3), (torch.float32, 2e-5)):
        for _ in range(2):
            out = torch.full((m, n), float("nan"), dtype=dt, device=gpu)
            if not K.gemm_vendor(x.to(gpu), w.to(gpu), out):
                assert torch.isnan(out).all()
                continue
            err = (out.double().cpu() - want).abs().max() / want.abs().max()
            assert err <= tol, f"{dt}: {err:.3g}"


@pytest.mark.parametrize("m", [17, 31, 48, 64])
@pytest.mark.parametrize("n, k", [(2048, 8192), (2048, 2048), (100, 128), (389, 384), (48, 1024), (3072, 3072)])
def test_partial_products_over_ranges_of_k_add_up_to_the_product(m, n, k, gpu):
    """17 to 64 rows of a matrix with few rows of tiles: K is cut into ranges across workgroups
    (as many as fill the chip; one for a small K), each range leaves an fp32 partial product, and
    their sum is the product.  The norm kernel takes the ranges in place of a bf16 delta: the
    stream and the normalised rows are bit for bit what the rounded sum gives.  Fewer rows, and
    a K that 128 does not divide, are refused."""
    ranges = K.gemm_skinny_partial_ranges(m, n, k)
    assert ranges >= 1 and k % (ranges * 128) == 0
    x, w = rnd(m, k), rnd(n, k, scale=0.05, seed=7)
    want = x.double() @ w.double().t()
    ps = K.gemm_skinny_partials(x.to(gpu), K.TiledWeight(w.to(gpu)))
    assert ps.parts.shape == (ranges, m, n) and tuple(ps.shape) == (m, n)
    total = ps.parts.double().sum(0).cpu()
    assert (total - want).abs().max() <= 2e-5 * want.abs().max()
    # as a delta of the norm kernel: the same as its sum (ranges added in order, in fp32) rounded to bf16
    if n % 8 == 0:
        seq = ps.parts[0].clone()
        for r in range(1, ranges):
            seq += ps.parts[r]
        delta = seq.to(torch.bfloat16)
        hidden = rnd(m, n, seed=8)
        wn = (1 + 0.1 * rnd(n, seed=9).float()).to(torch.bfloat16).to(gpu)
        h1, h2 = hidden.clone().to(gpu), hidden.clone().to(gpu)
        o1, o2 = torch.empty_like(h1), torch.empty_like(h2)
        K.rmsnorm(h1, wn, 1e-5, o1, delta=ps)
        K.rmsnorm(h2, wn, 1e-5, o2, delta=delta)
        assert torch.equal(h1, h2) and torch.equal(o1, o2)
        rows = torch.tensor([m - 1, 0, 5, 5], dtype=torch.int32, device=gpu)
        g1, g2 = torch.empty((4, n), dtype=torch.bfloat16, device=gpu), torch.empty((4, n), dtype=torch.bfloat16, device=gpu)
        K.rmsnorm(h1, wn, 1e-5, g1, delta=ps, row_idx=rows)
        K.rmsnorm(h2, wn, 1e-5, g2, delta=delta, row_idx=rows)
        assert torch.equal(g1, g2) and torch.equal(h1, h2)
        assert torch.equal(ps.materialize(), delta)
    assert K.gemm_skinny_partial_ranges(16, n, k) == 0 and K.gemm_skinny_partial_ranges(65, n, k) == 0
    assert K.gemm_skinny_partial_ranges(m, n, 96) == 0
    with pytest.raises(K.KernelError):
        K.gemm_skinny_partials(x[:16].contiguous().to(gpu), K.TiledWeight(w.to(gpu)))


@pytest.mark.parametrize("m", [1, 7, 8, 9, 16, 40, 64])
@pytest.mark.parametrize("inter, hidden", [(8192, 2048), (256, 96), (96, 64)])
def test_activations_pass_between_two_products_in_lane_order(m, inter, hidden, gpu):
    """The gated product can leave its result as TiledRows ([columns / 8][rows rounded up to 16, or 8 rows for up to 8][8])
    and the residual product can read its X in that layout: bit for bit what the row-major route gives."""
    x = rnd(m, hidden).to(gpu)
    w_gu = K.TiledWeight(rnd(2 * inter, hidden, scale=0.2, seed=5).to(gpu), halves=2)
    w_down = K.TiledWeight(rnd(hidden, inter, scale=0.05, seed=6).to(gpu))
    act_rows = torch.empty((m, inter), dtype=torch.bfloat16, device=gpu)
    K.gemm_skinny(x, w_gu, act_rows, swiglu=True)
    act_tiled = K.TiledRows(m, inter, gpu)
    act_tiled.data.fill_(float("nan"))                       # rows past m stay unwritten and must not matter
    K.gemm_skinny(x, w_gu, act_tiled, swiglu=True, out_tiled=True)
    assert torch.equal(act_tiled.to_rows(), act_rows)
    parts = K.gemm_skinny_sumsq_parts(hidden)
    results = []
    for a in (act_rows, act_tiled):
        h = rnd(m, hidden, seed=7).to(gpu)
        scaled = torch.empty((m, hidden), dtype=torch.bfloat16, device=gpu)
        sumsq = torch.empty((m, parts), device=gpu)
        K.gemm_skinny(a, w_down, None, hidden=h, next_weight=None, scaled_out=scaled, sumsq_out=sumsq,
                      x_tiled=a is act_tiled)
        results.append((h, scaled, sumsq))
    for u, v in zip(*results):
        assert torch.equal(u, v)
    with pytest.raises(K.KernelError):
        K.TiledRows(65, 64, gpu)


def test_vendor_product_keeps_the_fastest_algorithm_and_the_same_result(gpu):
    """Timing every algorithm of the vendor library for a shape keeps one that is no slower than
    the library's own choice and computes the same product."""
    m, n, k = 64, 512, 1024
    ws = [rnd(n, k, scale=0.05, seed=s).to(gpu) for s in range(3)]
    x = rnd(m, k, seed=9).to(gpu)
    out = torch.empty((m, n), dtype=torch.bfloat16, device=gpu)
    assert K.gemm_vendor(x, ws[1], out)
    before = out.clone()
    first, best, tried = K.gemm_vendor_tune(m, ws)
    assert tried >= 1 and 0 < best <= first
    assert K.gemm_vendor(x, ws[1], out)
    want = x.double().cpu() @ ws[1].double().cpu().t()
    for got in (before, out):
        assert (got.double().cpu() - want).abs().max() / want.abs().max() <= 2 ** -8
    # a row count that was not timed itself takes the algorithm of the timed one above it
    x40 = rnd(40, k, seed=10).to(gpu)
    out40 = torch.empty((40, n), dtype=torch.bfloat16, device=gpu)
    assert K.gemm_vendor(x40, ws[2], out40)
    want40 = x40.double().cpu() @ ws[2].double().cpu().t()
    assert (out40.double().cpu() - want40).abs().max() / want40.abs().max() <= 2 ** -8
    with pytest.raises(K.KernelError):
        K.gemm_vendor_tune(m, [ws[0], rnd(n, k + 32, seed=1).to(gpu)])


@pytest.mark.parametrize("m, n, k", [(4096, 4128, 64), (2000, 8224, 96), (2048, 4128, 64), (4096, 4129, 32), (2048, 8208, 2048), (1793, 8193, 512)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_a_few_outputs_past_a_multiple_of_256_in_a_product_of_their_own(m, n, k, out_dtype, gpu):
    """Both sides of where the product is cut in two, by turns of tiles and by what is left of the outputs; nothing else of the result is
    written."""
    from kv_cache_optimization_for_llm_amd.ops.gemm_bf16 import linear_bf16, vendor_cut
    assert vendor_cut(m, n) == {(4096, 4128): 4096, (2000, 8224): 8192, (2048, 8208): 8192, (1793, 8193): 8192}.get((m, n), 0)
    g = torch.Generator().manual_seed(m + n)
    x, w = torch.randn((m, k), generator=g).bfloat16(), torch.randn((n, k), generator=g).bfloat16()
    room = torch.full((m + 2, n), 7.0, dtype=out_dtype, device=gpu)
    linear_bf16(x.to(gpu), w.to(gpu), room[1:m + 1])
    want = x.float() @ w.float().t()
    # fp32 sums of K exact products; a bf16 result is rounded once (2^-9 of it)
    bound = want.abs() * (2.0 ** -8 if out_dtype == torch.bfloat16 else 0) + 2.0 ** -20 * k * 4
    assert ((room[1:m + 1].float().cpu() - want).abs() <= bound).all()
    assert (room[0] == 7.0).all() and (room[m + 1] == 7.0).all()


def test_a_cut_product_is_timed_both_ways_and_stays_the_same(gpu, monkeypatch):
    from kv_cache_optimization_for_llm_amd.ops import gemm_bf16 as G
    monkeypatch.setattr(G, "_TIMED_CUTS", {})
    m, n, k = 2048, 8208, 96
    ws = [rnd(n, k, scale=0.05, seed=s).to(gpu) for s in range(2)]
    x = rnd(m, k, seed=9).to(gpu)
    want = x.float().cpu() @ ws[1].float().cpu().t()
    first, best, tried = G.tune_linear(m, ws)
    assert tried >= 3 and 0 < best and first > 0
    two = G._TIMED_CUTS[(x.device, n, k, torch.bfloat16)][m]
    for decided in (two, True, False):
        G._TIMED_CUTS[(x.device, n, k, torch.bfloat16)][m] = decided
        seen, one = [], K.gemm_vendor
        with monkeypatch.context() as patch:
            patch.setattr(K, "gemm_vendor", lambda a, w, out, **kw: seen.append(w.shape[0]) or one(a, w, out, **kw))
            got = G.linear_bf16(x, ws[1], torch.full((m, n), 7.0, dtype=torch.bfloat16, device=gpu))
        assert seen == ([8192, 16] if decided else [8208])
        assert ((got.float().cpu() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -20 * k).all()
