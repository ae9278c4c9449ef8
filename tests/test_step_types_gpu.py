"""The passes between branches, one kernel for each set of types that is common and one for any: every set against 64 bits."""
import itertools

import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu
B, F, D = torch.bfloat16, torch.float32, torch.float64
TYPES = list(itertools.product((B, F), repeat=3))           # branch output, weights, result


def close(got, want):
    """fp32 sums of up to 8,192 terms and a few roundings (2^-24 each), then one rounding of the result (bf16: 2^-9 of a value)."""
    tol = 2.0 ** -8 if got.dtype == B else 2e-5
    assert (got.to(D) - want).abs().max() <= tol * want.abs().max(), float((got.to(D) - want).abs().max())


def norm(v, w, b, center):
    v = v - v.mean(1, keepdim=True) if center else v
    return v / torch.sqrt((v * v).mean(1, keepdim=True) + 1e-6) * w.to(D) + (0.0 if b is None else b.to(D))


def experts(T, W, g, extra):
    rows, gate = torch.randn(T * 3, W, generator=g).cuda(), torch.randn(T, generator=g).cuda()
    e = None if extra is None else torch.randn(T, W, generator=g).to(extra).cuda()
    x = torch.empty((T, W), dtype=B, device="cuda")
    er = K.ExpertRows(x, rows, torch.zeros((T, 3), dtype=torch.int32, device="cuda"), torch.ones((T, 3), device="cuda"), 3, e, None if e is None else gate)
    want = rows.to(D).view(T, 3, W).sum(1)
    return er, want if e is None else want + torch.sigmoid(gate.to(D))[:, None] * e.to(D)


@pytest.mark.parametrize("y_t, w_t, out_t", TYPES)
@pytest.mark.parametrize("T, W", [(1, 2048), (5, 36), (3, 4096)])
def test_steps(T, W, y_t, w_t, out_t, gpu):
    g = torch.Generator().manual_seed(T * W)

    def r(*shape, t=F):
        return torch.randn(*shape, generator=g).to(t).cuda()
    w, b, w2, b2 = (r(W, t=w_t) for _ in range(4))
    for y, yd in ((None, None), (r(T, W, t=y_t),) * 2, experts(T, W, g, y_t), experts(T, W, g, None)):
        yd = None if yd is None else yd.to(D)
        x = r(T, W)
        want = x.to(D) + (0.0 if yd is None else norm(yd, w, b, True))
        out = torch.empty((T, W), dtype=out_t, device="cuda")
        K.sandwich_step(x, y=y, post=None if y is None else (w, b, 1e-6, True), pre=(w2, None, 1e-6, False), out=out)
        close(x, want)
        close(out, norm(want, w2, None, False))
        x = r(T, W)
        want = x.to(D) + (0.0 if yd is None else torch.tanh(0.7 * yd) * w.to(D) + b.to(D))
        K.tanh_step(x, y=y, post=None if y is None else (w, b, 0.7), pre=(w2, b2, 0.3), out=out)
        close(x, want)
        close(out, torch.tanh(0.3 * want) * w2.to(D) + b2.to(D))


@pytest.mark.parametrize("x_t, w_t, out_t", TYPES)
@pytest.mark.parametrize("d_t", [B, F])
@pytest.mark.parametrize("T, W", [(1, 2048), (5, 40), (2, 4096), (2, 4104), (512, 8192), (513, 6152)])
def test_layer_norm(T, W, d_t, x_t, w_t, out_t, gpu):
    g = torch.Generator().manual_seed(T * W + 1)

    def r(*shape, t=F):
        return torch.randn(*shape, generator=g).to(t).cuda()
    w, w2, d = r(W, t=w_t), r(W, t=w_t), r(T, W, t=d_t)
    for second, sd in ((None, 0.0), (r(T, W, t=d_t),) * 2, experts(T, W, g, d_t)):
        x = r(T, W, t=x_t)
        want = x.to(D) + d.to(D) + (sd if second is None else sd.to(D))
        out, out2 = (torch.empty((T, W), dtype=out_t, device="cuda") for _ in range(2))
        K.layernorm(x, w, 1e-6, out, deltas=(d,) if second is None else (d, second), weight2=w2, out2=out2)
        close(x, want)
        want = x.to(D) if x_t == B else want                # (what is normed is what the stream holds)
        close(out, norm(want, w, None, True))
        close(out2, norm(want, w2, None, True))


@pytest.mark.parametrize("y_t, w_t, out_t", TYPES)
def test_copies_of_the_stream(y_t, w_t, out_t, gpu):
    T, W, S = 3, 1028, 2
    g = torch.Generator().manual_seed(3)
    x, y, w = torch.randn(T, S * W, generator=g).cuda(), torch.randn(T, W, generator=g).to(y_t).cuda(), torch.randn(W, generator=g).to(w_t).cuda()
    mix, ow, iw = (torch.randn(n, generator=g).cuda() for n in ((S, S), (S,), (S,)))
    out = torch.empty((T, W), dtype=out_t, device="cuda")
    old = x.to(D).view(T, S, W)
    want = torch.stack([sum(mix[s, t].to(D) * old[:, s] for s in range(S)) + 0.5 * ow[t].to(D) * y.to(D) for t in range(S)], 1)
    K.hyper_step(x, S, y=y, mix=mix, out_w=ow, mult=0.5, in_w=iw, norm_weight=w, eps=1e-6, out=out)
    close(x.view(T, S, W), want)
    close(out, norm(sum(iw[s].to(D) * want[:, s] for s in range(S)), w, None, True))
