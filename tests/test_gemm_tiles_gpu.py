"""Products of more than 64 bf16 rows over the tiled copy of a weight (``csrc/gemm_tiles.hip``) against 64-bit sums."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import kernels as K

pytestmark = pytest.mark.gpu

# rows and outputs a workgroup of every shape, in the order of the kernel's list
SHAPES = [(256, 256), (128, 256), (128, 128), (160, 256), (160, 128), (96, 128), (192, 256), (128, 192), (64, 64), (128, 64)]


@pytest.fixture
def gpu():
    return torch.device("cuda:0")


def operands(m, n, k, gpu, halves=1):
    g = torch.Generator().manual_seed(m * 31 + n * 7 + k)
    x, w = torch.randn((m, k), generator=g).bfloat16(), torch.randn((n, k), generator=g).bfloat16()
    return x, w, x.to(gpu), K.TiledWeight(w.to(gpu), halves)


def sums(x, w):
    """The product and a bound on 32-bit sums of its exact terms: half a unit of the last place an addition, of no more than the sum of the
    terms' sizes."""
    return x.double() @ w.double().t(), (x.double().abs() @ w.double().abs().t()) * (x.shape[1] + 8) * 2.0 ** -24


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("k", [64, 128, 192, 704])
def test_every_shape_at_the_edges_of_its_tiles(shape, k, gpu):
    """One row past a tile, one short of two; outputs that end inside a tile of 16 and inside a workgroup's; fewer stages of K than
    stand in LDS, odd and even numbers of them; nothing else is written."""
    rows, outs = SHAPES[shape]
    for m, n in ((rows + 1, outs + 21), (2 * rows - 1, 3 * outs), (rows, outs - 14)):
        x, w, xd, wt = operands(m, n, k, gpu)
        room = torch.full((m + 16, n), 7.0, dtype=torch.bfloat16, device=gpu)
        K.gemm_tiles(xd, wt, room[8:m + 8], shape + 256)
        want, bound = sums(x, w)
        assert ((room[8:m + 8].double().cpu() - want).abs() <= want.abs() * 2.0 ** -8 + bound).all(), (m, n)
        assert (room[:8] == 7.0).all() and (room[m + 8:] == 7.0).all()


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("splits, k", [(2, 128), (3, 448), (4, 704)])
def test_partial_products_over_ranges_of_k(shape, splits, k, gpu):
    rows, outs = SHAPES[shape]
    m, n = rows + 3, outs + 8
    x, w, xd, wt = operands(m, n, k, gpu)
    parts = torch.full((splits, m, n), 7.0, device=gpu)
    K.gemm_tiles(xd, wt, parts, shape + 256 * splits, K.TILES_PARTS)
    each = -(-(k // 64) // splits) * 64
    for s in range(splits):
        want, bound = sums(x[:, s * each:(s + 1) * each], w[:, s * each:(s + 1) * each])
        assert ((parts[s].double().cpu() - want).abs() <= bound).all()


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_the_activation_of_a_joined_matrix(shape, activation, gpu):
    """Halves that end inside a tile; gates far out on both sides."""
    rows, outs = SHAPES[shape]
    m, n, k = rows + 5, 2 * (outs // 2 + 25), 192
    x, w, xd, wt = operands(m, n, k, gpu, halves=2)
    out = torch.empty((m, n // 2), dtype=torch.bfloat16, device=gpu)
    K.gemm_tiles(xd, wt, out, shape + 256, K.TILES_GATED, activation)
    z, bound = sums(x, w)
    act = torch.nn.functional.silu if activation == "silu" else lambda t: torch.nn.functional.gelu(t, approximate="tanh")
    gate, up = z[:, :n // 2], z[:, n // 2:]
    want = act(gate) * up
    # the activation's slope is below 1.2; its own rounding, 2^-18 of numbers up to |gate|, is far below the result's 2^-8
    slack = 1.2 * bound[:, :n // 2] * up.abs() + act(gate).abs() * bound[:, n // 2:] + 2.0 ** -18 * gate.abs() * up.abs()
    assert ((out.double().cpu() - want).abs() <= want.abs() * 2.0 ** -8 + slack + 1e-30).all()


def test_the_choice_leaves_few_rows_odd_sizes_and_full_turns_to_others(gpu):
    for m, n, k, form in ((64, 4096, 4096, K.TILES_PLAIN), (512, 4096, 4064, K.TILES_PLAIN), (8190, 4096, 14336, K.TILES_PLAIN),
                          (2048, 16, 2048, K.TILES_PLAIN), (512, 1023, 2048, K.TILES_GATED), (512, 2050, 2048, K.TILES_PARTS)):
        assert K.gemm_tiles_plan(m, n, k, form) == -1, (m, n, k, form)
    for m, n, k, form in ((65, 16384, 2048, K.TILES_GATED), (1203, 2048, 8192, K.TILES_PLAIN), (517, 2048, 8192, K.TILES_PARTS)):
        plan = K.gemm_tiles_plan(m, n, k, form)
        assert 0 <= plan % 256 < len(SHAPES) and 1 <= plan >> 8 <= 4
    assert K.gemm_tiles_plan(517, 2048, 8192, K.TILES_PARTS) >> 8 > 1


def test_operands_that_do_not_fit_are_refused(gpu):
    _, _, x, wt = operands(100, 128, 128, gpu)
    out = torch.empty((100, 128), dtype=torch.bfloat16, device=gpu)
    for bad in (dict(out=out[:99]), dict(out=out.float()), dict(x=x.t()), dict(x=x.float()), dict(plan=2), dict(plan=len(SHAPES) + 256),
                dict(plan=8 + 512), dict(form=K.TILES_GATED)):
        with pytest.raises(K.KernelError):
            K.gemm_tiles(bad.get("x", x), wt, bad.get("out", out), bad.get("plan", 8 + 256), bad.get("form", K.TILES_PLAIN))


@pytest.mark.parametrize("rows", [65, 203, 700])
def test_a_feed_forward_of_many_rows_by_tiles(rows, gpu):
    """Joined product with its activation, then the second product whole and as partial sums for a norm that takes them: both run here."""
    from kv_cache_optimization_for_llm_amd.parts.base import BranchTail
    from kv_cache_optimization_for_llm_amd.parts.mlp import SwiGLU
    from kv_cache_optimization_for_llm_amd.parts.norm import RMSNorm
    H, I = 512, 2048
    g = torch.Generator().manual_seed(rows)
    w = {n: (torch.randn(s, generator=g) * 0.03).bfloat16() for n, s in (("gate_proj.weight", (I, H)), ("up_proj.weight", (I, H)),
                                                                         ("down_proj.weight", (H, I)))}
    mlp = SwiGLU("", hidden_size=H, intermediate_size=I)
    mlp.load({n: t.to(gpu) for n, t in w.items()})
    norm = RMSNorm("n.", width=H, eps=1e-5)
    norm.load({n: torch.ones(H, dtype=torch.bfloat16, device=gpu) for n in norm.tensor_specs()})
    x = torch.randn((rows, H), generator=g).bfloat16()
    hidden = torch.zeros((rows, H), dtype=torch.bfloat16, device=gpu)
    z = x.double()
    act = torch.nn.functional.silu(z @ w["gate_proj.weight"].double().t()) * (z @ w["up_proj.weight"].double().t())
    want = act @ w["down_proj.weight"].double().t()
    gated = mlp.gate_up.gated_tiles(x.to(gpu), "silu")
    assert gated is not None and (gated.double().cpu() - act).norm() <= 2.0 ** -8 * act.norm()
    whole = mlp.forward(x.to(gpu), None)
    branch = mlp.forward(x.to(gpu), None, BranchTail(hidden, norm))
    assert isinstance(branch, K.PartialSums) and branch.parts.shape[0] > 1
    for got in (whole, branch.materialize()):
        # activations and result are rounded once each, 2^-9 of them
        assert (got.double().cpu() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("picked", [False, True])
@pytest.mark.parametrize("rows, width", [(300, 2048), (700, 2048), (300, 4096), (700, 4096), (257, 512), (700, 8192)])
def test_the_norm_adds_up_the_ranges_of_many_rows(rows, width, picked, gpu):
    """The stream gets the ranges' sum, rounded to bf16 as a whole product is, and the norm is that of the new stream; where only some rows are asked for,
    they are normed so and the stream stays."""
    from kv_cache_optimization_for_llm_amd.parts.norm import RMSNorm
    g = torch.Generator().manual_seed(rows + width)
    k = 2048
    x, w, xd, wt = operands(rows, width, k, gpu)
    ranges = 2 if rows == 300 else 3
    parts = torch.empty((ranges, rows, width), device=gpu)
    K.gemm_tiles(xd, wt, parts, 9 + 256 * ranges, K.TILES_PARTS)
    stream = (torch.randn((rows, width), generator=g) * 40).bfloat16()
    weight = (torch.rand(width, generator=g) + 0.5).bfloat16()
    norm = RMSNorm("n.", width=width, eps=1e-5)
    norm.load({"n.weight": weight.to(gpu)})
    which = torch.tensor([rows - 1, 0, 130, 255]) if picked else torch.arange(rows)
    hidden = stream.to(gpu)
    out = norm.forward(hidden, delta=K.PartialSums(parts), row_idx=which.to(torch.int32).to(gpu) if picked else None)
    # the ranges in order, in 32 bits, then two roundings to bf16, the sum's and the new stream's: the same bits
    total = parts[0].cpu()
    for r in range(1, ranges):
        total = total + parts[r].cpu()
    want = (stream.float() + total.bfloat16().float()).bfloat16()
    assert torch.equal(hidden.cpu(), stream if picked else want)
    row = want[which].double()
    normed = row / torch.sqrt((row * row).mean(-1, keepdim=True) + 1e-5) * weight.double()
    # one rounding to bf16, half a unit of eight bits, and 32-bit sums of squares in front of it
    assert ((out.double().cpu() - normed).abs() <= normed.abs() * (2.0 ** -8 + 2.0 ** -16)).all()
