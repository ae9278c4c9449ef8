"""The workgroup kernel for prompt portions in blocks of 64 keys and with two groups of wavefronts (``csrc/attention_lds.hip``)."""
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import attention as A
from kv_cache_optimization_for_llm_amd.ops import kernels as K
from test_kernels_gpu import LONG_ENTRIES, attention_case, close

pytestmark = pytest.mark.gpu
FORMS = [A.LDS_BLOCKS_OF_64, A.LDS_TWO_GROUPS]


@pytest.fixture
def gpu():
    return torch.device("cuda:0")


def items(dev, lens, group, gpu):
    qs, sp, seat = dev["q_start"].cpu(), dev["start_pos"].cpu(), dev["entry_seat"].cpu()
    rows = [(int(qs[e]), n, int(sp[e]), int(seat[e]), r0, 0, 0, 0) for e, n in enumerate(lens) for r0 in range(0, n * group, 128)]
    rows.sort(key=lambda m: -(m[2] + (min(m[4] + 128, m[1] * group) - 1) // group))
    return torch.tensor(rows, dtype=torch.int32, device=gpu)


@pytest.mark.parametrize("kind", FORMS)
@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("nq, nkv, d, window, entries", [
    (4, 2, 32, 0, LONG_ENTRIES), (32, 8, 64, 0, LONG_ENTRIES), (8, 2, 64, 70, LONG_ENTRIES), (6, 2, 96, 0, LONG_ENTRIES), (24, 8, 128, 0, LONG_ENTRIES),
    (5, 1, 64, 0, LONG_ENTRIES), (3, 3, 128, 150, LONG_ENTRIES),
    # one key; contexts that end at, one before and one behind a block of 32 and of 64; pages of more keys than stand in LDS at once
    (4, 1, 64, 0, [(0, 1), (0, 31), (0, 32), (1, 32), (0, 63), (1, 63), (33, 32), (96, 33)]),
    (4, 1, 128, 0, [(0, 1), (0, 31), (0, 32), (1, 32), (0, 63), (1, 63), (33, 32), (96, 33)]),
    (2, 1, 64, 0, [(16300, 150), (16384, 3)]), (2, 1, 128, 0, [(16300, 150), (16384, 3)])])
def test_other_forms_of_the_workgroup_kernel(kind, pair, nq, nkv, d, window, entries, gpu):
    """Against the plain formulation, with what the pages held before set to NaN: masked keys and blocks without a key leave nothing.  (Probabilities
    are rounded to bf16 in front of the second product, the result once more: 2 x 2^-9 of the largest, as for the other forms.)"""
    dev, want, T, stride, scale, lens = attention_case("bfloat16", nq, nkv, d, 16, window, entries, 3, gpu, stale=float("nan"))
    out = torch.full((T, nq * d), float("nan"), dtype=torch.bfloat16, device=gpu)
    K.attention_lds(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], items(dev, lens, nq // nkv, gpu), nq, nkv, d, scale, window, pair,
                    kind=kind)
    close(out, want, torch.bfloat16, f"kind={kind} pair={pair}", tol16=8e-3)


@pytest.mark.parametrize("kind", FORMS)
def test_forms_with_key_ranges_are_refused(kind, gpu):
    dev, _, T, stride, scale, lens = attention_case("bfloat16", 4, 2, 64, 16, 0, LONG_ENTRIES, 3, gpu)
    out = torch.empty((T, 4 * 64), dtype=torch.bfloat16, device=gpu)
    with pytest.raises(K.KernelError):
        K.attention_lds(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], items(dev, lens, 2, gpu), 4, 2, 64, scale, 0, False, 2, 192, kind=kind)
    with pytest.raises(K.KernelError):
        K.attention_lds(dev["qkv"], stride, out, dev["kc"], dev["vc"], dev["table"], items(dev, lens, 2, gpu), 4, 2, 64, scale, kind=3)
