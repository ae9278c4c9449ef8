"""Per-row arguments of a sampling: the native reader against the comprehensions it stands for, bit for bit."""
import types

import numpy as np
import pytest
import torch

from kv_cache_optimization_for_llm_amd.ops import build
from kv_cache_optimization_for_llm_amd.ops.library import sample_rows
from kv_cache_optimization_for_llm_amd.sampling import sampler as S


def staging(rows):
    s = types.SimpleNamespace(pinned=torch.full((5, rows), -7, dtype=torch.int32))
    s.i32 = s.pinned.numpy()
    s.u32, s.f32 = s.i32.view(np.uint32), s.i32.view(np.float32)
    return s


ROWS = [S.SampleRow(0), S.SampleRow(3, 0.8, 8, 100), S.SampleRow(7, -1.0, -5, 1 << 40, True), S.SampleRow(np.int64(2), np.float32(1.5), np.int64(-1), np.uint8(9)),
        S.SampleRow(5, 2, (1 << 70) + 3, 7.9, np.bool_(True)), S.SampleRow(1, float("nan"), True, 2), S.SampleRow(4, 1e-45, np.uint32(0xFFFFFFFF), -(1 << 33))]


@pytest.mark.parametrize("rows, room", [([], 1), (ROWS[:1], 1), (ROWS, 7), (tuple(ROWS * 20), 256)])
@pytest.mark.parametrize("seats", [False, True])
def test_native_reader_against_the_comprehensions(rows, room, seats, monkeypatch):
    assert sample_rows() is not None
    got, want = staging(room), staging(room)
    with np.errstate(over="ignore"):
        flags = S._read_rows(rows, len(rows), got, seats)
        assert flags == S._read_rows(rows, len(rows), None, False)
        monkeypatch.setattr(S, "sample_rows", lambda: None)
        assert flags == S._read_rows(rows, len(rows), want, seats)
    assert np.array_equal(got.i32, want.i32)


@pytest.mark.parametrize("rows", [ROWS, ROWS[:1] * 3, [r for r in ROWS if not r.apply_penalty], []])
@pytest.mark.parametrize("mask", [False, True])
def test_what_is_used_in_one_call(rows, mask, monkeypatch):
    got, want = S._Staging(8, pin=False), S._Staging(8, pin=False)
    with np.errstate(over="ignore"):
        flags = S._read_rows_as_used(rows, len(rows), got, mask)
        monkeypatch.setattr(S, "sample_rows", lambda: None)
        assert flags == S._read_rows_as_used(rows, len(rows), want, mask)
    if not flags & 1:                       # (no temperature: nothing of the first array is used)
        want.i32[0] = got.i32[0]
    assert np.array_equal(got.i32, want.i32)


def test_what_the_comprehensions_raise_is_raised():
    with pytest.raises(AttributeError):
        S._read_rows([types.SimpleNamespace(temperature=0.5)], 1, staging(1), False)
    with pytest.raises(TypeError):
        S._read_rows([S.SampleRow(0, None)], 1, staging(1), False)
    with pytest.raises((ValueError, TypeError)):
        S._read_rows([S.SampleRow(0, 0.5, "x")], 1, staging(1), False)
    with pytest.raises(OverflowError):
        S._read_rows([S.SampleRow(1 << 40, 0.5)], 1, staging(1), True)


def test_what_a_sampling_does_not_need_is_not_read():
    """Rows need no more than what is asked for, and a seat may be of any type that an array takes."""
    greedy, seated = types.SimpleNamespace(temperature=0.0), types.SimpleNamespace(seat=3.0)
    assert S._read_rows([greedy] * 2, 2, None, False, penalty=False) == 0
    got = staging(2)
    assert S._read_rows([seated] * 2, 2, got, True, sampled=False, penalty=False) == 0
    assert got.i32.tolist() == [[-7, -7]] * 4 + [[3, 3]]
    drawn = types.SimpleNamespace(temperature=0.5, rng_key=4, rng_step=5)
    got = staging(1)
    assert S._read_rows([drawn], 1, got, False, penalty=False) == 1
    assert got.f32[0, 0] == 2.0 and got.i32[1:, 0].tolist() == [4, 5, -7, -7]
    for asked in (dict(sampled=False), dict(penalty=False)):
        with pytest.raises(AttributeError):
            S._read_rows([types.SimpleNamespace()], 1, None, False, **asked)


@pytest.mark.gpu
def test_greedy_rows_need_a_temperature_and_with_a_penalty_a_seat(gpu):
    logits = torch.randn((3, 300), generator=torch.Generator().manual_seed(1)).to(gpu)
    best = logits.argmax(1).tolist()
    assert S.Sampler(300, 4, gpu).sample(logits, [types.SimpleNamespace(temperature=0.0)] * 3).tolist() == best
    rows = [types.SimpleNamespace(temperature=0.0, apply_penalty=False, seat=i) for i in range(3)]
    assert S.Sampler(300, 4, gpu, repetition_penalty=1.5).sample(logits, rows).tolist() == best


def test_every_interpreter_has_a_host_library_of_its_own(monkeypatch, tmp_path):
    name, digest, var, paths = build.host_name(), build.host_digest(), build.sysconfig.get_config_var, build.sysconfig.get_paths()
    with monkeypatch.context() as m:
        m.setattr(build.sysconfig, "get_config_var", lambda key: "cpython-399-elsewhere" if key == "SOABI" else var(key))
        assert build.host_name() != name and build.host_digest() != digest
    with monkeypatch.context() as m:            # built without the headers: not what is asked for once they are there
        m.setattr(build.sysconfig, "get_paths", lambda: dict(paths, include=str(tmp_path)))
        assert build.host_name() == name and build.host_digest() != digest
    assert (build.host_name(), build.host_digest()) == (name, digest)
