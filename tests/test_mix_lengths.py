"""Chunk lengths of a mixed-queue plan: named ones are kept (and with them the
checkpoints of long chunks), open ones and the tuner's choice are upper bounds."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import cpu as oracle_cpu
from trex_amd.mix import MixEngine, MixParams


def test_when_lengths_are_upper_bounds():
    assert MixParams().upper_bounds() and MixParams(form="slice").upper_bounds()
    assert not MixParams(nfa_chunk=8192, nfa_split=8192).upper_bounds() and not MixParams(ck=256).upper_bounds()
    assert MixParams(nfa_chunk=8192, nfa_split=8192, at_most=True).upper_bounds()
    assert not MixParams(at_most=False).upper_bounds()


def _engines():
    from trex_amd.engine import DfaEngine, NfaEngine
    from trex_amd.nfa_matrices import compile_nfa_matrices
    from trex_amd.regex_to_dfa import compile_regex
    from trex_amd.tables import dfa_byte_table
    dfa = DfaEngine(dfa_byte_table(compile_regex("[A-Z]*(ERROR|WARN)[A-Z]*")))
    nfas = [NfaEngine.from_matrices(compile_nfa_matrices(p)) for p in
            ("[A-Z]*A[A-Z][A-Z][A-Z][A-Z][A-Z]", "([A-Z][A-Z][A-Z])*",
             "(([A-Y][A-Y][A-Y])*([A-Y]|[A-Y][A-Y])?Z)*([A-Y][A-Y][A-Y])*")]
    return [dfa] + nfas


def _longest(m):
    """Longest DFA and NFA chunk of the plan."""
    L = m.layout()
    out = {1: 0, 3: 0}
    for first, count, role in zip(L["bfirst"], L["bcount"], L["brole"]):
        if role in out:
            items = slice(first, first + count)
            out[role] = max(out[role], int((L["iend"][items] - L["ibeg"][items]).max()))
    return out[1], out[3]


def _batch(rng, n, size, kinds):
    offsets = np.arange(n + 1, dtype=np.int64) * size
    return offsets, np.arange(n, dtype=np.int32) % kinds


@pytest.mark.gpu
@pytest.mark.parametrize("params,longest", [
    (MixParams(dfa_split=1 << 16, dfa_chunk=1 << 16, nfa_split=1 << 15, nfa_chunk=1 << 15), (1 << 16, 1 << 15)),
    (MixParams(nfa_split=1 << 14, nfa_chunk=1 << 13, ck=256, dfa_split=1 << 17), (1 << 16, 1 << 13)),
    (MixParams(dfa_split=4096, dfa_chunk=2048, nfa_split=2048, nfa_chunk=1024), (2048, 1024)),
    (MixParams(), (1024, 512)),
    (MixParams(dfa_split=1 << 16, dfa_chunk=1 << 14, nfa_split=1 << 13, nfa_chunk=1 << 13, at_most=True), (1024, 512)),
])
def test_planned_lengths(gpu_lib, params, longest):
    offsets, pattern_of = _batch(None, 8, 300_000, 4)
    m = MixEngine(_engines())
    m.plan(offsets[:-1], offsets[1:], pattern_of, params)
    assert _longest(m) == longest


@pytest.mark.gpu
def test_short_nfa_chunks_leave_dfa_chunks_in_position_order(gpu_lib):
    """DFA bytes that fill the device beside few NFA bytes (no data behind the plan)."""
    from trex_amd._lib import device_info
    n = device_info()["cus"] * 512 * (64 << 10) // (8 << 20) + 1
    begin = np.arange(n + 1, dtype=np.int64) * (8 << 20)
    end = begin + (8 << 20)
    end[-1] = begin[-1] + 100_000
    m = MixEngine(_engines())
    m.plan(begin, end, np.array([0] * n + [1], np.int32))
    assert _longest(m) == (64 << 10, 512)
    L = m.layout()
    b = int(np.flatnonzero(L["brole"] == 1)[0])
    assert np.all(L["iflags"][L["bfirst"][b]:L["bfirst"][b] + L["bcount"][b]] & 1)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["nibble", "slice"])
@pytest.mark.parametrize("n", [40, 1500])
@pytest.mark.parametrize("ck", [64, 256])
def test_checkpoints_of_long_chunks(gpu_lib, form, n, ck):
    """Chunks of 8 KiB record their sets: guesses that are right, that are wrong
    until a letter comes every 4,000 bytes and meet a checkpoint, and that never
    do; strings on and off the checkpoints' grid, fix-ups by wave and by lane."""
    rng = np.random.default_rng(n + ck)
    engines = _engines()[1:]
    lengths = rng.integers(17_000, 19_000, n)
    lengths[:6] = 60_000
    lengths[rng.random(n) < 0.3] = 64 * 300
    begin = np.cumsum(lengths) - lengths + 64 * np.arange(n) // 64 * 64
    begin[1::2] = begin[1::2] // 256 * 256
    data = rng.choice(np.frombuffer(b"BCDFGHIJKLMPQSTUVXYA", np.uint8), int(begin[-1] + lengths[-1]) + 64)
    data[rng.random(len(data)) < 1 / 4000] = ord("Z")
    end = np.minimum(begin + lengths, len(data))
    for eng in engines:
        m = MixEngine([eng])
        offsets = np.zeros(n + 1, np.int64)
        np.cumsum(end - begin, out=offsets[1:])
        packed = np.concatenate([data[x:y] for x, y in zip(begin, end)])
        want, _ = oracle_cpu.nfa_walk(eng.succ, eng.byte_to_sym, eng.start, eng.accept, packed, offsets)
        from trex_amd.device import DeviceBuffer, Stream
        stream = Stream()
        d, d_mask, d_acc = DeviceBuffer.from_array(data, stream), DeviceBuffer(8 * n), DeviceBuffer(n)
        info = m.plan(begin, end, np.zeros(n, np.int32),
                      MixParams(nfa_split=1 << 13, nfa_chunk=1 << 13, ck=ck, form=form))
        m.run(d.ptr, d_mask.ptr, d_acc.ptr, stream)
        assert m.error(stream) == 0
        assert np.array_equal(d_mask.download(np.uint64, n, stream), want)
        later, taken = info["chunks"] - info["fixups"], m.converged(stream)
        if eng is engines[0]:
            assert taken == later
        elif eng is engines[1]:
            assert taken < later
        else:   # nearly all meet a checkpoint in their 8,192 bytes, few are guessed in 256
            assert taken > 0.3 * later


@pytest.mark.gpu
def test_tuner_times_the_lengths_it_names(gpu_lib, tmp_path, monkeypatch):
    from trex_amd.autotune import tune_mix
    from trex_amd.device import DeviceBuffer, Stream
    monkeypatch.setenv("TREX_AMD_TUNE_CACHE", str(tmp_path / "tune.json"))
    offsets, pattern_of = _batch(None, 8, 300_000, 4)
    data = np.full(int(offsets[-1]), ord("A"), np.uint8)
    stream = Stream()
    d = DeviceBuffer.from_array(data, stream)
    timed = []
    run = MixEngine.run
    monkeypatch.setattr(MixEngine, "run", lambda m, *a, **k: (timed.append((m.params, _longest(m))), run(m, *a, **k))[1])
    grid = {"dfa_split": (64 << 10,), "dfa_chunk": (16 << 10, 64 << 10), "nfa_split": (32 << 10,),
            "nfa_chunk": (8 << 10, 32 << 10), "ck": (64,)}
    engines = _engines()
    for source in ("tuned", "cache"):
        params, info = tune_mix(engines, offsets[:-1], offsets[1:], pattern_of, d.ptr, stream, grid=grid)
        assert info["source"] == source and params.upper_bounds()
    assert len({longest for _, longest in timed}) == 4
    assert all(longest == (p.dfa_chunk, p.nfa_chunk) for p, longest in timed)
