"""Long NFA strings of a mixed queue: chunks entered by a guess, and what the
fix-up makes of guesses that are wrong. Results against the C oracle, and the
count of chunks whose recorded end was taken (the others are walked again by
one lane per string, one after another)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import cpu as oracle_cpu
from trex_amd.engine import NfaEngine
from trex_amd.mix import MixEngine, MixParams
from trex_amd.nfa_matrices import compile_nfa_matrices

pytestmark = pytest.mark.gpu
TEXT = np.frombuffer(b"BCDFGHIJKLMPQSTUVXYZA", np.uint8)   # no E, R, O, W, N: words are put in by hand


def _run(eng, data, offsets, params=None):
    """Results checked; chunks after their string's first, and how many were taken as recorded."""
    from trex_amd.device import DeviceBuffer, Stream
    n = len(offsets) - 1
    m = MixEngine([eng])
    info = m.plan(offsets[:-1], offsets[1:], np.zeros(n, np.int32), params)
    stream = Stream()
    d = DeviceBuffer.from_array(data, stream)
    d_mask, d_acc = DeviceBuffer(8 * n), DeviceBuffer(n)
    m.run(d.ptr, d_mask.ptr, d_acc.ptr, stream)
    assert m.error(stream) == 0
    want_mask, want_acc = oracle_cpu.nfa_walk(eng.succ, eng.byte_to_sym, eng.start, eng.accept, data, offsets)
    assert np.array_equal(d_mask.download(np.uint64, n, stream), want_mask)
    assert np.array_equal(d_acc.download(np.uint8, n, stream), want_acc)
    return info["chunks"] - info["fixups"], m.converged(stream)


def _strings(rng, lengths):
    offsets = np.zeros(len(lengths) + 1, np.int64)
    np.cumsum(lengths, out=offsets[1:])
    return rng.choice(TEXT, int(offsets[-1])), offsets


@pytest.mark.parametrize("form", ["nibble", "slice"])
@pytest.mark.parametrize("pattern", ["[A-Z]*(ERROR|WARN)[A-Z]*", "[A-Z]*ERROR[A-Z]*|[A-Z]*WARN[A-Z]*", "(ERROR)[A-Z]*",
                                     "[A-Z]*ERROR[A-Z]*WARN[A-Z]*"])
def test_found_text_stays_known(gpu_lib, pattern, form):
    """Text that is absent, at the start, in the middle or in every chunk: the
    chunks before and behind it are taken as recorded, but for those where a
    string finds it across a chunk's end."""
    rng = np.random.default_rng(5)
    eng = NfaEngine.from_matrices(compile_nfa_matrices(pattern))
    n, size = 24, 70_001
    data, offsets = _strings(rng, np.full(n, size))
    for k in range(n):
        for at in ([], [0], [3000], [size // 2], range(0, size - 8, 300), [0, 40_000])[k % 6]:
            word = b"WARN" if at > 30_000 and k % 2 else b"ERROR"
            data[k * size + at:k * size + at + len(word)] = np.frombuffer(word, np.uint8)
    chunks, taken = _run(eng, data, offsets, MixParams(form=form))
    assert chunks > n * 8
    if pattern.startswith("("):   # a string without its text at byte 0 is empty from its first chunk on
        chunks = chunks * sum(k % 6 in (1, 4, 5) for k in range(n)) // n
    assert taken >= chunks - 2 * n


@pytest.mark.parametrize("form", ["nibble", "slice"])
def test_words_and_rejects_around_chunk_ends(gpu_lib, form):
    """A word at every offset around a chunk's end (512 bytes), with and without
    a rejecting byte (inside the window and outside it) before, in or behind it."""
    rng = np.random.default_rng(6)
    for pattern in ("[A-Z]*(ERROR|WARN)[A-Z]*", "[A-Z]*ERROR[A-Z]*|[A-Z]*WARN[A-Z]*", "[A-Z]*ERROR[A-Z]*WARN[A-Z]*",
                    "[A-Z]*ERROR([A-Z]*X)?", "[A-Z]*ERROR([A-Z][A-Z])*", "[A-Z]*ERR[A-Z]*OR[A-Z]*AR[A-Z]*",
                    "ERROR[A-Z]*|[A-Z]*WARN"):
        eng = NfaEngine.from_matrices(compile_nfa_matrices(pattern))
        size = 34_000
        places = list(range(512 - 70, 512 + 70, 3)) + list(range(16 * 512 - 8, 16 * 512 + 8)) + [size - 5]
        data, offsets = _strings(rng, np.full(len(places) * 4, size))
        for i, at in enumerate(places):
            for k, reject in enumerate((None, 0x5B, 0x20, 0x5F)):
                base = (4 * i + k) * size
                data[base + at:base + at + 5] = np.frombuffer(b"ERROR", np.uint8)
                data[base + size - 300:base + size - 296] = np.frombuffer(b"WARN", np.uint8)
                if reject is not None:
                    data[base + int(rng.choice([at - 40, at - 1, at + 5, at + 300, size // 2, size - 1]) % size)] = reject
        _run(eng, data, offsets, MixParams(form=form))


def _run_ms(eng, data, offsets, params):
    """Time of the second of two runs."""
    from trex_amd.device import DeviceBuffer, Event, Stream
    n = len(offsets) - 1
    m = MixEngine([eng])
    m.plan(offsets[:-1], offsets[1:], np.zeros(n, np.int32), params)
    stream = Stream()
    d = DeviceBuffer.from_array(data, stream)
    d_mask, d_acc = DeviceBuffer(8 * n), DeviceBuffer(n)
    a, b = Event(), Event()
    for event in (Event(), a):
        event.record(stream)
        m.run(d.ptr, d_mask.ptr, d_acc.ptr, stream)
    b.record(stream)
    stream.synchronize()
    assert m.error(stream) == 0
    return a.elapsed_ms(b)


@pytest.mark.parametrize("form", ["nibble", "slice"])
@pytest.mark.parametrize("params", [{}, {"nfa_split": 2048, "nfa_chunk": 1024}], ids=["open", "1 KiB"])
def test_sets_that_coincide_late(gpu_lib, params, form):
    """Walks from different sets coincide at a letter that comes every hundred
    bytes: the walk ahead of a chunk mostly does not reach one, the chunk mostly
    does. Walked again by one lane per string, chunk after chunk, 16 strings of
    1 MiB take 180 ms and more."""
    rng = np.random.default_rng(7)
    eng = NfaEngine.from_matrices(compile_nfa_matrices("(([A-Y][A-Y][A-Y])*([A-Y]|[A-Y][A-Y])?Z)*([A-Y][A-Y][A-Y])*"))
    params = MixParams(form=form, **params)
    data, offsets = _strings(rng, np.array([200_000, 0, 5000, 64, 40_001, 33_000]))
    data[data == ord("Z")] = ord("A")
    rare = data.copy()
    rare[rng.random(len(data)) < 0.002] = ord("Z")
    _run(eng, rare, offsets, params)
    data[rng.random(len(data)) < 0.01] = ord("Z")
    _run(eng, data, offsets, params)
    data, offsets = _strings(rng, np.full(16, 1 << 20))
    data[data == ord("Z")] = ord("A")
    data[rng.random(len(data)) < 0.01] = ord("Z")
    assert _run_ms(eng, data, offsets, params) < 40


@pytest.mark.parametrize("form", ["nibble", "slice"])
@pytest.mark.parametrize("n", [500, 700])
def test_fixups_by_wave_and_by_lane(gpu_lib, n, form):
    """Up to two fix-ups a CU a wave each, beyond them a lane each: guesses that
    are right, wrong to some letter, and always wrong, the empty set, and a
    string of more than 64 chunks."""
    rng = np.random.default_rng(n)
    for pattern in ("(([A-Y][A-Y][A-Y])*([A-Y]|[A-Y][A-Y])?Z)*([A-Y][A-Y][A-Y])*", "([A-Z][A-Z][A-Z])*",
                    "[A-Z]*ERROR[A-Z]*WARN[A-Z]*", "[A-Y]*(WARN)[A-Z]*"):
        eng = NfaEngine.from_matrices(compile_nfa_matrices(pattern))
        lengths = rng.integers(1100, 4000, n)
        lengths[5] = 200_000
        data, offsets = _strings(rng, lengths)
        data[data == ord("Z")] = ord("A")
        data[rng.random(len(data)) < 0.002] = ord("Z")
        for at in rng.integers(0, len(data) - 5, 400):
            data[at:at + 5] = np.frombuffer(rng.choice([b"ERROR", b"WARNE"]), np.uint8)
        _run(eng, data, offsets, MixParams(nfa_split=1024, nfa_chunk=1024, ck=64, form=form))
