"""NFA-64 dispatch against the C oracle: one, two and four lanes a string of
the slice kernels at the batch sizes where the rule changes, and automata that
reach few sets (matched as DFAs) around the limit of 256."""

import numpy as np
import pytest

from oracle import cpu as oracle_cpu
from trex_amd.engine import NfaEngine
from trex_amd.workloads import random_nfa64

pytestmark = pytest.mark.gpu


def _check(eng, data, offsets):
    mask, accept, _, _ = eng.match_arrays(data, offsets)
    want_mask, want_accept = oracle_cpu.nfa_walk(eng.succ, eng.byte_to_sym, eng.start, eng.accept, data, offsets)
    assert np.array_equal(mask, want_mask) and np.array_equal(accept, want_accept)
    return mask


def _batch(rng, n, most, lo=0x40, hi=0x60, stray=0.02):
    lengths = rng.integers(0, most, n)
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(lengths, out=offsets[1:])
    data = rng.integers(lo, hi, int(offsets[-1]), dtype=np.uint8)
    hits = rng.integers(0, max(len(data), 1), int(stray * n)) if len(data) else np.zeros(0, np.int64)
    data[hits] = rng.integers(0, 256, len(hits), dtype=np.uint8)
    return data, offsets + 3, np.concatenate([np.zeros(3, np.uint8), data])


@pytest.mark.parametrize("n", [1, 65, 16384, 16385, 40960, 40961, 70001])
def test_slice_kernels_by_batch_size(gpu_lib, n):
    """At most 64 strings a CU: four lanes a string; at most 160: two."""
    rng = np.random.default_rng(n)
    eng = NfaEngine.from_matrices(random_nfa64(rng))
    assert eng.info()["variant"] == "window6"
    _, offsets, data = _batch(rng, n, 90)
    _check(eng, data, offsets)


def _counter(k):
    """A cycle of k states on 'A', 'B' keeps the state, 'C' is skipped, all else rejects: k + 1 sets."""
    succ = np.zeros((2, 64), np.uint64)
    for s in range(k):
        succ[0, s] = np.uint64(1) << np.uint64((s + 1) % k)
        succ[1, s] = np.uint64(1) << np.uint64(s)
    b2s = np.full(256, -1, np.int16)
    b2s[ord("A")], b2s[ord("B")], b2s[ord("C")] = 0, 1, -2
    return NfaEngine(succ, b2s, 1, 1 << (k - 1))


def _window_bits(k):
    """The last k letters as a set ('A' starts a bit, every letter moves it): about 2^k sets."""
    succ = np.zeros((2, 64), np.uint64)
    for c in range(2):
        succ[c, 0] = np.uint64(1 | (2 if c == 0 else 0))
        for s in range(1, k):
            succ[c, s] = np.uint64(1) << np.uint64(s + 1)
    b2s = np.full(256, -1, np.int16)
    b2s[ord("A")], b2s[ord("B")] = 0, 1
    return NfaEngine(succ, b2s, 1, 1 << k)


@pytest.mark.parametrize("make", [lambda: _counter(5), lambda: _counter(9), lambda: _counter(14), lambda: _counter(63),
                                  lambda: _window_bits(3), lambda: _window_bits(6), lambda: _window_bits(7),
                                  lambda: _window_bits(8)],
                         ids=["6sets", "10sets", "15sets", "64sets", "9sets", "65sets", "129sets", "over"])
def test_automata_of_few_sets(gpu_lib, make):
    rng = np.random.default_rng(1)
    eng = make()
    _, offsets, data = _batch(rng, 3000, 200, ord("A"), ord("D"), stray=0.1)
    got = _check(eng, data, offsets)
    eng.set_variant("window6")   # the bit-parallel kernels give the same sets
    assert np.array_equal(_check(eng, data, offsets), got)


@pytest.mark.parametrize("pattern,found", [("[A-Z]*(ERROR|WARN)[A-Z]*", False), ("[A-Z]*(ERROR|WARN)[A-Z]*", True),
                                           ("[A-Z]*A[A-Z][A-Z][A-Z][A-Z][A-Z]", True), ("([A-Z][A-Z][A-Z])*", True)],
                         ids=["not found", "found", "last letters", "length"])
def test_long_strings_in_short_chunks(gpu_lib, pattern, found):
    """Few long strings are cut into chunks far below the given lengths; their
    guesses hold always, until a word is found, or never."""
    from trex_amd.mix import MixParams
    from trex_amd.nfa_matrices import compile_nfa_matrices
    rng = np.random.default_rng(8)
    eng = NfaEngine.from_matrices(compile_nfa_matrices(pattern))
    lengths = np.array([300_000, 0, 5, 33_000, 70_001, 512, 513])
    offsets = np.zeros(len(lengths) + 1, np.int64)
    np.cumsum(lengths, out=offsets[1:])
    data = rng.choice(np.frombuffer(b"BCDFGHIJKLMPQSTUVXYZA", np.uint8), int(offsets[-1]))
    if found:
        for at in (150_003, 310_000):
            data[at:at + 5] = np.frombuffer(b"ERROR", np.uint8)
    want, _ = oracle_cpu.nfa_walk(eng.succ, eng.byte_to_sym, eng.start, eng.accept, data, offsets)
    for params in (MixParams(), MixParams(form="slice"), MixParams(nfa_split=1 << 14, nfa_chunk=1 << 13, ck=256)):
        mask, _, _, _ = eng.match_split(data, offsets, params)
        assert np.array_equal(mask, want)
