"""Pinned staging of host dispatches, shared by all handles of the process."""

from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from oracle import cpu as ocpu
from trex_amd import _lib
from trex_amd.engine import DfaEngine
from trex_amd.regex_to_dfa import compile_regex
from trex_amd.tables import dfa_byte_table

pytestmark = pytest.mark.gpu
BLOCK = 640 << 10


def _held():
    v = ctypes.c_int64()
    _lib.call("trex_dfa_staging_bytes", ctypes.byref(v))
    return v.value


def _match(engine, rng, n=48, size=100):
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(rng.integers(0, size, n), out=offsets[1:])
    data = rng.choice(np.frombuffer(b"warneo r", np.uint8), int(offsets[-1]))
    final, accept, _, _ = engine.match_arrays(data, offsets)
    t = engine.table
    want = ocpu.dfa_walk(t.delta, t.accept, t.start, data, offsets)
    return np.array_equal(final, want[0]) and np.array_equal(accept, want[1])


def test_resident_patterns_share_one_block(gpu_lib):
    """64 resident patterns, matched one after another; first calls make no block."""
    rng = np.random.default_rng(1)
    tab = dfa_byte_table(compile_regex(".*(warn|error).*"))
    engines = [DfaEngine(tab) for _ in range(64)]
    before = _held()
    assert all(_match(e, rng) for e in engines) and _held() == before
    for _ in range(3):
        assert all(_match(e, rng) for e in engines)
    assert _held() <= max(before, BLOCK)
    for e in engines:
        e.close()
    assert _match(DfaEngine(tab), rng)


def test_threads_with_engines_of_their_own(gpu_lib):
    """More threads than there may be blocks, small and large requests; engines come and go."""
    tab = dfa_byte_table(compile_regex(".*(warn|error).*"))
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for _ in range(4):
            engine = DfaEngine(tab)
            for _ in range(6):
                if not _match(engine, rng, int(rng.integers(1, 3000)), int(rng.integers(1, 400))):
                    bad.append(seed)
            engine.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(20)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    assert _held() <= 16 * BLOCK
