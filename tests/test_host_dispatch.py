"""Host dispatch of the DFA engine (``trex_dfa_match_host``) at the edges of its
pinned staging: 512 KiB of offsets and bytes, 128 KiB of results."""

from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest

from oracle import cpu as ocpu
from trex_amd.regex_to_dfa import compile_regex
from trex_amd.tables import dfa_byte_table

pytestmark = pytest.mark.gpu
STAGED = 512 << 10


def _call(engine, data, offsets):
    from trex_amd import _lib
    n = len(offsets) - 1
    final, acc = np.full(n, 99, np.uint8), np.full(n, 99, np.uint8)
    ms = ctypes.c_float(), ctypes.c_float()
    _lib.call("trex_dfa_match_host", engine.handle, data.ctypes.data, offsets.ctypes.data_as(_lib.i64p), n,
              final.ctypes.data_as(_lib.u8p), acc.ctypes.data_as(_lib.u8p), ctypes.byref(ms[0]), ctypes.byref(ms[1]))
    assert 0 <= ms[0].value <= ms[1].value
    return final, acc


def _batch(rng, n, total, base):
    cuts = np.sort(rng.integers(0, total + 1, n - 1)) if n > 1 else np.zeros(0, np.int64)
    offsets = base + np.concatenate([[0], cuts, [total]]).astype(np.int64)
    data = rng.choice(np.frombuffer(b"warneo r", np.uint8), base + total + 1)
    return np.ascontiguousarray(data), offsets


@pytest.mark.parametrize("n,spare", [(1, 0), (1, -1), (1, 1), (48, 0), (48, 1), (48, -17), (48, 1 << 20),
                                     (65000, 0), (65000, 1), (65535, 0), (65535, 5), (65536, 100), (70000, 1000)])
def test_staging_edges(gpu_lib, n, spare):
    """Inputs that just fit the staging, are a byte over or far over it, results
    that fit and that do not, a first offset that is not 0; a small call
    follows on the same engine."""
    from trex_amd.engine import DfaEngine
    rng = np.random.default_rng(n + spare)
    tab = dfa_byte_table(compile_regex(".*(warn|error).*"))
    engine = DfaEngine(tab)
    room = max(STAGED - (8 * (n + 1) + 255) // 256 * 256, 0)
    for count, total, base in ((n, room + spare, 0), (n, max(room + spare, 0), 13), (3, 40, 5)):
        data, offsets = _batch(rng, count, max(total, 0), base)
        final, acc = _call(engine, data, offsets)
        rf, ra = ocpu.dfa_walk(tab.delta, tab.accept, tab.start, data[base:], offsets - base)
        assert np.array_equal(final, rf) and np.array_equal(acc, ra)


def test_threads_share_an_engine(gpu_lib):
    """Calls of several threads on one engine get their own results."""
    from trex_amd.engine import DfaEngine
    tab = dfa_byte_table(compile_regex(".*(warn|error).*"))
    engine = DfaEngine(tab)
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        for _ in range(20):
            data, offsets = _batch(rng, int(rng.integers(1, 300)), int(rng.integers(0, 5000)), 0)
            final, acc = _call(engine, data, offsets)
            rf, ra = ocpu.dfa_walk(tab.delta, tab.accept, tab.start, data, offsets)
            if not (np.array_equal(final, rf) and np.array_equal(acc, ra)):
                bad.append(seed)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
