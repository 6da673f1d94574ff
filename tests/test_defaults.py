"""A handle's own choice of kernel: restored after a setting, and among the
candidates of the tuners."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _time(fn, stream, reps=20):
    from trex_amd.device import Event
    fn()
    a, b = Event(), Event()
    a.record(stream)
    for _ in range(reps):
        fn()
    b.record(stream)
    stream.synchronize()
    return a.elapsed_ms(b) / reps


def test_nfa_default_is_restored(gpu_lib):
    """Words over an automaton of few sets: 28 us as a DFA, 300 us and more bit-parallel."""
    from trex_amd.device import DeviceBuffer, Stream
    from trex_amd.engine import DeviceBatch, NfaEngine
    from trex_amd.nfa_matrices import compile_nfa_matrices
    rng = np.random.default_rng(1)
    eng = NfaEngine.from_matrices(compile_nfa_matrices("[a-z0-9 ]*(error|warning|fail) [a-z0-9 ]*"))
    n = 30_000
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(rng.integers(300, 1000, n), out=offsets[1:])
    data = rng.choice(np.frombuffer(b"abcdefghil ", np.uint8), int(offsets[-1]))
    stream = Stream()
    batch = DeviceBatch(data, offsets, "csr")
    d_mask, d_acc = DeviceBuffer(8 * n), DeviceBuffer(n)
    run = lambda: eng.match_batch_device(batch, d_mask.ptr, d_acc.ptr, stream)
    default = eng.info()["variant"]
    own = _time(run, stream)
    want = d_mask.download(np.uint64, n, stream)
    eng.set_variant("bytes")
    forced = _time(run, stream)
    assert np.array_equal(d_mask.download(np.uint64, n, stream), want)
    eng.set_variant("auto")
    assert eng.info()["variant"] == default
    again = _time(run, stream)
    assert np.array_equal(d_mask.download(np.uint64, n, stream), want)
    assert own < forced / 2 and again < forced / 2


def test_pnfa_default_is_restored(gpu_lib):
    """100 sequences: workgroups of one sequence beat two of 64, whatever the box."""
    from trex_amd.device import DeviceBuffer, Stream
    from trex_amd.engine import ProbNfaEngine
    from trex_amd.workloads import dirichlet_pnfa
    rng = np.random.default_rng(2)
    T, start, accept = dirichlet_pnfa(rng)
    eng = ProbNfaEngine(T, start, accept)
    n, length = 100, 500
    stream = Stream()
    d = DeviceBuffer.from_array(rng.integers(0, T.shape[0], n * length, dtype=np.uint8), stream)
    d_ll, d_lm = DeviceBuffer(8 * n), DeviceBuffer(8 * n)
    run = lambda: eng.loglik_device(d.ptr, n, length, d_ll.ptr, d_lm.ptr, stream)
    own = _time(run, stream, 5)
    want = d_ll.download(np.float64, n, stream)
    eng.set_waves(8)
    forced = _time(run, stream, 5)
    eng.set_waves(0)
    assert eng.info()["waves"] == 8
    again = _time(run, stream, 5)
    assert np.array_equal(d_ll.download(np.float64, n, stream), want)
    assert own < 0.8 * forced and again < 0.8 * forced


def test_tuners_know_the_engines_own_choice(gpu_lib, tmp_path, monkeypatch):
    """Lines of unequal lengths (half the time of any variant) and 100 sequences."""
    from trex_amd.autotune import tune_dfa, tune_pnfa
    from trex_amd.device import DeviceBuffer, Stream
    from trex_amd.engine import DeviceBatch, DfaEngine, ProbNfaEngine
    from trex_amd.regex_to_dfa import compile_regex
    from trex_amd.tables import dfa_byte_table
    from trex_amd.workloads import dirichlet_pnfa
    monkeypatch.setenv("TREX_AMD_TUNE_CACHE", str(tmp_path / "tune.json"))
    rng = np.random.default_rng(3)
    stream = Stream()
    n = 100_000
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(rng.integers(20, 400, n), out=offsets[1:])
    batch = DeviceBatch(rng.integers(32, 127, int(offsets[-1]), dtype=np.uint8), offsets, "csr")
    d_out = [DeviceBuffer(n) for _ in range(2)]
    table = dfa_byte_table(compile_regex(".*(error|warn).*"))
    for source in ("tuned", "cache"):
        eng = DfaEngine(table)
        choice = tune_dfa(eng, batch, d_out[0].ptr, d_out[1].ptr, stream)
        assert (choice["source"], choice["variant"], choice["prefetch"]) == (source, "auto", 8)
    T, start, accept = dirichlet_pnfa(rng)
    n, length = 100, 500
    d = DeviceBuffer.from_array(rng.integers(0, T.shape[0], n * length, dtype=np.uint8), stream)
    d_ll = [DeviceBuffer(8 * n) for _ in range(2)]
    choice = tune_pnfa(ProbNfaEngine(T, start, accept), d.ptr, n, length, d_ll[0].ptr, d_ll[1].ptr, stream)
    assert choice["waves"] == 0


def test_rotation_is_reported_as_launched(gpu_lib):
    """A search table synchronises, but its functions stay apart until the text is
    found, so its launches are not rotated unless a variant or a mode asks for it."""
    from trex_amd.engine import DfaEngine
    from trex_amd.regex_to_dfa import compile_regex
    from trex_amd.tables import dfa_byte_table
    search = DfaEngine(dfa_byte_table(compile_regex("[A-Z]*(ERROR|WARN|FAIL)[A-Z]*")))
    recent = DfaEngine(dfa_byte_table(compile_regex("(A|B|C|D)*(A|B)(C|D)")))
    only = DfaEngine(dfa_byte_table(compile_regex("[@-_]*")))   # one live state: every function is its constant
    assert search.rotation() == (False, True) and recent.rotation() == (True, True) and only.rotation() == (True, True)
    search.set_variant("k2_window_f")
    assert search.rotation() == (True, True)
    search.set_variant("auto")
    assert search.rotation() == (False, True)
    search.set_rotation(1)
    assert search.rotation() == (True, True)


def test_multi_pattern_group_outlives_the_form(gpu_lib):
    """A group of one is eight launches, also after the form went back to the
    default; without a group the default form takes all patterns in one."""
    from trex_amd.device import DeviceBuffer, Stream
    from trex_amd import _lib
    from trex_amd.engine import DeviceBatch, DfaEngine, DfaMultiEngine
    from trex_amd.regex_to_dfa import compile_regex
    from trex_amd.tables import dfa_byte_table
    rng = np.random.default_rng(4)
    words = ["ERROR", "TIMEOUT", "LOGIN", "LOGOUT", "REFUSED", "DENIED", "CLOSED", "BROKEN"]
    engines = [DfaEngine(dfa_byte_table(compile_regex(f"[A-Z]*{w}[A-Z]*"))) for w in words]
    multi = DfaMultiEngine(engines)
    n = 50_000
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(rng.integers(300, 600, n), out=offsets[1:])
    data = rng.integers(0x41, 0x5B, int(offsets[-1]), dtype=np.uint8)
    stream = Stream()
    batch = DeviceBatch(data, offsets, "csr")
    d_out = [DeviceBuffer(len(words) * n) for _ in range(2)]
    run = lambda: multi.match_batch_device(batch, d_out[0].ptr, d_out[1].ptr, stream)
    together = _time(run, stream)
    want = d_out[0].download(np.uint8, len(words) * n, stream)
    multi.set_group(1)
    apart = _time(run, stream)
    _lib.call("trex_dfa_multi_set_form", multi.handle, 0)
    assert _time(run, stream) > 0.6 * apart > 0.9 * together
    assert np.array_equal(d_out[0].download(np.uint8, len(words) * n, stream), want)
