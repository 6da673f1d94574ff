"""Byte-class DFA kernels (contiguous strings) against the C oracle, at the
edges of their forms: states per function word, classes, vector boundaries and
alignments, workgroup sizes and the ordering by length."""

import numpy as np
import pytest

from oracle import cpu as oracle_cpu
from trex_amd import _lib
from trex_amd.device import DeviceBuffer
from trex_amd.engine import DfaEngine
from trex_amd.regex_to_dfa import compile_regex
from trex_amd.tables import DfaByteTable, dfa_byte_table

pytestmark = pytest.mark.gpu


def _table(rng, n_states, n_classes):
    """A random table whose bytes fall into n_classes distinct columns (as far as n_states allows)."""
    columns = rng.integers(0, n_states, size=(n_classes, n_states), dtype=np.uint8)
    cls = np.concatenate([np.arange(n_classes), rng.integers(0, n_classes, 256 - n_classes)])
    delta = columns[rng.permutation(cls)].T
    return DfaByteTable(delta, rng.integers(0, 2, n_states, dtype=np.uint8), int(rng.integers(n_states)), -1, n_states)


def _check(table, data, begin, end):
    eng = DfaEngine(table)
    n = len(begin)
    d, b, e = DeviceBuffer.from_array(data), DeviceBuffer.from_array(begin), DeviceBuffer.from_array(end)
    outs = [DeviceBuffer.from_array(np.full(n, 255, np.uint8)) for _ in range(2)]
    _lib.call("trex_dfa_match_ranges", eng.handle, d.ptr, b.ptr, e.ptr, n, outs[0].ptr, outs[1].ptr, None)
    final, accept = outs[0].download(np.uint8, n), outs[1].download(np.uint8, n)
    # the oracle takes packed strings
    offsets = np.zeros(len(begin) + 1, np.int64)
    np.cumsum(end - begin, out=offsets[1:])
    packed = np.concatenate([data[x:y] for x, y in zip(begin, end)]) if offsets[-1] else np.zeros(0, np.uint8)
    want_final, want_accept = oracle_cpu.dfa_walk(table.delta, table.accept, table.start, packed, offsets)
    assert np.array_equal(final, want_final)
    assert np.array_equal(accept, want_accept)


@pytest.mark.parametrize("n_states,n_classes", [(1, 1), (2, 3), (10, 31), (11, 5), (15, 31), (16, 31), (16, 32), (17, 6),
                                                (31, 32), (64, 40), (200, 12), (256, 200)])
def test_class_kernels_match_oracle(gpu_lib, n_states, n_classes):
    """Every length 0 .. 80 from every offset modulo 16, and lengths around the
    long strings' block boundaries, overlapping ranges of one buffer."""
    rng = np.random.default_rng(100 * n_states + n_classes)
    table = _table(rng, n_states, n_classes)
    data = rng.integers(0, 256, 9000, dtype=np.uint8)
    begin, end = [], []
    for shift in range(16):
        for length in list(range(81)) + [127, 128, 129, 1023, 1024, 1040, 1087, 2048, 4095, 8000]:
            begin.append(shift + int(rng.integers(0, 3)) * 16)
            end.append(begin[-1] + length)
    _check(table, data, np.array(begin, np.int64), np.array(end, np.int64))


@pytest.mark.parametrize("n_strings", [1, 63, 65, 65535, 65536, 65537, 131075])
@pytest.mark.parametrize("n_states", [9, 13, 40])
def test_class_kernels_launch_shapes(gpu_lib, n_strings, n_states):
    """One-wave and 256-thread workgroups, full and partial, with lengths that
    are ordered (0 .. 300 bytes) in some workgroups and equal in others."""
    rng = np.random.default_rng(n_strings + n_states)
    table = _table(rng, n_states, 7)
    lengths = rng.integers(0, 300, n_strings)
    lengths[: n_strings // 3] = 40
    offsets = np.zeros(n_strings + 1, np.int64)
    np.cumsum(lengths, out=offsets[1:])
    data = rng.integers(0, 256, int(offsets[-1]) + 1, dtype=np.uint8)
    _check(table, data, offsets[:-1].copy(), offsets[1:].copy())


def test_alike_strings_take_the_rotated_order(gpu_lib):
    """131,072 strings and a table that synchronises: workgroups of 4 KiB
    strings on one offset modulo 4 KiB beside workgroups of other strings."""
    rng = np.random.default_rng(3)
    table = dfa_byte_table(compile_regex("(A|B|C|D)*(A|B)(C|D)"))
    n, n_alike = 131072, 700
    data = rng.choice(np.frombuffer(b"ABCD", np.uint8), 4096 * n_alike + 5000)
    begin = np.arange(n, dtype=np.int64) % n_alike * 4096
    end = begin + 4096
    other = np.arange(n) >= 1024
    begin[other] = rng.integers(0, 4096 * n_alike, int(other.sum()))
    end[other] = begin[other] + rng.integers(0, 120, int(other.sum()))
    begin[600] += 3   # one string keeps its workgroup from being alike
    data[4096 * 5 + 77] = 0x20
    _check(table, data, begin, end)


def _ranges_ms(eng, data, begin, end):
    from trex_amd.device import Event, Stream
    n = len(begin)
    stream = Stream()
    d, b, e = (DeviceBuffer.from_array(x, stream) for x in (data, begin, end))
    outs = [DeviceBuffer(n) for _ in range(2)]
    marks = Event(), Event()
    for reps, mark in ((3, marks[0]), (20, marks[1])):
        for _ in range(reps):
            _lib.call("trex_dfa_match_ranges", eng.handle, d.ptr, b.ptr, e.ptr, n, outs[0].ptr, outs[1].ptr, stream.handle)
        mark.record(stream)
    stream.synchronize()
    return marks[0].elapsed_ms(marks[1]) / 20


@pytest.mark.parametrize("n_states,n_classes,n", [(200, 200, 60000), (256, 250, 33000), (256, 250, 60000)])
def test_large_tables_take_whole_workgroups(gpu_lib, n_states, n_classes, n):
    """Batches whose waves would not all find LDS for a table of their own: as
    long as the next larger batch at most (twice as long by waves)."""
    rng = np.random.default_rng(n)
    table = _table(rng, n_states, n_classes)
    lengths = rng.integers(1000, 2000, 65536)
    offsets = np.zeros(65537, np.int64)
    np.cumsum(lengths, out=offsets[1:])
    data = rng.integers(0, 256, int(offsets[-1]) + 1, dtype=np.uint8)
    eng = DfaEngine(table)
    few = _ranges_ms(eng, data, offsets[:n].copy(), offsets[1:n + 1].copy())
    assert few < 1.3 * _ranges_ms(eng, data, offsets[:-1].copy(), offsets[1:].copy())
    _check(table, data, offsets[:n:37].copy(), offsets[1:n + 1:37].copy())


@pytest.mark.parametrize("n_states,n_classes", [(17, 40), (100, 100), (256, 250)])
def test_tables_without_pairs_are_no_slower_by_rows(gpu_lib, n_states, n_classes):
    """100,000 strings of 1 to 2 KB: the rows' kernel against the generic one
    (rows by class: 1.28 times its time)."""
    rng = np.random.default_rng(n_states)
    table = _table(rng, n_states, n_classes)
    offsets = np.zeros(100_001, np.int64)
    np.cumsum(rng.integers(1000, 2000, 100_000), out=offsets[1:])
    data = rng.integers(0, 256, int(offsets[-1]) + 1, dtype=np.uint8)
    eng = DfaEngine(table)
    rows = _ranges_ms(eng, data, offsets[:-1].copy(), offsets[1:].copy())
    eng.set_variant("k1_generic")
    assert rows < 1.12 * _ranges_ms(eng, data, offsets[:-1].copy(), offsets[1:].copy())
