"""Slice kernels of the NFA at the batch sizes where the lanes a string change
(96 and 256 strings a compute unit), against the C oracle."""

import numpy as np
import pytest

from oracle import cpu as oracle_cpu
from trex_amd.engine import NfaEngine
from trex_amd.workloads import random_nfa64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cu,more", [(96, 0), (96, 1), (256, 0), (256, 1)])
def test_lanes_by_batch_size(gpu_lib, per_cu, more):
    from trex_amd._lib import device_info
    n = per_cu * device_info()["cus"] + more
    rng = np.random.default_rng(n)
    eng = NfaEngine.from_matrices(random_nfa64(rng))
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(rng.integers(0, 90, n), out=offsets[1:])
    data = rng.integers(0x40, 0x60, int(offsets[-1]) + 1, dtype=np.uint8)
    data[rng.integers(0, len(data), n // 50)] = rng.integers(0, 256, n // 50, dtype=np.uint8)
    mask, accept, _, _ = eng.match_arrays(data, offsets)
    want_mask, want_accept = oracle_cpu.nfa_walk(eng.succ, eng.byte_to_sym, eng.start, eng.accept, data, offsets)
    assert np.array_equal(mask, want_mask) and np.array_equal(accept, want_accept)
