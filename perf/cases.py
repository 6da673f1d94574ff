"""Timed cases: what a program that uses this package asks of it, by its public
entry points, over the sizes such programs have.

A case is a dict of plain values; ``kind`` names the entry point:

* ``api``    ``OptimizedEngine.match`` / ``match_arrays`` on host data, whole
             call (packing, copies, kernel, results on the host);
* ``dfa``    ``DfaEngine`` over a batch resident in HBM (packed CSR or
             interleaved rows);
* ``multi``  ``DfaMultiEngine``: several patterns in one pass;
* ``long``   ``DfaEngine.match_plan``: few long texts cut into chunks;
* ``nfa``    ``NfaEngine`` (bit-parallel Boolean NFA of up to 64 states);
* ``prob``   ``ProbNfaEngine``: log-likelihoods, equal or ragged lengths;
* ``mix``    ``MixEngine``: many patterns, strings of any length, one queue.

``prepare`` makes what the program has in hand: the compiled patterns, the
batch in device memory (host memory for ``api``) and the output buffers.
"""

import ctypes
import math

import numpy as np
import torch

from trex_amd.engine import (ChunkPlan, DeviceBatch, DfaEngine, DfaMultiEngine, NfaEngine, ProbNfaEngine,
                             lookback_chunk_len, lookback_target_chunks)
from trex_amd.mix import MixEngine
from trex_amd.nfa_matrices import compile_nfa_matrices
from trex_amd.optimized_engine import OptimizedEngine
from trex_amd.regex_to_dfa import compile_regex
from trex_amd.tables import dfa_byte_table
from trex_amd.workloads import ALPHABET_32, dirichlet_pnfa, random_nfa64

# Alphabets of the texts: one aligned 32-byte window, and log lines.
UPPER = "ABCDEFGHIJKLMNOPQRSTUVWXYZ"
LINE = "etaoinshrdlucmfwypvbgkqjxz" * 3 + "etaoinshrd" * 4 + " " * 22 + "0123456789" * 2 + ".:/=-_[]()"
WORDS = "etaoinshrdlucmfwypvbgkqjxz" * 3 + " " * 14 + "0123456789"

PATTERNS = {
    # at most 16 states over one window
    "upper_search": "[A-Z]*(ERROR|WARN|FAIL)[A-Z]*",
    "upper_recent": "[A-Z]*[AEIOU][A-Z][A-Z]",          # what the last three characters were
    "upper_even": "([A-Z][A-Z])*",                      # never synchronises: parity of the length
    "upper_mod3": "([^A]*A[^A]*A[^A]*A)*[^A]*".replace("[^A]", "[B-Z]"),   # count modulo 3
    # at most 16 states over printable text
    "line_search": ".*(error|warn).*",
    "line_recent": ".*[aeiou]..",
    "line_time": ".*[0-9][0-9]:[0-9][0-9].*",
    "line_field": "[a-z ]*[0-9]+(ms|us)?[ -~]*",
    # more than 16 states
    "line_levels": ".*(error|warning|failure|timeout|refused).*",
    "line_request": ".*(get|post|put) /[a-z0-9/]*(=[a-z0-9]*)? (done|failed).*",
    # Boolean NFAs of printable words
    "words_levels": "[a-z0-9 ]*(error|warning|fail) [a-z0-9 ]*",
    "words_tail": "([a-z0-9 ]*e)?[a-z0-9][a-z0-9 ][a-z0-9 ][a-z0-9 ][a-z0-9 ]t[a-z0-9 ]*",
}

# rules of at most 16 states, matched several in one pass
RULES = ["[A-Z]*ERROR[A-Z]*", "[A-Z]*(WARN|FAIL)[A-Z]*", "[A-Z]*QU[A-Z]*", "([A-Z][A-Z])*", "[A-Z]*TIMEOUT[A-Z]*",
         "[A-Z]*X", "[B-Z]*(A[B-Z]*A[B-Z]*)*", "[A-Z]*(LOGIN|LOGOUT)[A-Z]*"]

DEVICE = "cuda"


def listed():
    return [
        # one interactive request: a handful of short strings, the whole call
        {"name": "small_request", "kind": "api", "pattern": "line_search", "n": 48, "lo": 8, "hi": 120, "texts": True},
        # the host batch of the benchmark's `host` leg: 10,000 x about 1,000 characters
        {"name": "host_batch", "kind": "api", "pattern": "upper_search", "n": 10000, "lo": 600, "hi": 1500, "texts": False},
        # the headline layout: equal strings as interleaved rows, one pattern
        {"name": "rows", "kind": "dfa", "pattern": "upper_search", "layout": "interleaved", "n": 65536, "lo": 4096, "hi": 4096},
        # a day's log lines in HBM, packed, printable text, at most 16 states
        {"name": "lines", "kind": "dfa", "pattern": "line_search", "layout": "csr", "n": 400000, "lo": 20, "hi": 400},
        # the same kind of lines and an ordinary larger DFA (17 .. 64 states)
        {"name": "lines_wide", "kind": "dfa", "pattern": "line_levels", "layout": "csr", "n": 100000, "lo": 40, "hi": 1000},
        # a rule set over one batch: eight patterns in one pass
        {"name": "rule_set", "kind": "multi", "patterns": 8, "n": 50000, "lo": 200, "hi": 3000},
        # a few long documents, split in chunks
        {"name": "long_text", "kind": "long", "pattern": "upper_recent", "n": 6, "lo": 20_000_000, "hi": 40_000_000},
        # the NFA-64 workload of the benchmark at an ordinary batch
        {"name": "nfa_dense", "kind": "nfa", "source": "random", "n": 40000, "lo": 2048, "hi": 2048},
        # a regex run as an NFA over lines of words
        {"name": "nfa_lines", "kind": "nfa", "source": "words_levels", "n": 100000, "lo": 40, "hi": 1000},
        # the probabilistic workload of the benchmark: 16,384 sequences of 2,048 symbols
        {"name": "prob_batch", "kind": "prob", "n": 16384, "lo": 2048, "hi": 2048, "ragged": False},
        # a served request of sequences of unequal lengths
        {"name": "prob_request", "kind": "prob", "n": 600, "lo": 64, "hi": 1024, "ragged": True},
        # mixed traffic: 16 patterns (DFA and NFA), strings of 32 bytes to 1 MiB in one queue
        {"name": "mixed_queue", "kind": "mix", "patterns": 16, "n": 1024, "lo": 32, "hi": 1 << 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["api", "dfa", "dfa", "dfa", "multi", "long", "nfa", "nfa", "prob", "prob", "mix"])
    if kind == "api":
        n, lo = _log(rng, 1, 20000), _log(rng, 8, 800)
        return {"kind": kind, "pattern": rng.choice(["line_search", "line_time", "upper_search", "line_levels"]), "n": n,
                "lo": lo, "hi": lo + _log(rng, 1, 1000), "texts": n <= 2000}
    if kind == "dfa":
        layout = rng.choice(["csr", "csr", "interleaved"])
        pattern = rng.choice(["upper_search", "upper_mod3", "line_search", "line_time", "line_field", "line_levels",
                              "line_request"])
        lo = _log(rng, 8, 3000)
        hi = lo + rng.choice([0, _log(rng, 8, 3000)])
        most = 200_000_000 // hi if layout == "csr" else 60_000_000 // hi
        n = _log(rng, 1000, min(most, 1_000_000 if layout == "csr" else 30_000))
        return {"kind": kind, "pattern": pattern, "layout": layout, "n": n, "lo": lo, "hi": hi}
    if kind == "multi":
        lo = _log(rng, 50, 2000)
        return {"kind": kind, "patterns": rng.randint(2, 8), "n": _log(rng, 2000, 60000), "lo": lo,
                "hi": lo + _log(rng, 8, 2000)}
    if kind == "long":
        total = _log(rng, 4_000_000, 200_000_000)
        n = _log(rng, 2, 40)
        mean = total // n
        return {"kind": kind, "pattern": rng.choice(["upper_recent", "upper_even", "upper_mod3", "line_recent"]), "n": n,
                "lo": max(1, mean // 2), "hi": mean + mean // 2}
    if kind == "nfa":
        lo = _log(rng, 32, 2000)
        hi = lo + rng.choice([0, _log(rng, 8, 1000)])
        return {"kind": kind, "source": rng.choice(["random", "words_levels", "words_tail"]),
                "n": _log(rng, 2000, min(300_000, 100_000_000 // hi)), "lo": lo, "hi": hi}
    if kind == "prob":
        lo = _log(rng, 16, 2000)
        ragged = rng.random() < 0.5
        hi = lo + _log(rng, 8, 500) if ragged else lo
        return {"kind": kind, "n": _log(rng, 32, min(16384, 30_000_000 // hi)), "lo": lo, "hi": hi, "ragged": ragged}
    return {"kind": "mix", "patterns": rng.randint(2, 24), "n": _log(rng, 200, 4000), "lo": rng.randint(16, 64),
            "hi": _log(rng, 4000, 400_000)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _text(seed, alphabet, total):
    """``total`` characters drawn from ``alphabet`` (its repetitions are weights), uint8 on the GPU."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    pool = torch.from_numpy(np.frombuffer(alphabet.encode(), np.uint8).copy()).to(DEVICE)
    return pool[torch.randint(0, len(alphabet), (total,), generator=g, device=DEVICE)]


def _offsets(case, seed):
    """Offsets of ``n`` strings with lengths log-uniform in [lo, hi]."""
    rng = np.random.default_rng(seed)
    n, lo, hi = case["n"], case["lo"], case["hi"]
    lengths = np.full(n, lo) if lo == hi else np.exp(rng.uniform(np.log(lo), np.log(hi + 1), n)).astype(np.int64)
    offsets = np.zeros(n + 1, np.int64)
    np.cumsum(np.clip(lengths, lo, hi), out=offsets[1:])
    return offsets


def _plant(data, offsets, seed, words, share=0.1):
    """Writes a word into about ``share`` of the strings (searches find something)."""
    rng = np.random.default_rng(seed + 1)
    n = len(offsets) - 1
    for w in words:
        w = torch.from_numpy(np.frombuffer(w.encode(), np.uint8).copy()).to(data.device)
        pick = rng.choice(n, max(1, int(n * share / len(words))))
        room = offsets[pick + 1] - offsets[pick] - len(w)
        pick, room = pick[room > 0], room[room > 0]
        at = torch.from_numpy(offsets[pick] + (rng.random(len(pick)) * room).astype(np.int64)).to(data.device)
        for k in range(len(w)):
            data[at + k] = w[k]
    return data


def _strings(case, seed):
    """(bytes on the GPU, offsets on the host) of a pattern's kind of text."""
    name = case["pattern"]
    offsets = _offsets(case, seed)
    data = _text(seed, UPPER if name.startswith("upper") else LINE, int(offsets[-1]))
    words = ["ERROR", "FAIL"] if name.startswith("upper") else ["error", "timeout", "12:30", "get /ab failed", "17ms"]
    return _plant(data, offsets, seed, words), offsets


def _table(name):
    return dfa_byte_table(compile_regex(PATTERNS[name]))


def _bytes_out(n, size=1):
    return torch.zeros(n, dtype={1: torch.uint8, 8: torch.int64}[size], device=DEVICE)


def _rule_set(count):
    return [DfaEngine(dfa_byte_table(compile_regex(RULES[i % len(RULES)]))) for i in range(count)]


_used = set()


def _first_use(state):
    """Runs a case of each form once in a process. The first launch of a kernel looks its name up in
    every code object, and the runtime keeps the "not found" of the others as the thread's last error,
    which torch would report at its next launch: read it here, as a program that mixes the two does."""
    key = tuple((k, v) for k, v in sorted(state["case"].items()) if k not in ("name", "n", "lo", "hi"))
    if key not in _used:
        _used.add(key)
        run(state)
        torch.cuda.synchronize()
        ctypes.CDLL("libamdhip64.so.7").hipGetLastError()
    return state


def prepare(case, seed):
    kind = case["kind"]
    if kind == "api":
        data, offsets = _strings(case, seed)
        data = data.cpu().numpy()
        state = {"engine": OptimizedEngine(PATTERNS[case["pattern"]]), "data": data, "offsets": offsets}
        if case["texts"]:
            text = data.tobytes().decode("latin-1")
            state["strings"] = [text[a:b] for a, b in zip(offsets[:-1], offsets[1:])]
    elif kind == "dfa":
        data, offsets = _strings(case, seed)
        state = {"engine": DfaEngine(_table(case["pattern"])), "final": _bytes_out(case["n"]),
                 "accept": _bytes_out(case["n"])}
        if case["layout"] == "csr":
            state["bytes"] = data
            state["offsets"] = torch.from_numpy(offsets).to(DEVICE)
        else:
            state["batch"] = DeviceBatch(data.cpu().numpy(), offsets, layout="interleaved")
    elif kind == "multi":
        offsets = _offsets(case, seed)
        data = _plant(_text(seed, UPPER, int(offsets[-1])), offsets, seed, ["ERROR", "FAIL", "LOGIN", "TIMEOUT"])
        patterns = _rule_set(case["patterns"])
        size = case["patterns"] * case["n"]
        state = {"patterns": patterns, "engine": DfaMultiEngine(patterns), "final": _bytes_out(size),
                 "accept": _bytes_out(size), "batch": DeviceBatch(data.cpu().numpy(), offsets, layout="csr")}
    elif kind == "long":
        data, offsets = _strings(case, seed)
        table = _table(case["pattern"])
        length = lookback_chunk_len(int(offsets[-1]), lookback_target_chunks(table))
        state = {"engine": DfaEngine(table), "bytes": data, "plan": ChunkPlan(offsets[:-1], offsets[1:], length),
                 "final": _bytes_out(case["n"]), "accept": _bytes_out(case["n"])}
    elif kind == "nfa":
        offsets = _offsets(case, seed)
        if case["source"] == "random":
            engine = NfaEngine.from_matrices(random_nfa64(np.random.default_rng(5)))
            data = _text(seed, ALPHABET_32, int(offsets[-1]))
        else:
            engine = NfaEngine.from_matrices(compile_nfa_matrices(PATTERNS[case["source"]]))
            data = _plant(_text(seed, WORDS, int(offsets[-1])), offsets, seed, ["error ", "fail "])
        state = {"engine": engine, "batch": DeviceBatch(data.cpu().numpy(), offsets, layout="csr"),
                 "mask": _bytes_out(case["n"], 8), "accept": _bytes_out(case["n"])}
    elif kind == "prob":
        offsets, symbols = _symbols(case, seed)
        state = {"engine": ProbNfaEngine(*dirichlet_pnfa(np.random.default_rng(2), 32)), "symbols": symbols,
                 "ll": torch.zeros(case["n"], dtype=torch.float64, device=DEVICE),
                 "mass": torch.zeros(case["n"], dtype=torch.float64, device=DEVICE)}
        if case["ragged"]:
            state["begin"] = torch.from_numpy(offsets[:-1].copy()).to(DEVICE)
            state["end"] = torch.from_numpy(offsets[1:].copy()).to(DEVICE)
    else:
        offsets = _offsets(case, seed)
        count, rng = case["patterns"], np.random.default_rng(7)
        patterns = _rule_set((count + 1) // 2)
        patterns += [NfaEngine.from_matrices(random_nfa64(rng)) for _ in range(count // 2)]
        queue = MixEngine(patterns)
        queue.plan(offsets[:-1], offsets[1:], np.random.default_rng(seed).integers(0, count, case["n"]))
        state = {"queue": queue, "bytes": _text(seed, UPPER, int(offsets[-1])), "mask": _bytes_out(case["n"], 8),
                 "accept": _bytes_out(case["n"])}
    return _first_use(dict(state, case=dict(case)))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "api":
        if case["texts"]:
            return np.asarray(state["engine"].match(state["strings"]), dtype=bool)
        return state["engine"].match_arrays(state["data"], state["offsets"])
    if kind == "dfa":
        out = state["final"], state["accept"]
        if case["layout"] == "csr":
            state["engine"].match_device(state["bytes"].data_ptr(), state["offsets"].data_ptr(), case["n"],
                                         out[0].data_ptr(), out[1].data_ptr())
        else:
            state["engine"].match_batch_device(state["batch"], out[0].data_ptr(), out[1].data_ptr())
        return out
    if kind == "multi":
        state["engine"].match_batch_device(state["batch"], state["final"].data_ptr(), state["accept"].data_ptr())
        return state["final"], state["accept"]
    if kind == "long":
        state["engine"].match_plan(state["plan"], state["bytes"].data_ptr(), state["final"].data_ptr(),
                                   state["accept"].data_ptr())
        return state["final"], state["accept"]
    if kind == "nfa":
        state["engine"].match_batch_device(state["batch"], state["mask"].data_ptr(), state["accept"].data_ptr())
        return state["mask"], state["accept"]
    if kind == "prob":
        if case["ragged"]:
            state["engine"].loglik_ranges_device(state["symbols"].data_ptr(), state["begin"].data_ptr(),
                                                 state["end"].data_ptr(), case["n"], state["ll"].data_ptr(),
                                                 state["mass"].data_ptr())
        else:
            state["engine"].loglik_device(state["symbols"].data_ptr(), case["n"], case["lo"], state["ll"].data_ptr(),
                                          state["mass"].data_ptr())
        return state["ll"], state["mass"]
    state["queue"].run(state["bytes"].data_ptr(), state["mask"].data_ptr(), state["accept"].data_ptr())
    return state["mask"], state["accept"]


def work(case):
    """Bytes: every character once, every string's range and results once. Operations: the
    matrix-vector products of the probabilistic automaton (the others only look up)."""
    n, lo, hi = case["n"], case["lo"], case["hi"]
    mean = lo if lo == hi else (hi - lo) / math.log(hi / lo)   # of a log-uniform length
    chars = n * mean
    results = {"prob": 16, "nfa": 9, "mix": 9, "multi": 2 * case.get("patterns", 1)}.get(case["kind"], 2)
    return {"bytes": chars + n * (8 + results), "flops": 2 * 64 * 64 * chars if case["kind"] == "prob" else 0}


def _symbols(case, seed):
    offsets = _offsets(case, seed)
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return offsets, torch.randint(0, 32, (int(offsets[-1]),), generator=g, device=DEVICE, dtype=torch.uint8)


def exact(case, seed):
    """The forward recurrence s <- T[c] s in 64 bits with the state's mass divided out of each step;
    the other kinds return whole numbers. The log of the mass has no value of its own to compare: the
    columns of T sum to one, so it is the rounding of T alone, about 1e-7."""
    if case["kind"] != "prob":
        return None
    offsets, symbols = _symbols(case, seed)
    T, start, accept = (torch.from_numpy(np.asarray(x, np.float64)).to(DEVICE)
                        for x in dirichlet_pnfa(np.random.default_rng(2), 32))
    lengths = torch.from_numpy(np.diff(offsets)).to(DEVICE)
    begin = torch.from_numpy(offsets[:-1].copy()).to(DEVICE)
    s = start.repeat(case["n"], 1)
    log = torch.zeros(case["n"], dtype=torch.float64, device=DEVICE)
    for t in range(int(lengths.max())):
        live = lengths > t
        c = symbols[(begin + t).clamp(max=len(symbols) - 1)].long()
        x = torch.bmm(T[c], s.unsqueeze(-1)).squeeze(-1)
        m = x.sum(-1)
        s = torch.where(live.unsqueeze(-1), x / m.unsqueeze(-1), s)
        log = torch.where(live, log + m.log(), log)
    return (s @ accept).log() + log, None
