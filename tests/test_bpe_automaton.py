"""The automaton of a merge table (csrc/bpe_automaton.hpp) against the oracle, on the CPU: the same
tokens for every row, and no automaton for the tables it cannot stand for."""
from __future__ import annotations

import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
from tests import util

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("automaton") / "automaton.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-shared", "-fPIC",
                           os.path.join(HERE, "support", "bpe_automaton_host.cpp"), "-o", path])
    so = ctypes.CDLL(path)
    so.automaton_create.restype = ctypes.c_void_p
    so.automaton_states.restype = ctypes.c_int64
    so.automaton_max_states.restype = ctypes.c_int64
    so.automaton_encode.restype = ctypes.c_int64
    return so


class Automaton:
    def __init__(self, lib, pair_a, pair_b, new_id, n_symbols, max_states=0):
        self.lib, self.b2s = lib, np.arange(256, dtype=np.int32)
        a, b, p = (np.ascontiguousarray(x, dtype=np.int32) for x in (pair_a, pair_b, new_id))
        last = {(int(x), int(y)): i for i, (x, y) in enumerate(zip(a, b))}
        eff = np.array([last[(int(x), int(y))] == i for i, (x, y) in enumerate(zip(a, b))], dtype=np.uint8)
        self.h = lib.automaton_create(O._p(self.b2s), O._p(a), O._p(b), O._p(p), O._p(eff), ctypes.c_int32(a.size),
                                      ctypes.c_int32(n_symbols), ctypes.c_int64(max_states))

    def encode(self, row):
        row = np.ascontiguousarray(row, dtype=np.uint8)
        out = np.empty(max(1, row.size), dtype=np.int32)
        n = self.lib.automaton_encode(ctypes.c_void_p(self.h), O._p(self.b2s), O._p(row), ctypes.c_int64(row.size), O._p(out))
        assert n >= 0
        return out[:n].copy()

    def __del__(self):
        if self.h:
            self.lib.automaton_destroy(ctypes.c_void_p(self.h))


def monotone(pair_a, pair_b, new_id):
    last = {(int(a), int(b)): i for i, (a, b) in enumerate(zip(pair_a, pair_b))}
    first_use = {}
    for i, (a, b) in enumerate(zip(pair_a, pair_b)):
        if last[(int(a), int(b))] == i:
            first_use.setdefault(int(a), i)
            first_use.setdefault(int(b), i)
    return all(first_use.get(int(p), 1 << 30) > i for i, p in enumerate(new_id)
               if last[(int(pair_a[i]), int(pair_b[i]))] == i)


def rows_over(rng, letters):
    """Random rows, tandem repeats, and rows with bytes that no rule names."""
    for n in (0, 1, 2, 3, 7, 30, 200, 1000):
        yield rng.choice(letters, n)
    for unit in (1, 2, 3, 5):
        yield np.tile(rng.choice(letters, unit), 400 // unit)
        yield np.concatenate([rng.choice(letters, 11), np.tile(rng.choice(letters, unit), 200 // unit), rng.choice(letters, 40)])
    row = rng.choice(letters, 600)
    row[rng.integers(0, 600, 30)] = rng.choice(np.frombuffer(b"NnX\x00\xff", dtype=np.uint8), 30)
    yield row


@pytest.mark.parametrize("which", ["4096", "32000"])
def test_trained_vocabularies(lib, which):
    bo = util.bpe_oracle(which)
    fa = Automaton(lib, bo.pair_a, bo.pair_b, bo.new_id, len(bo.vocab))
    assert fa.h and 0 < lib.automaton_states(ctypes.c_void_p(fa.h)) < (1 << 18)
    rng = np.random.default_rng(5)
    for _ in range(20):
        for row in rows_over(rng, np.frombuffer(b"ACGT", dtype=np.uint8)):
            np.testing.assert_array_equal(fa.encode(row), bo.encode_row(row, remap=False))


@pytest.mark.parametrize("letters", ["A", "AC", "ACG", "ACGT", "acgt"])
def test_random_tables(lib, letters):
    """Random merge lists (sides drawn from the tokens made so far, texts with more than one
    derivation, repeated pairs, rules that never fire): an automaton for every one whose rules are in
    order, and the oracle's tokens from it."""
    rng = np.random.default_rng(len(letters) + ord(letters[0]))
    built = 0
    for _ in range(60):
        toks, merges = list(letters), []
        for _ in range(int(rng.integers(1, 60))):
            a, b = toks[int(rng.integers(len(toks)))], toks[int(rng.integers(len(toks)))]
            if len(a) + len(b) > 40:
                continue
            merges.append((a, b))
            if a + b not in toks:
                toks.append(a + b)
        bo = O.BpeOracle(merges)
        if not monotone(bo.pair_a, bo.pair_b, bo.new_id):
            continue
        fa = Automaton(lib, bo.pair_a, bo.pair_b, bo.new_id, len(bo.vocab))
        assert fa.h
        built += 1
        for row in rows_over(rng, np.frombuffer(letters.encode(), dtype=np.uint8)):
            np.testing.assert_array_equal(fa.encode(row), bo.encode_row(row, naive=True, remap=False))
    assert built >= 5


def test_tables_without_an_automaton(lib):
    def make(merges):
        bo = O.BpeOracle(merges)
        return Automaton(lib, bo.pair_a, bo.pair_b, bo.new_id, len(bo.vocab)).h

    assert make([("A", "C")])
    assert not make([])                                              # no rules
    assert not make([("A", "C"), ("G", "T"), ("N", "A")])            # five letters
    assert not make([("A", "a")])                                    # letters that bits 1 and 2 do not tell apart
    doubled = [("A" * 2 ** i, "A" * 2 ** i) for i in range(8)]       # a token of 256 letters
    assert make(doubled[:7]) and not make(doubled)
    b2 = Automaton(lib, [65, 67], [67, 71], [256, 256], 257)         # one symbol for two texts
    assert not b2.h


def test_limit_of_states(lib):
    """As many states as the limit allows are built, one more is not (the shipped limit is the one the
    kernels were measured to)."""
    bo = util.bpe_oracle("4096")
    tables = (bo.pair_a, bo.pair_b, bo.new_id, len(bo.vocab))
    fa = Automaton(lib, *tables)
    n = lib.automaton_states(ctypes.c_void_p(fa.h))
    assert lib.automaton_max_states() == 1 << 19
    assert Automaton(lib, *tables, max_states=n).h and not Automaton(lib, *tables, max_states=n - 1).h
