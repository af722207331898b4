"""How the rows of a large batch are dealt out to waves (csrc/bpe_shares.hpp), on the CPU: every row is in one share,
and no share takes a wave many more steps than the others, whatever the rows' lengths are."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))
SHARES = 4096                                          # sixteen waves on 256 CUs


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("shares") / "shares.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-shared", "-fPIC",
                           os.path.join(HERE, "support", "bpe_shares_host.cpp"), "-o", path])
    return ctypes.CDLL(path)


def lengths_of(form):
    rng = np.random.default_rng(len(form))
    reads = rng.integers(100, 301, size=100000)
    if form == "filled up":                            # to a fixed number of rows
        return np.concatenate([reads[:50000], np.zeros(50000, dtype=np.int64)])
    if form == "empty in front":
        return np.concatenate([np.zeros(50000, dtype=np.int64), reads[:50000]])
    if form == "short and long":
        return np.concatenate([np.full(200000, 3), np.full(10000, 2048)])
    if form == "mixed":
        return rng.choice([0, 1, 31, 32, 33, 300, 2048], size=60000)
    return np.sort(reads) if form == "sorted" else reads


@pytest.mark.parametrize("front", [0, 777])
@pytest.mark.parametrize("form", ["reads", "sorted", "filled up", "empty in front", "short and long", "mixed"])
def test_shares_cost_about_the_same(lib, form, front):
    lens = lengths_of(form)
    n = len(lens)
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64) + front
    first, guess = np.zeros(SHARES + 1, dtype=np.int32), np.zeros(SHARES, dtype=np.int32)
    lib.shares_deal(O._p(offsets), ctypes.c_int32(n), ctypes.c_int32(SHARES), O._p(first), O._p(guess))
    assert first[0] == 0 and first[-1] == n and (np.diff(first) >= 0).all()
    assert (guess >= 0).all() and (guess <= n + 1).all()
    if form == "reads":                                # (rows of about one length lie where they are looked for)
        assert np.abs(guess - first[:-1]).max() < 256
    lanes = np.maximum(1, (lens + 31) // 32)           # what a row takes of a wave
    to = np.concatenate([[0], np.cumsum(lanes)])
    of_share = to[first[1:]] - to[first[:-1]]
    # a share has room for its part of the cost, in lanes, and takes the rows that begin in it
    room = (lens.sum() + 32 * n) / 32 / SHARES + 1
    assert of_share.max() <= room + lanes.max()
