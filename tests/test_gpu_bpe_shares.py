"""BPE batches of tens of thousands of rows of mixed lengths, with bytes in front of the first row among them (larger
batches, of several steps per wave: test_gpu_bpe_even_shares.py).  Against the CPU oracle, bit-exact."""
import numpy as np
import pytest
import torch

from dnatok_amd import bpe_vocab, encoders
from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", params=["4096", "32000"])
def made(request):
    cfg = util.tokenizer_json(request.param)
    kv = bpe_vocab.KernelVocab(bpe_vocab.split_merges(cfg["model"]["merges"]))
    remap = kv.remap_to(cfg["model"]["vocab"], cfg["model"]["vocab"]["[UNK]"])
    enc = encoders.BpeEncoder(kv.pair_a, kv.pair_b, kv.new_id, len(kv), out_remap=remap)
    return enc, O.bpe_oracle_from_tokenizer_json(cfg), cfg["model"]["vocab"]["[PAD]"]


def lengths_of(form, rng):
    if form in ("reads", "behind"):                    # any length up to 300
        return rng.integers(0, 301, size=26000)
    if form == "sorted":                               # no row is where the mean length puts it
        return np.sort(rng.integers(0, 301, size=26000))
    if form == "steps":                                # two lengths, far apart
        return np.repeat([300, 3], [2000, 30000])
    if form == "empty":                                # more rows to a share than a wave looks at at once
        n = rng.integers(1, 301, size=30000)
        n[5000:9000] = 0
        n[20000:20070] = 0
        n[29000:] = 0
        return n
    n = rng.integers(0, 40, size=9000)                 # "long": rows of a whole step between short ones
    n[rng.integers(0, 9000, size=40)] = 2048
    n[rng.integers(0, 9000, size=40)] = 2047
    return n


@pytest.mark.parametrize("form", ["reads", "behind", "sorted", "steps", "empty", "long"])
def test_bpe_rows_dealt_out_by_bytes(made, form):
    enc, oracle, pad = made
    print(f"bpe shares {form}", flush=True)
    rng = np.random.default_rng(len(form))
    lens = lengths_of(form, rng)
    longest, n = int(lens.max()), len(lens)
    front = 777 if form == "behind" else 0             # bytes in front of the first row
    host = rng.choice(np.frombuffer(b"ACGTN", dtype=np.uint8), p=[.25, .25, .25, .2498, .0002], size=front + int(lens.sum()))
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64) + front
    rows = oracle.encode_batch(host, offsets)
    want_len = np.array([r.size for r in rows])
    data, off = torch.from_numpy(host).to(DEV), torch.from_numpy(offsets).to(DEV)
    width = (int(want_len.max()) + 7) // 4 * 4
    for pad_left in (False, True):
        ids, mask, lengths, m = enc.encode_padded(data, off, longest, width, pad, pad_left=pad_left)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(lengths.cpu().numpy(), want_len)
        eids, emask = O.pad_rows(rows, pad, width, pad_left=pad_left)
        np.testing.assert_array_equal(ids.cpu().numpy(), eids)
        np.testing.assert_array_equal(mask.cpu().numpy(), emask)
        assert int(m.item()) == int(want_len.max())
    tok, lengths = enc.encode(data, off, longest)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(lengths.cpu().numpy(), want_len)
    at = np.repeat(offsets[:-1] - np.concatenate([[0], np.cumsum(want_len)[:-1]]), want_len) + np.arange(int(want_len.sum()))
    np.testing.assert_array_equal(tok.cpu().numpy()[at], np.concatenate(rows))
