"""BPE batches of more rows than surely fit the waves' steps: every wave gets its even share of the rows, of any lengths.
Against the CPU oracle, bit-exact."""
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
    if form in ("reads", "behind", "buffer"):          # any length up to 300
        return rng.integers(0, 301, size=90000)
    if form == "few":
        return rng.integers(0, 301, size=40000)
    if form == "sorted":                               # the last waves' rows take the most steps
        return np.sort(rng.integers(0, 301, size=90000))
    if form == "steps":                                # two lengths, far apart
        return np.repeat([300, 3], [30000, 100000])
    if form == "many":                                 # two items to a wave
        return rng.integers(0, 151, size=300000)
    if form == "empty":                                # items without a byte
        n = rng.integers(1, 301, size=90000)
        n[5000:15000] = 0
        n[20000:20070] = 0
        n[85000:] = 0
        return n
    n = rng.integers(0, 40, size=15000)                # "long": rows of a whole step between short ones
    n[rng.integers(0, 15000, size=3000)] = 2048
    n[rng.integers(0, 15000, size=3000)] = 2047
    return n


@pytest.mark.parametrize("form", ["reads", "behind", "buffer", "few", "sorted", "steps", "many", "empty", "long"])
def test_bpe_rows_in_even_shares(made, form):
    enc, oracle, pad = made
    print(f"bpe shares {form}", flush=True)
    rng = np.random.default_rng(len(form))
    lens = lengths_of(form, rng)
    longest, n = int(lens.max()), len(lens)
    front = 777 if form == "behind" else 0             # bytes in front of the first row
    behind = int(lens.sum()) // 2 if form in ("buffer", "few") else 0       # room that the batch leaves
    host = rng.choice(np.frombuffer(b"ACGTN", dtype=np.uint8), p=[.25, .25, .25, .2498, .0002], size=front + int(lens.sum()) + behind)
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


def test_bpe_run_of_empty_rows_costs_what_they_cost_apart(made):
    """A batch that is filled up with empty rows takes about the time of the same rows in any order (as one share the
    run took a single wave sixty times as long)."""
    enc, _, pad = made
    print("bpe shares: a run of empty rows", flush=True)
    rng = np.random.default_rng(7)
    lens = np.concatenate([rng.integers(100, 301, size=50000), np.zeros(50000, dtype=np.int64)])
    data = torch.from_numpy(rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), size=int(lens.sum()))).to(DEV)
    out = (torch.empty((lens.size, 96), dtype=torch.int32, device=DEV), torch.empty((lens.size, 96), dtype=torch.uint8, device=DEV),
           torch.empty(lens.size, dtype=torch.int32, device=DEV), torch.empty(1, dtype=torch.int32, device=DEV))
    took = []
    for order in (lens, rng.permutation(lens)):
        off = torch.from_numpy(np.concatenate([[0], np.cumsum(order)]).astype(np.int64)).to(DEV)
        least = float("inf")
        for _ in range(8):
            began, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            began.record()
            for _ in range(4):
                enc.encode_padded(data, off, 300, 96, pad, out=out)
            ended.record()
            torch.cuda.synchronize()
            least = min(least, began.elapsed_time(ended))
        took.append(least)
    assert took[0] < 8 * took[1]
