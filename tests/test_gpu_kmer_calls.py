"""k-mer calls whose launches depend on their arguments, against the CPU oracle.  Bit-exact."""
import numpy as np
import pytest
import torch

from dnatok_amd import encoders, kmer_tables
from tests.support import hf_tokenizers as hf
from oracle import oracle as O
from tests import util

pytestmark = pytest.mark.gpu
DEV = "cuda"
K = 6


@pytest.fixture(scope="module")
def enc():
    t = kmer_tables.tables_from_vocab(hf.kmer_vocab(K), K, 0)
    return encoders.KmerEncoder(K, t.digit, t.kmer_lut, t.single, pad_id=1, missing_id=0,
                                exp_off=t.exp_off, exp_len=t.exp_len, exp_flat=t.exp_flat)


def batch(lens, seed, n_rate=0.01):
    rng = np.random.default_rng(seed)
    p = [(1 - n_rate) / 4] * 4 + [n_rate]
    b = util.batch_from_strings(["".join(rng.choice(list("ACGTN"), p=p, size=n)) for n in lens])
    rows, status = O.kmer_encode(O.kmer_tables_from_vocab(hf.kmer_vocab(K), K, 0), b.data, b.offsets)
    return b, rows, status


def on_gpu(b):
    return torch.from_numpy(b.data).to(DEV), torch.from_numpy(b.offsets).to(DEV)


def fixed_width_out(n, cap):
    # (a maximum that no row reaches: the call must not build on what it finds)
    return (torch.full((n, cap), -7, dtype=torch.int32, device=DEV), torch.full((n, cap), 9, dtype=torch.uint8, device=DEV),
            torch.full((n,), -7, dtype=torch.int32, device=DEV), torch.full((n,), -7, dtype=torch.int32, device=DEV),
            torch.full((1,), 1 << 29, dtype=torch.int32, device=DEV))


def check_fixed(out, rows, status, cap, fill_to):
    ids, mask, lengths, st, longest = out
    kept = [r[:cap] for r in rows]
    assert int(longest.item()) == max((r.size for r in kept), default=0)
    np.testing.assert_array_equal(lengths.cpu().numpy(), [r.size for r in rows])
    np.testing.assert_array_equal(st.cpu().numpy() & 3, status & 3)
    eids, emask = O.pad_rows([r[:fill_to] for r in rows], 1, fill_to)
    np.testing.assert_array_equal(ids[:, :fill_to].cpu().numpy(), eids)
    np.testing.assert_array_equal(mask[:, :fill_to].cpu().numpy(), emask)


# rows, their lengths, the stride: a workgroup per row, sixteen lanes per row, a wave per row, both of them,
# and a stride beyond what the maximum's fields hold
FIXED = {"few": (7, (0, 3000), 640), "one": (1, (6000, 6000), 1280), "empty": (5, (0, 0), 128),
         "reads": (3000, (0, 300), 384), "odd_stride": (900, (0, 300), 333), "rows": (2500, (0, 900), 1000),
         "classes": (1500, (0, 3000), 3328), "cut": (300, (500, 2000), 96), "wide": (4, (0, 9000), 70000)}


@pytest.mark.parametrize("form", list(FIXED))
def test_kmer_fixed_width_reports_the_longest_row(enc, form):
    n, (lo, hi), cap = FIXED[form]
    for seed, fill_to in ((1, cap), (2, cap), (3, cap - 5)):
        print(f"kmer fixed width {form} fill_to={fill_to}", flush=True)
        lens = np.random.default_rng(seed).integers(lo, hi + 1, size=n)
        b, rows, status = batch(lens, seed)
        data, off = on_gpu(b)
        out = fixed_width_out(n, cap)
        enc.encode_padded(data, off, cap, fill_to=fill_to, out=out)
        torch.cuda.synchronize()
        check_fixed(out, rows, status, cap, fill_to)


@pytest.mark.parametrize("form", ["few", "reads", "rows"])
def test_kmer_fixed_width_call_replayed_from_a_graph(enc, form):
    """A captured call keeps to its own buffers: its replays on two streams at once, with eager calls on the
    stream it was captured on in between, all report their own longest row."""
    print(f"kmer fixed width from a graph {form}", flush=True)
    n, (lo, hi), cap = FIXED[form]
    made = [batch(np.random.default_rng(seed).integers(lo, hi + 1, size=n), seed) for seed in (11, 12, 13)]
    room = max(b.data.size for b, _, _ in made)
    side, graphs = torch.cuda.Stream(), []
    for _ in range(2):
        data, off = torch.zeros(room, dtype=torch.uint8, device=DEV), torch.zeros(n + 1, dtype=torch.int64, device=DEV)
        out = fixed_width_out(n, cap)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            enc.encode_padded(data, off, cap, fill_to=cap, out=out)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            enc.encode_padded(data, off, cap, fill_to=cap, out=out)
        graphs.append((g, data, off, out))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    eager_in, eager_out = on_gpu(made[2][0]), fixed_width_out(n, cap)
    for first in (0, 1, 0):
        for q, (g, data, off, out) in enumerate(graphs):
            b = made[(first + q) % 2][0]
            data[:b.data.size].copy_(torch.from_numpy(b.data))
            off.copy_(torch.from_numpy(b.offsets))
            out[4].fill_(1 << 29)
        torch.cuda.synchronize()
        for q, (g, *_) in enumerate(graphs):
            with torch.cuda.stream(streams[q]):
                g.replay()
        with torch.cuda.stream(side):
            enc.encode_padded(*eager_in, cap, fill_to=cap, out=eager_out)
        torch.cuda.synchronize()
        for q, (_, _, _, out) in enumerate(graphs):
            _, rows, status = made[(first + q) % 2]
            check_fixed(out, rows, status, cap, cap)
        check_fixed(eager_out, made[2][1], made[2][2], cap, cap)
