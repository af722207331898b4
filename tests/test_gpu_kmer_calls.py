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
