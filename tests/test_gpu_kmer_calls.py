"""k-mer calls whose launches depend on their arguments, against the CPU oracle.  Bit-exact."""
import threading

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


def test_kmer_longest_row_of_a_batch_split_by_class_costs_little(enc):
    """Thousands of waves that are done at once do not raise the maximum one after the other (with it the call took
    more than twice as long as without)."""
    print("kmer longest row of a split batch", flush=True)
    n, cap = 20000, 512
    lens = np.random.default_rng(4).integers(1900, 2101, size=n)
    b = batch(lens, 4)[0]
    data, off = on_gpu(b)
    out = fixed_width_out(n, cap)
    took = []
    for longest in (out[4], None):
        least = float("inf")
        for _ in range(8):
            began, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            began.record()
            for _ in range(4):
                enc.encode_padded(data, off, cap, fill_to=cap, out=(*out[:4], longest))
            ended.record()
            torch.cuda.synchronize()
            least = min(least, began.elapsed_time(ended))
        took.append(least)
    assert int(out[4].item()) == min(cap, int(out[2].max().item()))
    assert took[0] < 1.7 * took[1]


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


def check_longest(out, rows, status):
    ids, mask, lengths, st, longest = out
    kept = [r[:ids.shape[1]] for r in rows]
    width = max(r.size for r in kept)
    assert int(longest.item()) == width
    np.testing.assert_array_equal(lengths.cpu().numpy(), [r.size for r in rows])
    np.testing.assert_array_equal(st.cpu().numpy() & 3, status & 3)
    eids, emask = O.pad_rows(kept, 1, width)
    np.testing.assert_array_equal(ids[:, :width].cpu().numpy(), eids)
    np.testing.assert_array_equal(mask[:, :width].cpu().numpy(), emask)


@pytest.mark.parametrize("form,guess", [("few", 600), ("reads", 300), ("rows", 900), ("rows", 0)])
def test_kmer_graphs_padded_to_the_longest_row_beside_eager_calls(enc, form, guess):
    """Captured calls that pad to their longest row (with a guess: reported by the kernel itself), replayed on other
    streams than the one they were captured on, where eager calls of a fixed width and of the longest row are made
    meanwhile: every call reports its own longest row, also in the rounds after."""
    print(f"kmer padded to the longest row from graphs {form} guess={guess}", flush=True)
    n, (lo, hi), cap = FIXED[form]
    made = [batch(np.random.default_rng(seed).integers(lo, hi // (1 + seed % 2) + 1, size=n), seed) for seed in (31, 32, 33, 34)]
    room = max(b.data.size for b, _, _ in made)
    side, graphs = torch.cuda.Stream(), []
    for _ in range(2):
        data, off = torch.zeros(room, dtype=torch.uint8, device=DEV), torch.zeros(n + 1, dtype=torch.int64, device=DEV)
        out = fixed_width_out(n, cap)
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            enc.encode_padded(data, off, cap, width_guess=guess, out=out)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            enc.encode_padded(data, off, cap, width_guess=guess, out=out)
        graphs.append((g, data, off, out))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    fixed_in, fixed = on_gpu(made[2][0]), fixed_width_out(n, cap)
    eager_in, eager = on_gpu(made[3][0]), fixed_width_out(n, cap)
    for first in (0, 1, 0, 1):
        for q, (_, data, off, out) in enumerate(graphs):
            b = made[(first + q) % 2][0]
            data[:b.data.size].copy_(torch.from_numpy(b.data))
            off.copy_(torch.from_numpy(b.offsets))
            out[4].fill_(1 << 29)
        torch.cuda.synchronize()
        for _ in range(4):
            for q, (g, *_) in enumerate(graphs):
                with torch.cuda.stream(streams[q]):
                    g.replay()
            with torch.cuda.stream(side):
                enc.encode_padded(*fixed_in, cap, fill_to=cap, out=fixed)
                enc.encode_padded(*eager_in, cap, width_guess=guess, out=eager)
        torch.cuda.synchronize()
        for q, (_, _, _, out) in enumerate(graphs):
            check_longest(out, *made[(first + q) % 2][1:])
        check_fixed(fixed, made[2][1], made[2][2], cap, cap)
        check_longest(eager, *made[3][1:])


def test_kmer_calls_of_two_threads_on_their_own_default_streams(enc):
    """hipStreamPerThread is one handle and a stream for every host thread: calls on it may overlap."""
    print("kmer calls on hipStreamPerThread", flush=True)
    n, (lo, hi), cap = FIXED["rows"]
    made = [batch(np.random.default_rng(seed).integers(lo, hi // (1 + seed % 2) + 1, size=n), seed) for seed in (41, 42)]
    per_thread = torch.cuda.ExternalStream(2)
    inputs, outs, failed = [on_gpu(b) for b, _, _ in made], [fixed_width_out(n, cap) for _ in made], []
    torch.cuda.synchronize()

    def calls(q):
        try:
            with torch.cuda.stream(per_thread):
                for fill_to in (cap, 0) * 10 + (cap,):
                    enc.encode_padded(*inputs[q], cap, fill_to=fill_to, width_guess=900, out=outs[q])
        except Exception as e:                           # (an assertion in a thread is not seen by pytest)
            failed.append(e)

    threads = [threading.Thread(target=calls, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed
    for q in range(2):
        check_fixed(outs[q], made[q][1], made[q][2], cap, cap)


def check_packed(out, rows, status, total):
    ids, out_off, mask, lengths, st = out
    want = np.concatenate([[0], np.cumsum([r.size for r in rows])])
    np.testing.assert_array_equal(out_off.cpu().numpy(), want)
    np.testing.assert_array_equal(lengths.cpu().numpy(), [r.size for r in rows])
    np.testing.assert_array_equal(st.cpu().numpy() & 7, status)
    n = int(want[-1])
    np.testing.assert_array_equal(ids[:n].cpu().numpy(), np.concatenate(rows))
    assert bool((ids[n:] == -7).all())
    if mask is not None:
        assert bool((mask[:n] == 1).all()) and bool((mask[n:] == 9).all())


def packed_out(n, total, shift=0):
    # (nothing of an earlier content may count: the offsets' cells look like offsets)
    ids = torch.full((total + shift,), -7, dtype=torch.int32, device=DEV)[shift:]
    mask = torch.full((total + shift,), 9, dtype=torch.uint8, device=DEV)[shift:]
    return (ids, torch.full((n + 1,), 77, dtype=torch.int64, device=DEV), mask,
            torch.full((n,), -7, dtype=torch.int32, device=DEV), torch.full((n,), -7, dtype=torch.int32, device=DEV))


def packed_lens(n, seed, most=300):
    """Reads with rows of no byte, of less than a window, at the borders between the rows that are read once
    (up to 389 bytes), those walked by sixteen lanes (773) and the others, and of several steps of a wave, anywhere
    among them."""
    rng = np.random.default_rng(seed)
    lens = rng.integers(0, most + 1, size=n)
    for v in (0, 1, 5, 6, 383, 384, 385, 389, 390, 768, 773, 774, 1536, 1537, 2304, 2311, 9001):
        lens[rng.integers(0, n)] = v
    return lens


@pytest.mark.parametrize("n,polls", [(n, -1) for n in (1, 31, 32, 33, 127, 129, 2500, 24577, 25000, 49153, 70001, 98304 + 129, 123000, 160001)] +
                         [(n, 0) for n in (1, 33, 513, 2500, 24577, 25000, 49153)])
def test_kmer_packed_reads(enc, n, polls):
    """Batches of fewer and of more tiles than the chip holds (and than a wave looks back on in one trip), of
    tiles of 32 to 192 rows; the tiles' sums waited for, and counted by whoever finds one missing."""
    print(f"kmer packed n={n} polls={polls}", flush=True)
    lens = packed_lens(n, n, 300 if n < 50000 else 60)
    if n == 1:
        lens[:] = 300
    b, rows, status = batch(lens, n + 1, n_rate=0.004)
    data, off = on_gpu(b)
    enc.set_packed_polls(polls)
    try:
        for shift in (0, 1, 3):
            out = packed_out(n, b.data.size, shift)
            enc.encode_packed(data, off, want_mask=True, out=out)
            torch.cuda.synchronize()
            check_packed(out, rows, status, b.data.size)
        out = packed_out(n, b.data.size)
        enc.encode_packed(data, off, out=(out[0], out[1], None, out[3], out[4]))
        torch.cuda.synchronize()
        check_packed((out[0], out[1], None, out[3], out[4]), rows, status, b.data.size)
    finally:
        enc.set_packed_polls(-1)


@pytest.mark.parametrize("k", [2, 3, 4, 5, 7, 8])
def test_kmer_packed_reads_of_other_k(k):
    print(f"kmer packed k={k}", flush=True)
    vocab = hf.kmer_vocab(k)
    t = kmer_tables.tables_from_vocab(vocab, k, 0)
    e = encoders.KmerEncoder(k, t.digit, t.kmer_lut, t.single, pad_id=1, missing_id=0, exp_off=t.exp_off, exp_len=t.exp_len, exp_flat=t.exp_flat)
    rng = np.random.default_rng(k)
    lens = rng.integers(0, 301, size=3000)
    lens[7:14] = 65 * k - 1, 65 * k, 129 * k - 1, 129 * k, 256 * k, 256 * k + 1, 384 * k + 5
    lens[2999] = 64 * k
    b = util.batch_from_strings(["".join(rng.choice(list("ACGTNx"), p=[.247, .247, .247, .247, .008, .004], size=n)) for n in lens])
    rows, status = O.kmer_encode(O.kmer_tables_from_vocab(vocab, k, 0), b.data, b.offsets)
    out = packed_out(len(lens), b.data.size)
    e.encode_packed(*on_gpu(b), want_mask=True, out=out)
    torch.cuda.synchronize()
    check_packed(out, rows, status, b.data.size)


@pytest.mark.parametrize("k,polls", [(2, -1), (3, -1), (5, -1), (6, -1), (6, 0), (7, -1), (8, -1), (8, 0)])
def test_kmer_packed_long_rows_in_parts(k, polls):
    """Rows that several waves share, at the borders where a part more begins and where a part is empty, beside each
    other and among reads; also counted by those that find a sum missing."""
    print(f"kmer packed, long rows k={k} polls={polls}", flush=True)
    vocab = hf.kmer_vocab(k)
    t = kmer_tables.tables_from_vocab(vocab, k, 0)
    e = encoders.KmerEncoder(k, t.digit, t.kmer_lut, t.single, pad_id=1, missing_id=0, exp_off=t.exp_off, exp_len=t.exp_len, exp_flat=t.exp_flat)
    rng = np.random.default_rng(k)
    n = 9000
    lens = rng.integers(0, 40 * k, size=n)
    windows = [1023, 1024, 1025, 2047, 2048, 2049, 2304, 3071, 3072, 6 * 1024 + 1, 7 * 1024, 8 * 1024 - 1, 8 * 1024, 8 * 1024 + 1, 9 * 1024, 40001]
    long = [w * k + int(rng.integers(0, k)) for w in windows] + [2048 * k + k - 1]
    lens[:5] = long[-5:]
    lens[4000:4000 + len(long)] = long
    lens[n - 1] = 2049 * k
    text = rng.choice(np.frombuffer(b"ACGTNx", dtype=np.uint8), p=[.248, .248, .248, .248, .007, .001], size=int(lens.sum()))
    at = int(lens[:4003].sum())
    text[at:at + int(lens[4003])] = np.where(np.isin(text[at:at + int(lens[4003])], list(b"Nx")), ord("A"), text[at:at + int(lens[4003])])
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    rows, status = O.kmer_encode(O.kmer_tables_from_vocab(vocab, k, 0), text, offsets)
    out = packed_out(n, text.size)
    e.set_packed_polls(polls)
    e.encode_packed(torch.from_numpy(text).to(DEV), torch.from_numpy(offsets).to(DEV), want_mask=True, out=out)
    torch.cuda.synchronize()
    check_packed(out, rows, status, text.size)


def test_kmer_packed_reads_behind_a_long_row_wait_for_it(enc):
    """A row that takes longer than all others costs about the same in front of them as behind them (three times as
    much where everybody behind it counted the rows around it)."""
    print("kmer packed, a long row in front", flush=True)
    rng = np.random.default_rng(8)
    reads = rng.integers(100, 301, size=100000)
    took = []
    for lens in (np.concatenate([[200000], reads]), np.concatenate([reads, [200000]])):
        off = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)).to(DEV)
        data = torch.from_numpy(rng.choice(np.frombuffer(b"ACGT", dtype=np.uint8), size=int(lens.sum()))).to(DEV)
        out = packed_out(lens.size, int(lens.sum()))
        least = float("inf")
        for _ in range(8):
            began, ended = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            began.record()
            for _ in range(4):
                enc.encode_packed(data, off, out=out)
            ended.record()
            torch.cuda.synchronize()
            least = min(least, began.elapsed_time(ended))
        took.append(least)
    assert took[0] < 2 * took[1]


def test_kmer_packed_reads_replayed_from_a_graph(enc):
    print("kmer packed from a graph", flush=True)
    n = 9000
    made = [batch(packed_lens(n, seed), seed, n_rate=0.004) for seed in (21, 22)]
    room = max(b.data.size for b, _, _ in made)
    data, off = torch.zeros(room, dtype=torch.uint8, device=DEV), torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    out = packed_out(n, room)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        enc.encode_packed(data, off, want_mask=True, out=out)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        enc.encode_packed(data, off, want_mask=True, out=out)
    for which in (0, 1, 1, 0):
        b, rows, status = made[which]
        data[:b.data.size].copy_(torch.from_numpy(b.data))
        off.copy_(torch.from_numpy(b.offsets))
        out[0].fill_(-7), out[2].fill_(9)
        g.replay()
        torch.cuda.synchronize()
        check_packed(out, rows, status, room)


def test_kmer_packed_reads_full_of_n(enc):
    """More spelled windows than a tile's list has room for, in some tiles; in others none."""
    print("kmer packed, many N", flush=True)
    rng = np.random.default_rng(5)
    rows = []
    for i in range(1200):
        p = [.1, .1, .1, .1, .6] if 300 <= i < 500 else [.25, .25, .25, .25, 0] if i < 800 else [.24, .24, .24, .24, .04]
        rows.append("".join(rng.choice(list("ACGTN"), p=p, size=int(rng.integers(0, 390)))))
    b = util.batch_from_strings(rows)
    want, status = O.kmer_encode(O.kmer_tables_from_vocab(hf.kmer_vocab(K), K, 0), b.data, b.offsets)
    out = packed_out(len(rows), b.data.size)
    enc.encode_packed(*on_gpu(b), want_mask=True, out=out)
    torch.cuda.synchronize()
    check_packed(out, want, status, b.data.size)


def test_kmer_packed_reads_of_a_table_with_gaps():
    """Plain windows without an id are spelled as well."""
    print("kmer packed, table with gaps", flush=True)
    vocab = {w: i for w, i in hf.kmer_vocab(K).items() if not (len(w) == K and w.startswith("CG"))}
    t = kmer_tables.tables_from_vocab(vocab, K, 0)
    e = encoders.KmerEncoder(K, t.digit, t.kmer_lut, t.single, pad_id=1, missing_id=0, exp_off=t.exp_off, exp_len=t.exp_len, exp_flat=t.exp_flat)
    rng = np.random.default_rng(6)
    b = util.batch_from_strings(["".join(rng.choice(list("ACGTN"), p=[.248, .248, .248, .248, .008], size=n)) for n in packed_lens(3000, 7)])
    want, status = O.kmer_encode(O.kmer_tables_from_vocab(vocab, K, 0), b.data, b.offsets)
    assert any((r < 0).any() for r in want) is False
    out = packed_out(3000, b.data.size)
    e.encode_packed(*on_gpu(b), want_mask=True, out=out)
    torch.cuda.synchronize()
    check_packed(out, want, status, b.data.size)
