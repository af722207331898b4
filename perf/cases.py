"""What the framework is timed on: the encode calls that a program makes through the public entry
points (``DNATok``, ``encoders``), over the sizes that such programs bring.

Kinds of case, and what each stands for:

strings      sequences as Python strings through ``DNATok``: ids on the host (``encode_batch_to_ids``, what
             the command line and a data loader call) or narrow padded ids with masks on the GPU
             (``encode_batch_with_padding``, what an embedding loop calls), as wide as the model
bpe_rows     windows of one length through the BPE engine to padded rows on the GPU: training batches
             of fixed windows, and contigs of 100 kbp that are cut into chunks inside the call
bpe_reads    sequencing reads of 100 - 300 bp through the BPE engine to padded rows
bpe_ragged   long reads of mixed lengths through the BPE and the character tokenizer in one pass,
             packed back to back
kmer_rows    windows of one length through the 6-mer encoder to rows of a model's fixed width
kmer_packed  reads through the 6-mer encoder, packed back to back
char_rows    windows of one length through the single-nucleotide table
char_embed   the single-nucleotide table fused with the embedding gather

The BPE vocabularies are the two trained ones of the test fixtures (4,096 and 32,000 entries), and the
bases come from the Markov chains these were trained on, with the N and the tandem repeats of the
benchmark's configurations.
"""
import functools
import json
import os

import numpy as np
import torch

from dnatok_amd import bpe_vocab, builtin_tokenizers, encoders, kmer_tables
from dnatok_amd.dna_tokenizer import DNATok

GOLDEN = os.path.join("tests", "golden")
BASES = b"ACGT"
N = ord("N")
ID_TYPES = {"int32": torch.int32, "int64": torch.int64}


def listed():
    return [
        # one chunk of the command line's benchmark: a call whose length is its latency
        {"name": "bpe4096_strings_32x4k", "kind": "strings", "tok": "bpe4096", "api": "ids", "rows": 32, "length": 4096},
        # an embedding loop's batch with a k-mer tokenizer: narrow ids, padded on the left, mask
        {"name": "kmer6_strings_256x4k", "kind": "strings", "tok": "kmer6", "api": "padding", "rows": 256, "length": 4096},
        # a training batch of windows, about a row per team of threads that the chip holds
        {"name": "bpe4096_rows_1024x1k", "kind": "bpe_rows", "vocab": 4096, "rows": 1024, "length": 1024, "ids": "int32"},
        # a shard of windows in one call: throughput with every CU busy
        {"name": "bpe4096_rows_16384x1k", "kind": "bpe_rows", "vocab": 4096, "rows": 16384, "length": 1024, "ids": "int32"},
        # contigs: rows cut into chunks and joined at seams
        {"name": "bpe32000_rows_32x100k", "kind": "bpe_rows", "vocab": 32000, "rows": 32, "length": 100000, "ids": "int32"},
        # short reads, in the id type that the tokenizer backend returns
        {"name": "bpe4096_reads_100k", "kind": "bpe_reads", "vocab": 4096, "rows": 100000, "ids": "int64"},
        # long reads of mixed lengths for a model that takes both tokenizations
        {"name": "bpe4096_ragged_4096", "kind": "bpe_ragged", "vocab": 4096, "rows": 4096},
        # one batch of 6-mer windows: a single launch
        {"name": "kmer6_rows_256x6k", "kind": "kmer_rows", "rows": 256, "length": 6000},
        # a shard of them: the memory system's rate
        {"name": "kmer6_rows_65536x6k", "kind": "kmer_rows", "rows": 65536, "length": 6000},
        # short reads, packed
        {"name": "kmer6_packed_100k", "kind": "kmer_packed", "rows": 100000},
        # single nucleotides, a shard
        {"name": "char_rows_21760x8k", "kind": "char_rows", "rows": 21760, "length": 8192},
        # single nucleotides straight to embedding rows
        {"name": "char_embed_64x8k", "kind": "char_embed", "rows": 64, "length": 8192, "dim": 512},
    ]


def _between(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["strings", "bpe_rows", "bpe_rows", "bpe_reads", "bpe_ragged", "kmer_rows", "kmer_packed",
                       "char_rows", "char_embed"])
    case = {"kind": kind}
    if kind == "strings":
        length = _between(rng, 60, 20000)
        case.update(tok=rng.choice(["bpe4096", "bpe32000", "kmer6", "char"]), api=rng.choice(["ids", "padding"]),
                    rows=_between(rng, 1, min(1024, max(1, 524288 // length))), length=length)
    elif kind == "bpe_rows":
        vocab = rng.choice([4096, 32000])
        length = _between(rng, 100, 100000)
        most = 16777216 if vocab == 4096 and length <= 1024 else 3200000
        case.update(vocab=vocab, rows=_between(rng, 1, max(1, most // length)), length=length,
                    ids=rng.choice(["int32", "int64"]))
    elif kind == "bpe_reads":
        case.update(vocab=rng.choice([4096, 32000]), rows=_between(rng, 64, 60000), ids=rng.choice(["int32", "int64"]))
    elif kind == "bpe_ragged":
        case.update(vocab=4096, rows=_between(rng, 64, 4096))
    elif kind == "kmer_rows":
        length = _between(rng, 200, 60000)
        case.update(rows=_between(rng, 1, 390000000 // length if length > 2000 else 65536), length=length)
    elif kind == "kmer_packed":
        case.update(rows=_between(rng, 64, 100000))
    elif kind == "char_rows":
        length = _between(rng, 100, 131072)
        case.update(rows=_between(rng, 1, 170000000 // length), length=length)
    else:
        dim = rng.choice([128, 256, 512, 768])
        length = _between(rng, 100, 32768)
        case.update(rows=_between(rng, 1, 262144000 // (length * dim)), length=length, dim=dim)
    return case


# ---- inputs ---------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _chain(order):
    """Cumulative transition table of the chain that the vocabulary was trained on (GC 41 %)."""
    rng = np.random.Generator(np.random.PCG64(3000 + order))
    p = rng.dirichlet(np.array([0.295, 0.205, 0.205, 0.295]) * 24.0, size=4 ** order)
    return torch.from_numpy(np.cumsum(p, axis=1)[:, :3].astype(np.float32)).cuda()


def _ascii(codes):
    return torch.tensor(list(BASES), dtype=torch.uint8, device="cuda")[codes.long()]


def _markov(total, order, gen):
    """``total`` bases of the chain as codes 0 - 3: stretches of about a thousand bases laid end to end."""
    cdf = _chain(order)
    n_ctx = cdf.shape[0]
    lanes = max(64, -(-total // 1024))
    steps = -(-total // lanes)
    ctx = torch.randint(0, n_ctx, (lanes,), generator=gen, device="cuda")
    u = torch.rand((steps, lanes, 1), generator=gen, device="cuda")
    out = torch.empty((steps, lanes), dtype=torch.uint8, device="cuda")
    for t in range(steps):
        nxt = (u[t] > cdf[ctx]).sum(1)
        out[t] = nxt
        ctx = (ctx * 4 + nxt) % n_ctx
    return out.t().reshape(-1)[:total].contiguous()


def _tandem_repeats(codes, gen):
    """A tenth of the bases inside repeats: homopolymers of 5 - 40 bp and units of 2 - 6 bp copied
    5 - 30 times, one of them somewhere in every 460 bases."""
    slot = 460
    n = codes.numel() // slot
    if n == 0:
        return codes

    def some(lo, hi):
        return torch.randint(lo, hi + 1, (n, 1), generator=gen, device="cuda")

    homo = torch.rand((n, 1), generator=gen, device="cuda") < 0.5
    unit = torch.where(homo, 1, some(2, 6))
    length = torch.where(homo, some(5, 40), unit * some(5, 30))
    start = (torch.rand((n, 1), generator=gen, device="cuda") * (slot - length)).long()
    at = torch.arange(slot, device="cuda")[None, :]
    inside = (at >= start) & (at < start + length)
    src = torch.where(inside, start + (at - start) % unit, at)
    codes[:n * slot] = torch.gather(codes[:n * slot].view(n, slot), 1, src).reshape(-1)
    return codes


def _bpe_bases(total, vocab, gen, n_rate=0.0):
    codes = _markov(total, 2 if vocab == 4096 else 3, gen)
    if vocab == 32000:
        codes = _tandem_repeats(codes, gen)
    data = _ascii(codes)
    if n_rate:
        data[torch.rand(total, generator=gen, device="cuda") < n_rate] = N
    return data


def _uniform_bases(rows, length, gen, n_rate=0.0, n_runs=0.0):
    """Uniform bases with single N (a share ``n_rate`` of the bases) or runs of 1 - 50 N (a share ``n_runs``)."""
    total = rows * length
    data = _ascii(torch.randint(0, 4, (total,), generator=gen, device="cuda", dtype=torch.uint8))
    if n_rate:
        data[torch.rand(total, generator=gen, device="cuda") < n_rate] = N
    if n_runs:
        n = max(1, int(total * n_runs / 25.5))
        start = torch.randint(0, total, (n,), generator=gen, device="cuda")
        run = torch.randint(1, 51, (n,), generator=gen, device="cuda")
        first = torch.cumsum(run, 0) - run
        at = torch.repeat_interleave(start - first, run) + torch.arange(int(run.sum()), device="cuda")
        row = torch.repeat_interleave(start // length, run)
        data[at[at // length == row]] = N                        # (runs end with their row)
    return data


def _even_offsets(rows, length):
    return torch.arange(rows + 1, dtype=torch.int64, device="cuda") * length


def _offsets_of(lengths):
    off = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=off[1:])
    return off


def _in_any_order(lengths, gen):
    """The batch's lengths are those of its size; which row has which comes from the seed."""
    return lengths[torch.randperm(lengths.numel(), generator=gen, device="cuda")]


def _read_lengths(rows, gen):
    """100 - 300 bp, evenly."""
    return _in_any_order(100 + torch.arange(rows, device="cuda") * 201 // rows, gen)


def _long_read_lengths(rows, gen):
    """Lognormal with a median of 2 kbp, 100 bp to 131 kbp."""
    q = (torch.arange(rows, device="cuda", dtype=torch.float64) + 0.5) / rows
    z = torch.special.ndtri(q)
    return _in_any_order(torch.exp(z * 0.87 + float(np.log(2000.0))).round().long().clamp(100, 131072), gen)


# ---- tokenizers -----------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _vocab(which):
    with open(os.path.join(GOLDEN, "bpe%d_tokenizer.json" % which)) as fh:
        cfg = json.load(fh)
    vocab = cfg["model"]["vocab"]
    kernel = bpe_vocab.KernelVocab(bpe_vocab.split_merges(cfg["model"]["merges"]))
    return kernel, kernel.remap_to(vocab, vocab["[UNK]"]), vocab["[PAD]"]


def _bpe(which):
    kernel, remap, pad = _vocab(which)
    return encoders.BpeEncoder(kernel.pair_a, kernel.pair_b, kernel.new_id, len(kernel), out_remap=remap), pad


@functools.lru_cache(maxsize=None)
def _kmer6_tables():
    vocab = builtin_tokenizers.kmer_vocab(6)
    return kmer_tables.tables_from_vocab(vocab, 6, vocab["<unk>"]), vocab["<pad>"], vocab["<unk>"]


def _kmer6():
    t, pad, unk = _kmer6_tables()
    return encoders.KmerEncoder(6, t.digit, t.kmer_lut, t.single, pad, unk, t.exp_off, t.exp_len, t.exp_flat)


def _char_lut():
    vocab = builtin_tokenizers.char_vocab()
    lut = np.zeros(256, dtype=np.int32)
    for ch in "ACGTN":
        lut[ord(ch)] = vocab[ch]
    return lut, vocab["<pad>"]


class _Embedder:
    """What ``DNATok`` is given: a tokenizer and an embedding."""

    def __init__(self, tokenizer, pad_id):
        self.tokenizer, self.pad_id = tokenizer, pad_id

    def embed_tokens(self, ids):
        return ids


def _dnatok(tok):
    char = builtin_tokenizers.build_char_tokenizer()
    if tok == "char":
        emb = _Embedder(char, builtin_tokenizers.char_vocab()["<pad>"])
    elif tok == "kmer6":
        emb = _Embedder(builtin_tokenizers.build_kmer_tokenizer(6), builtin_tokenizers.kmer_vocab(6)["<pad>"])
    else:
        path = os.path.join(GOLDEN, "%s_tokenizer.json" % tok)
        emb = _Embedder(type(char).from_file(path), _vocab(int(tok[3:]))[2])
    dn = DNATok(emb)
    dn.discover()
    return dn


# ---- the cases ------------------------------------------------------------------------------

def _bpe_width(case):
    """Cells that a model leaves for a row: a token is five bases (4,096) or seven (32,000) long on average."""
    longest = 300 if case["kind"] == "bpe_reads" else case["length"]
    w = longest // (4 if case["vocab"] == 4096 else 5) + 8
    return w + (-w) % 32


def _strings_width(case):
    per_token = {"bpe4096": 4, "bpe32000": 5, "kmer6": 4, "char": 1}[case["tok"]]
    w = case["length"] // per_token + (64 if case["tok"] == "kmer6" else 16)         # (windows with N are spelled out)
    return w + (-w) % 16


def _kmer_width(case):
    w = case["length"] // 6 * 5 // 4 + 16
    return w + (-w) % 128


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, rows = case["kind"], case["rows"]
    s = {"case": case}
    if kind == "strings":
        tok, length = case["tok"], case["length"]
        # (lengths within a tenth of each other, as windows cut at feature borders are)
        lens = _in_any_order(length - torch.arange(rows, device="cuda") * (length // 10) // rows, gen).tolist()
        total = sum(lens)
        if tok.startswith("bpe"):
            data = _bpe_bases(total, int(tok[3:]), gen)
        else:
            data = _uniform_bases(1, total, gen, n_runs=0.005)
        text = bytes(data.cpu().numpy()).decode("ascii")
        ends = np.cumsum(lens).tolist()
        dn = _dnatok(tok)
        dn.token_len = _strings_width(case)                      # (the model's width)
        s.update(dn=dn, seqs=[text[e - n:e] for e, n in zip(ends, lens)])
    elif kind in ("bpe_rows", "bpe_reads"):
        if kind == "bpe_rows":
            off, total, longest = _even_offsets(rows, case["length"]), rows * case["length"], case["length"]
        else:
            off = _offsets_of(_read_lengths(rows, gen))
            total, longest = int(off[-1]), 300
        enc, pad = _bpe(case["vocab"])
        width = _bpe_width(case)
        s.update(enc=enc, pad=pad, data=_bpe_bases(total, case["vocab"], gen), off=off, longest=longest, width=width,
                 tok=torch.empty(total, dtype=torch.int32, device="cuda") if longest > 2048 else None,
                 out=(torch.empty((rows, width), dtype=ID_TYPES[case["ids"]], device="cuda"),
                      torch.empty((rows, width), dtype=torch.uint8, device="cuda"),
                      torch.empty(rows, dtype=torch.int32, device="cuda"),
                      torch.empty(1, dtype=torch.int32, device="cuda")))
    elif kind == "bpe_ragged":
        off = _offsets_of(_long_read_lengths(rows, gen))
        total = int(off[-1])
        enc, _ = _bpe(case["vocab"])
        s.update(enc=enc, data=_bpe_bases(total, case["vocab"], gen, n_rate=0.002), off=off,
                 longest=int((off[1:] - off[:-1]).max()), lut=torch.from_numpy(_char_lut()[0]).cuda(),
                 tok=torch.empty(total, dtype=torch.int32, device="cuda"),
                 lengths=torch.empty(rows, dtype=torch.int32, device="cuda"),
                 char_ids=torch.empty(total, dtype=torch.int32, device="cuda"),
                 char_mask=torch.empty(total, dtype=torch.uint8, device="cuda"),
                 # (room for a token per base: what lies behind the packed tokens stays zero)
                 out=(torch.zeros(total, dtype=torch.int32, device="cuda"),
                      torch.zeros(rows + 1, dtype=torch.int64, device="cuda"),
                      torch.zeros(total, dtype=torch.uint8, device="cuda")))
    elif kind == "kmer_rows":
        width = _kmer_width(case)
        s.update(enc=_kmer6(), data=_uniform_bases(rows, case["length"], gen, n_runs=0.005),
                 off=_even_offsets(rows, case["length"]), width=width,
                 out=(torch.empty((rows, width), dtype=torch.int32, device="cuda"),
                      torch.empty((rows, width), dtype=torch.uint8, device="cuda"),
                      torch.empty(rows, dtype=torch.int32, device="cuda"),
                      torch.empty(rows, dtype=torch.int32, device="cuda"),
                      torch.empty(1, dtype=torch.int32, device="cuda")))
    elif kind == "kmer_packed":
        off = _offsets_of(_read_lengths(rows, gen))
        total = int(off[-1])
        s.update(enc=_kmer6(), data=_uniform_bases(1, total, gen, n_rate=0.001), off=off,
                 out=(torch.zeros(total, dtype=torch.int32, device="cuda"),
                      torch.zeros(rows + 1, dtype=torch.int64, device="cuda"),
                      torch.zeros(total, dtype=torch.uint8, device="cuda"),
                      torch.zeros(rows, dtype=torch.int32, device="cuda"),
                      torch.zeros(rows, dtype=torch.int32, device="cuda")))
    else:
        lut, pad = _char_lut()
        total = rows * case["length"]
        s.update(enc=encoders.CharEncoder(lut, pad), data=_uniform_bases(rows, case["length"], gen, n_rate=0.001))
        if kind == "char_rows":
            s.update(ids=torch.empty(total, dtype=torch.int32, device="cuda"),
                     mask=torch.empty(total, dtype=torch.uint8, device="cuda"))
        else:
            s.update(weight=torch.randn((16, case["dim"]), generator=gen, device="cuda").bfloat16(),
                     out=torch.empty((total, case["dim"]), dtype=torch.bfloat16, device="cuda"))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "strings":
        if case["api"] == "ids":
            return s["dn"].encode_batch_to_ids(s["seqs"])
        return s["dn"].encode_batch_with_padding(s["seqs"], s["dn"].token_len, pad_to_max=True)
    if kind in ("bpe_rows", "bpe_reads"):
        return s["enc"].encode_padded(s["data"], s["off"], s["longest"], s["width"], s["pad"], out=s["out"],
                                      tok_tmp=s["tok"])
    if kind == "bpe_ragged":
        tok, lengths, char_ids, char_mask = s["enc"].encode_with_chars(
            s["data"], s["off"], s["longest"], s["lut"], tok_tmp=s["tok"], lengths=s["lengths"],
            char_ids=s["char_ids"], char_mask=s["char_mask"])
        ids, offsets, mask = encoders.pack_ragged(tok, s["off"], lengths, out=s["out"])
        return ids, offsets, mask, lengths, char_ids, char_mask
    if kind == "kmer_rows":
        return s["enc"].encode_padded(s["data"], s["off"], s["width"], fill_to=s["width"], out=s["out"])
    if kind == "kmer_packed":
        return s["enc"].encode_packed(s["data"], s["off"], want_mask=True, out=s["out"])
    if kind == "char_rows":
        return s["enc"].encode_packed(s["data"], row_len=case["length"], want_mask=True, ids=s["ids"], mask=s["mask"])
    return s["enc"].embed_packed(s["data"], s["weight"], row_len=case["length"], out=s["out"])


def work(case):
    """Each base read once, each id, mask byte and length written once (int64 ids on the host count
    as what crosses the bus); no arithmetic beyond table lookups."""
    kind, rows = case["kind"], case["rows"]
    if kind == "strings":
        cell = 8.0 if case["api"] == "ids" else (2.0 if case["tok"] == "char" else 3.0)
        return {"bytes": 0.95 * rows * case["length"] + 8.0 * (rows + 1) + rows * _strings_width(case) * cell, "flops": 0.0}
    if kind in ("bpe_rows", "bpe_reads"):
        bases = rows * (case["length"] if kind == "bpe_rows" else 200)
        cell = (4 if case["ids"] == "int32" else 8) + 1
        return {"bytes": bases + 8.0 * (rows + 1) + float(rows) * _bpe_width(case) * cell + 4.0 * rows, "flops": 0.0}
    if kind == "bpe_ragged":
        bases = rows * 2920.0
        return {"bytes": 6.0 * bases + 5.0 * bases / 5.2 + 20.0 * rows, "flops": 0.0}
    if kind == "kmer_rows":
        return {"bytes": float(rows) * (case["length"] + 5 * _kmer_width(case) + 16), "flops": 0.0}
    if kind == "kmer_packed":
        return {"bytes": rows * (200.0 + 5.0 * 36 + 24), "flops": 0.0}
    if kind == "char_rows":
        return {"bytes": 6.0 * rows * case["length"], "flops": 0.0}
    return {"bytes": float(rows) * case["length"] * (1 + 2 * case["dim"]), "flops": 0.0}


def tolerance(case):
    return "exact"
