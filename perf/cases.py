"""Timed cases of the text-deduplication path: what a user has the framework do, through the calls of cudf_amd.nvtext.

A case is a dict: `op` names the call, `rows` and `mean` (bytes a row on average) the size of the column, `text` what it
holds, `skip` the rows in front of the view (a column handed over in chunks is a view), `nulls` the share of null rows,
`long_offsets` 64-bit offsets, and then the arguments of the call.  Text is made on the GPU: words drawn by Zipf's law
(exponent 1.1) from a word list of cudf_amd.datagen, single spaces between them, row lengths lognormal.  The rows' lengths
are those of the case, in an order that the seed draws, so that results of two seeds are of one size; the words are the
seed's, except where they decide the size of the result (token ids, normalized text): there whole rows trade places.
"""
import functools
import math

import numpy as np
import torch

from cudf_amd import datagen, nvtext

DEVICE = "cuda"


def listed():
    return [
        # a request to a serving process: a few dozen short texts to the token ids of a BERT-sized vocabulary
        dict(name="tokenize_request", op="tokenize", text="ascii", rows=29, mean=180, sigma=0.6, skip=0, nulls=0.0, long_offsets=False, max_words=128),
        # titles or queries, a chunk of a larger column, some of them null, no word limit
        dict(name="tokenize_titles", op="tokenize", text="ascii", rows=32768, mean=120, sigma=0.4, skip=17, nulls=0.02, long_offsets=False, max_words=0),
        # the benchmark's rows (256 bytes on average, 15 % of the words unknown, 128 words at most), half its number
        dict(name="tokenize_corpus", op="tokenize", text="ascii", rows=2000003, mean=256, sigma=0.6, skip=0, nulls=0.0, long_offsets=False, max_words=128),
        # text of several scripts over the vocabulary of 250,000 entries, 64-bit offsets
        dict(name="tokenize_utf8", op="tokenize", text="mixed", rows=1200001, mean=512, sigma=0.6, skip=0, nulls=0.0, long_offsets=True, max_words=256),
        # documents that arrive in small batches, each to be signed before the next comes
        dict(name="minhash_batch", op="minhash", text="lexicon", rows=999, mean=2048, sigma=0.8, skip=0, nulls=0.0, long_offsets=False, bits=32, width=5, params=256),
        # a shard of a corpus of documents
        dict(name="minhash_corpus", op="minhash", text="lexicon", rows=400000, mean=2048, sigma=0.8, skip=0, nulls=0.0, long_offsets=False, bits=32, width=5, params=256),
        # books and reports: long rows of very different lengths, a tenth of them null
        dict(name="minhash64_long", op="minhash", text="lexicon", rows=20011, mean=16384, sigma=1.5, skip=0, nulls=0.1, long_offsets=False, bits=64, width=5, params=128),
        # the second half of the UTF-8 pipeline: short rows of several scripts, signed with 64-bit hashes
        dict(name="minhash64_utf8", op="minhash", text="mixed", rows=1000003, mean=512, sigma=0.6, skip=0, nulls=0.0, long_offsets=True, bits=64, width=8, params=64),
        # documents that are split into words already, signed over runs of words
        dict(name="minhash_ngrams_words", op="ngrams", text="lexicon", rows=200001, mean=2048, sigma=0.8, skip=0, nulls=0.0, long_offsets=False, bits=32, ngrams=5, params=256),
        # candidate pairs of near-duplicates, checked exactly
        dict(name="jaccard_pairs", op="jaccard", text="lexicon", rows=250001, mean=2048, sigma=0.8, skip=0, nulls=0.0, long_offsets=False, width=5),
        # the step before the tokenizer in a serving process
        dict(name="normalize_request", op="normalize", text="mixed", rows=61, mean=300, sigma=0.6, skip=0, nulls=0.0, long_offsets=False, lower=True),
        # the same for a shard of a corpus
        dict(name="normalize_utf8", op="normalize", text="mixed", rows=1500001, mean=512, sigma=0.6, skip=0, nulls=0.0, long_offsets=True, lower=True),
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["tokenize", "tokenize", "minhash", "minhash", "ngrams", "jaccard", "normalize"])
    bits = rng.choice([32, 64])
    if op == "tokenize" or op == "normalize":
        # 5 KB .. 600 MB, rows of a title to rows of a page
        case = dict(op=op, text=rng.choice(["ascii", "mixed"]), mean=_log_between(rng, 60, 2000), sigma=0.6)
        total = _log_between(rng, 5_000, 600_000_000)
    elif op == "minhash":
        # 200 KB .. 800 MB at 256 parameters of 32 bits, less where a window costs more
        params = rng.choice([26, 64, 100, 128, 256, 260])
        case = dict(op=op, text=rng.choice(["lexicon", "mixed"]), mean=_log_between(rng, 300, 16384), sigma=0.8, bits=bits,
                    width=rng.choice([4, 5, 8, 12, 24]), params=params)
        total = _log_between(rng, 200_000, min(800_000_000, 800_000_000 * 256 // (params * (1 if bits == 32 else 6))))
    elif op == "ngrams":
        params = rng.choice([64, 128, 256])
        case = dict(op=op, text="lexicon", mean=_log_between(rng, 300, 16384), sigma=0.8, bits=bits, ngrams=rng.choice([2, 3, 5, 8]), params=params)
        total = _log_between(rng, 200_000, 400_000_000)
    else:
        case = dict(op=op, text=rng.choice(["lexicon", "mixed"]), mean=_log_between(rng, 100, 8000), sigma=0.8, width=rng.choice([3, 5, 8]))
        total = _log_between(rng, 50_000, 400_000_000)
    case["rows"] = max(7, total // case["mean"])
    case["skip"] = rng.choice([0, 0, 0, rng.randrange(1, 100)])
    case["nulls"] = rng.choice([0.0, 0.0, 0.05]) if op != "ngrams" else 0.0
    case["long_offsets"] = rng.choice([False, True])
    if op == "tokenize":
        case["max_words"] = rng.choice([0, 32, 128, 256])
    if op == "normalize":
        case["lower"] = rng.choice([True, False])
    return case


# ------------------------------------------------------------------ text

@functools.lru_cache(maxsize=None)
def _vocabulary(text):
    kind, size, seed = {"ascii": (datagen.VOCAB_BERT, 30522, 1001), "lexicon": (datagen.VOCAB_LEXICON, 50000, 1003),
                        "mixed": (datagen.VOCAB_MULTILINGUAL, 250000, 1005)}[text]
    return datagen.make_vocab(kind, size, seed)


@functools.lru_cache(maxsize=None)
def _words(text):
    """The words that text of this kind is made of, on the GPU: their bytes one after the other, where each begins, how
    long it is, and the cumulated probability of each (words that the vocabulary does not hold among them)."""
    v = _vocabulary(text)
    raw = v.chars.tobytes()
    entries = [raw[v.offsets[i]: v.offsets[i + 1]] for i in range(v.size)]
    entries = [e for e in entries if len(e) > 1 and not e.startswith((b"##", b"["))]

    def zipf(n):
        p = 1.0 / np.arange(1, n + 1) ** 1.1
        return p / p.sum()

    rnd = np.random.default_rng(99)
    letters = [bytes(rnd.integers(97, 123, int(n), dtype=np.uint8)) for n in rnd.integers(3, 11, 40000)]
    if text == "lexicon":
        groups = [(entries, 1.0, True)]
    elif text == "ascii":
        groups = [(entries, 0.85, True), (letters, 0.15, False)]
    else:
        # seven words of ten ASCII, two with accents, one of Chinese characters; punctuation marks stand between them, and
        # one word in ten is unknown
        strange = []
        for n in rnd.integers(3, 11, 20000):
            strange.append("".join(chr(c) for c in np.where(rnd.random(n) < 0.33, rnd.integers(0xE0, 0x100, n), rnd.integers(97, 123, n))).encode())
        for n in rnd.integers(1, 5, 10000):
            strange.append("".join(chr(c) for c in rnd.integers(0x4E00, 0x4E00 + 3500, n)).encode())
        plain = [e for e in entries if e.isascii()]
        accents = [e for e in entries if not e.isascii() and e[0] < 0xE0]
        chinese = [e for e in entries if e[0] >= 0xE0]
        marks = [m.encode() for m in ".,;:!?'\"()-"]
        groups = [(plain, 0.58, True), (accents, 0.165, True), (chinese, 0.083, True), (letters, 0.064, False), (strange, 0.028, False), (marks, 0.08, False)]
    words, probs = [], []
    for g, share, ranked in groups:
        words += g
        probs.append(share * (zipf(len(g)) if ranked else np.full(len(g), 1.0 / len(g))))
    lens = np.array([len(w) for w in words], np.int64)
    probs = np.concatenate(probs)
    table = torch.from_numpy(np.frombuffer(b"".join(words), np.uint8).copy()).to(DEVICE)
    starts = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)[:-1]])).to(DEVICE)
    return table, starts, torch.from_numpy(lens).to(DEVICE), torch.from_numpy(np.cumsum(probs)).to(DEVICE), float((lens * probs).sum())


CHUNK = 1 << 24  # words whose bytes are written at a time


def _draw_words(text, n, gen):
    cdf = _words(text)[3]
    ids = torch.empty(n, dtype=torch.int32, device=DEVICE)
    for i in range(0, n, CHUNK):
        k = min(CHUNK, n - i)
        ids[i: i + k] = torch.searchsorted(cdf, torch.rand(k, generator=gen, device=DEVICE, dtype=torch.float64)).clamp_(max=cdf.numel() - 1)
    return ids


def _words_per_row(case, gen):
    """Number of words of every row (0: null or empty), and which rows are null."""
    n = case["rows"] + case["skip"]
    mu = math.log(case["mean"]) - 0.5 * case["sigma"] ** 2
    target = torch.exp(mu + case["sigma"] * torch.randn(n, generator=gen, device=DEVICE, dtype=torch.float64)).clamp_(max=64.0 * case["mean"])
    per = torch.round(target / (_words(case["text"])[4] + 1.0)).to(torch.int64).clamp_(min=1)
    u = torch.rand(n, generator=gen, device=DEVICE)
    null = u < case["nulls"]
    per[u < 1.1 * case["nulls"]] = 0  # some rows are empty where some are null
    return per, null


def _write(text, ids, last, cased, gen):
    """The bytes of the words, a space after each that is not the last of its row, and where each word begins."""
    table, starts, lens = _words(text)[:3]
    n = ids.numel()
    begin = torch.zeros(n + 1, dtype=torch.int64, device=DEVICE)
    for i in range(0, n, CHUNK):
        begin[i + 1: i + CHUNK + 1] = lens[ids[i: i + CHUNK].long()] + (~last[i: i + CHUNK]).long()
    begin = torch.cumsum(begin, 0)
    chars = torch.full((int(begin[-1]),), 0x20, dtype=torch.uint8, device=DEVICE)
    for i in range(0, n, CHUNK):
        which = ids[i: i + CHUNK].long()
        size, at = lens[which], begin[i: i + CHUNK + 1][: which.numel()]
        total = int(size.sum())
        within = torch.arange(total, device=DEVICE) - torch.repeat_interleave(torch.cumsum(size, 0) - size, size, output_size=total)
        source = torch.repeat_interleave(starts[which], size, output_size=total) + within
        chars[torch.repeat_interleave(at, size, output_size=total) + within] = table[source]
    if cased:  # one word in eight begins with a capital letter
        at = begin[:-1][torch.rand(n, generator=gen, device=DEVICE) < 0.125]
        first = chars[at]
        chars[at] = torch.where((first >= 97) & (first <= 122), first - 32, first)
    return chars, begin


def _column(case, per, null, ids, cased, gen):
    n = per.numel()
    ends = torch.cumsum(per, 0)
    last = torch.zeros(ids.numel(), dtype=torch.bool, device=DEVICE)
    last[ends[per > 0] - 1] = True
    chars, begin = _write(case["text"], ids, last, cased, gen)
    offsets = torch.zeros(n + 1, dtype=torch.int64, device=DEVICE)
    offsets[1:] = begin[ends]
    mask, view_nulls = None, int(null[case["skip"]:].sum())
    if view_nulls:
        bits = torch.zeros((n + 31) // 32 * 32, dtype=torch.int64, device=DEVICE)
        bits[:n] = (~null).long()
        mask = (bits.view(-1, 32) << torch.arange(32, device=DEVICE)).sum(1).to(torch.int32)
    if not case["long_offsets"]:
        offsets, begin = offsets.to(torch.int32), begin.to(torch.int32)
    return nvtext.DeviceStringsColumn(chars, offsets, mask, case["rows"], case["skip"], view_nulls), begin, ends


def _vocabulary_column(text):
    return nvtext.DeviceStringsColumn.from_host(_vocabulary(text), DEVICE)


def _generator(seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    return gen


def _rows(case, gen):
    """Words of every row, which rows are null, the words one row after the other."""
    of_case = _generator(case["rows"] + case["mean"])
    per, null = _words_per_row(case, of_case)
    n, skip = per.numel(), case["skip"]
    order = torch.cat([torch.arange(skip, device=DEVICE), skip + torch.randperm(n - skip, generator=gen, device=DEVICE)])
    total = int(per.sum())
    if case["op"] not in ("tokenize", "normalize"):
        return per[order], null[order], _draw_words(case["text"], total, gen)
    ids = _draw_words(case["text"], total, of_case)
    first = (torch.cumsum(per, 0) - per)[order]
    per, null = per[order], null[order]
    shift = torch.repeat_interleave(first - (torch.cumsum(per, 0) - per), per, output_size=total)
    return per, null, ids[shift + torch.arange(total, device=DEVICE)]


def prepare(case, seed):
    gen = _generator(seed)
    per, null, ids = _rows(case, gen)
    op = case["op"]
    column, begin, ends = _column(case, per, null, ids, op == "normalize", gen)
    state = dict(case=case, column=column)
    if op == "tokenize":
        state["vocabulary"] = nvtext.WordPieceVocabulary(_vocabulary_column(case["text"]))
    elif op == "normalize":
        special = nvtext.DeviceStringsColumn.from_host(nvtext.HostStringsColumn.from_pylist(["[CLS]", "[SEP]", "[PAD]", "[UNK]", "[MASK]"]), DEVICE)
        state["normalizer"] = nvtext.CharacterNormalizer(case["lower"], special)
    elif op == "jaccard":
        # the other document of the pair: the same one with none to six tenths of its words drawn anew
        share = torch.repeat_interleave(0.6 * torch.rand(per.numel(), generator=gen, device=DEVICE), per, output_size=ids.numel())
        anew = torch.rand(ids.numel(), generator=gen, device=DEVICE) < share
        state["other"] = _column(case, per, null, torch.where(anew, _draw_words(case["text"], ids.numel(), gen), ids), False, gen)[0]
    else:
        a, b = datagen.make_params(case["params"], case["bits"], seed)
        signed = np.int32 if case["bits"] == 32 else np.int64
        state["a"], state["b"] = (torch.from_numpy(x.view(signed)).to(DEVICE) for x in (a, b))
    if op == "ngrams":
        # the words as list elements, each with the space that follows it
        child = nvtext.DeviceStringsColumn(column.chars, begin, None, ids.numel(), 0, 0)
        lists = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEVICE), ends]).to(torch.int32)
        state["lists"] = nvtext.DeviceListStringsColumn(lists, child, None, case["rows"], case["skip"], 0)
    return state


# ------------------------------------------------------------------ calls

def run(state):
    case, column = state["case"], state["column"]
    op = case["op"]
    if op == "tokenize":
        out = nvtext.wordpiece_tokenize(column, state["vocabulary"], case["max_words"])
    elif op == "minhash":
        call, seed = (nvtext.minhash, 42) if case["bits"] == 32 else (nvtext.minhash64, 7)
        out = call(column, seed, state["a"], state["b"], case["width"])
    elif op == "ngrams":
        call, seed = (nvtext.minhash_ngrams, 42) if case["bits"] == 32 else (nvtext.minhash64_ngrams, 7)
        out = call(state["lists"], case["ngrams"], seed, state["a"], state["b"])
    elif op == "jaccard":
        out = nvtext.jaccard_index(column, state["other"], case["width"])
        return dict(values=out.data, mask=_mask(out), nulls=out.null_count)
    else:
        out = nvtext.normalize_characters(column, state["normalizer"])
        return dict(chars=out.chars, offsets=out.offsets, mask=_mask(out), nulls=out.null_count)
    return dict(offsets=out.offsets, child=out.child, mask=_mask(out), nulls=out.null_count)


def _mask(out):
    """The validity words, without what pads their buffer."""
    if out.mask is None:
        return None
    return out.mask[: (out.size + 31) // 32 * 4 // out.mask.element_size()]


def work(case):
    """Bytes: the column (and its partner) read once, the result written once.  Operations: where every window meets every
    parameter, a multiplication and an addition for each of these products; else one for every byte."""
    rows, chars = case["rows"], case["rows"] * case["mean"]
    column = chars + (rows + 1) * (8 if case["long_offsets"] else 4)
    op = case["op"]
    if op == "tokenize":
        return {"bytes": column + 4 * (rows + 1) + 4 * chars * 0.2, "flops": chars}
    if op == "normalize":
        return {"bytes": column + 4 * (rows + 1) + chars * 1.05, "flops": chars}
    if op == "jaccard":
        return {"bytes": 2 * column + 4 * rows, "flops": 2 * chars}
    items = chars
    if op == "ngrams":
        items = chars / 6.3
        column += items * (8 if case["long_offsets"] else 4)
    return {"bytes": column + 4 * (rows + 1) + rows * case["params"] * case["bits"] // 8, "flops": 2 * items * case["params"]}


def tolerance(case):
    """Token ids, hashes, bytes and a quotient of two counts: every correct implementation gives the same."""
    return "exact"
