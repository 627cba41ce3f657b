"""The sizes at which a kernel hands over to another, or a loop to its remainder, against the host oracle, bit for bit."""
import numpy as np
import pytest

from cudf_amd.arrow_host import HostListStringsColumn, HostStringsColumn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nv():
    import torch
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from cudf_amd import nvtext
    return nvtext


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def dev(nv, host):
    return nv.DeviceStringsColumn.from_host(host)


def random_text(rng, n, alphabet=b"abcdefghijklmnopqrstuvwxyz"):
    return bytes(rng.choice(np.frombuffer(alphabet, np.uint8), n))


JACCARD_SLOTS = (1024, 4096, 7008, 15488, 29440)  # of the sets in LDS


@pytest.mark.parametrize("width", [2, 7, 40])
def test_jaccard_sets_and_shares(nv, orc, width):
    """Pairs of the most bytes that each set takes (4/5 of 1024, 4096, 7008, 15488 and 29440 slots) and of one more, rows one window
    around whole units of 64, and of very different lengths, so that a wavefront's share ends in the one or the other."""
    rng = np.random.default_rng(width)
    sizes = [n * 4 // 5 + d for n in JACCARD_SLOTS for d in (0, 1)]
    lens = [(n // 2 + d, n - n // 2 - d) for n in sizes for d in (0, 1, n // 3)]
    lens += [(64 * k + width - 1 + d, 64 * m + width - 1 + e) for k, m in ((1, 0), (4, 5), (9, 23), (31, 16)) for d in (-1, 0, 1) for e in (-1, 0, 1)]
    left = [random_text(rng, max(n, 0)).decode() for n, _ in lens]
    right = [(a[: m // 2] + random_text(rng, max(m, 0) - len(a[: m // 2])).decode()) for a, (_, m) in zip(left, lens)]
    h1, h2 = HostStringsColumn.from_pylist(left), HostStringsColumn.from_pylist(right)
    got, exp = nv.jaccard_index(dev(nv, h1), dev(nv, h2), width).to_host(), orc.jaccard_index(h1, h2, width, nthreads=8)
    assert np.array_equal(got.values.view(np.uint32), exp.values.view(np.uint32))


def jaccard_set(size):
    """The slots of the set that a pair of so many bytes gets, and the parts that it is cut into."""
    if size <= 1024 * 4 // 5:
        return 1024, 1
    tier = next((n for n in JACCARD_SLOTS if size <= n * 4 // 5), None)
    return (29440, -(-size // 20_000)) if tier is None else (min(tier, max(1024, (2 * size + 63) // 32 * 32)), 1)


def jaccard_places(words, buckets, parts):
    """Where windows of four bytes belong in a set, which step they take from a bucket that is full to the next, and in which part
    they are: by the top and the low bits of products of their hash (MurmurHash3_x86_32, seed 0, without the final mix)."""
    def top(v, n):
        return v.astype(np.uint64) * np.uint64(n) >> np.uint64(32)
    with np.errstate(over="ignore"):
        k = words * np.uint32(0xCC9E2D51)
        k = (k << np.uint32(15) | k >> np.uint32(17)) * np.uint32(0x1B873593)
        h = ((k << np.uint32(13) | k >> np.uint32(19)) * np.uint32(5) + np.uint32(0xE6546B64)) ^ np.uint32(4)
        p = h * np.uint32(0x9E3779B1)
        return top(p, buckets), (p & np.uint32(15)) * 2 + 1, top((h ^ h >> np.uint32(15)) * np.uint32(0x85EBCA6B), parts)


def furthest_from_home(text, buckets, parts):
    """Steps from the home of a window of four bytes to where it finds a place, the most of part 0."""
    windows = np.unique(text[:-3] | text[1:-2].astype(np.uint32) << 8 | text[2:-1].astype(np.uint32) << 16 | text[3:].astype(np.uint32) << 24)
    home, step, part = jaccard_places(windows, buckets, parts)
    filled, furthest = [0] * buckets, 0
    for b, s in zip(home[part == 0].tolist(), step[part == 0].tolist()):
        far = 0
        while filled[b] == 4 and far < 500:
            b, far = (b + s) % buckets, far + 1
        filled[b] += 1
        furthest = max(furthest, far)
    return furthest


@pytest.mark.parametrize("count, slots, parts", [(90, 1024, 1), (190, 1024, 1), (600, 4096, 1), (1000, 7008, 1), (2000, 15488, 1), (5000, 29440, 1), (7000, 29440, 2)])
def test_jaccard_values_of_neighbouring_buckets(nv, orc, count, slots, parts):
    """Words that belong in one bucket of their set, or in a few side by side, and take the same steps from there: 90 that find a
    place within the 64 buckets that a packed set looks at, and so many in sets of every size that some do not, so that the pair
    is done once more with a plain set, or, where one of its parts has them all, that part is cut in two; among pairs that are not."""
    rng = np.random.default_rng(count)
    assert jaccard_set(4 * count) == (slots, parts)
    letters = np.concatenate([np.arange(65, 91), np.arange(97, 123)]).astype(np.uint32)
    words = (letters[:, None, None, None] | letters[:, None, None] << 8 | letters[:, None] << 16 | letters << 24).astype(np.uint32).ravel()
    home, step, part = jaccard_places(words, slots // 4, parts)
    from_there = np.flatnonzero((part == 0) & (home >= 77) & (step == 1))
    near = from_there[np.argsort(home[from_there], kind="stable")][:count]
    text = rng.permutation(words[near]).view(np.uint8).reshape(-1, 4)
    assert (furthest_from_home(text.ravel(), slots // 4, parts) >= 64) == (count != 90)
    row = lambda pick: bytes(text[pick].ravel()).decode()
    n = len(text)
    left = [row(np.arange(n * 3 // 4)), "some other text", row(np.arange(n // 2))] * 3
    right = [row(np.arange(n * 3 // 4, n)), "another text", row(np.arange(n // 2, n))] * 3
    h1, h2 = HostStringsColumn.from_pylist(left), HostStringsColumn.from_pylist(right)
    got, exp = nv.jaccard_index(dev(nv, h1), dev(nv, h2), 4).to_host(), orc.jaccard_index(h1, h2, 4, nthreads=8)
    assert np.array_equal(got.values.view(np.uint32), exp.values.view(np.uint32))


@pytest.mark.parametrize("copies", [1, 20, 55, 400])
def test_jaccard_lists_of_few_and_many_pairs(nv, orc, copies):
    """Pairs for every set and in parts, side by side, some of which find no place in theirs: fewer than there are CUs, so many
    that a workgroup has several of them at a time, and so many that the sets have kernels of their own."""
    rng = np.random.default_rng(copies)
    letters = np.concatenate([np.arange(65, 91), np.arange(97, 123)]).astype(np.uint32)
    words = (letters[:, None, None, None] | letters[:, None, None] << 8 | letters[:, None] << 16 | letters << 24).astype(np.uint32).ravel()
    rows = [random_text(rng, n).decode() for n in (10, 700, 900, 2500, 3276, 3277, 5000, 5606, 5607, 9000, 12_390, 12_391, 20_000)]
    rows += [random_text(rng, n).decode() for n in (23_552, 23_553, 61_000)] if copies < 100 else []
    for count, slots in ((600, 4096), (1000, 7008), (2000, 15488)):
        home, step, _ = jaccard_places(words, slots // 4, 1)
        from_there = np.flatnonzero((home >= 77) & (step == 1))
        near = from_there[np.argsort(home[from_there], kind="stable")][:count]
        rows.append(bytes(rng.permutation(words[near]).view(np.uint8)).decode())
    left, right = [t[: len(t) // 3] for t in rows], [t[len(t) // 4:] for t in rows]
    h1, h2 = (HostStringsColumn.from_pylist(side) for side in (left, right))
    exp = orc.jaccard_index(h1, h2, 4, nthreads=8).values.view(np.uint32)
    h1, h2 = (HostStringsColumn.from_pylist(side * copies) for side in (left, right))
    for _ in range(2):
        got = nv.jaccard_index(dev(nv, h1), dev(nv, h2), 4).to_host()
        assert np.array_equal(got.values.view(np.uint32), np.tile(exp, copies))


@pytest.mark.parametrize("width", [2, 7, 40])
def test_jaccard_pair_sizes(nv, orc, width):
    """Pairs of the most bytes that each set takes (4/5 of its slots) and of one more, around one
    and several parts of 20,000 bytes, and around sixteen parts; no window repeats, so the sets are as full as they get."""
    rng = np.random.default_rng(width)
    sizes = [n * 4 // 5 + d for n in JACCARD_SLOTS for d in (0, 1)]
    sizes += [40_000, 40_001, 60_001, 320_000, 320_001, 1, 2, 63, 64, 65]
    left, right = [], []
    for n in sizes:
        for share in (0.0, 0.37, 1.0):
            n1 = int(n * share)
            text = random_text(rng, n)
            left.append(text[:n1])
            right.append(text[n1:] if share != 0.37 else text[: n1 // 2] + text[n1 + n1 // 2:])
    h1, h2 = (HostStringsColumn.from_pylist([t.decode() for t in rows]) for rows in (left, right))
    got, exp = nv.jaccard_index(dev(nv, h1), dev(nv, h2), width).to_host(), orc.jaccard_index(h1, h2, width, nthreads=8)
    assert np.array_equal(got.values.view(np.uint32), exp.values.view(np.uint32))


@pytest.mark.parametrize("copies, sizes", [(1, (320_001, 640_000, 640_001)), (30_000, (700,) * 4 + (23_600,)), (33_000, (23_600,)), (150_000, (20, 2000))])
def test_jaccard_many_parts(nv, orc, copies, sizes):
    """Pairs of 17 and of the most parts (32), and of more; columns whose lists the host does not look at (more than 131,072 pairs), and
    more parts than have a place on their list (65,536)."""
    rng = np.random.default_rng(copies)
    sizes = list(sizes) + ([23_600, 50_000] if copies == 150_000 else [])
    rows = [random_text(rng, n).decode() for n in sizes]
    left, right = [t[: len(t) // 3] for t in rows], [t[len(t) // 4: len(t) // 4 * 3] for t in rows]
    left[-1], right[-1] = rows[-1][: sizes[-1] // 2], rows[-1][sizes[-1] // 2:]
    times = [copies] * len(rows) if copies < 150_000 else [copies, 100, 50, 20]
    h1, h2 = (HostStringsColumn.from_pylist(side) for side in (left, right))
    exp = orc.jaccard_index(h1, h2, 4, nthreads=8).values.view(np.uint32)
    h1, h2 = (HostStringsColumn.from_pylist([t for t, n in zip(side, times) for _ in range(n)]) for side in (left, right))
    got = nv.jaccard_index(dev(nv, h1), dev(nv, h2), 4).to_host()
    assert np.array_equal(got.values.view(np.uint32), np.repeat(exp, times))


@pytest.fixture
def filled_memory(monkeypatch):
    """Results and temporaries hold ones in all bits (NaN) when a call gets them: what it leaves unwritten cannot pass for an answer."""
    import torch
    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *args, **kw: empty(*args, **kw).fill_(255) if kw.get("dtype") == torch.uint8 else empty(*args, **kw))


@pytest.mark.parametrize("copies, others", [(33_000, {15_000: 300}), (33_000, {12_400: 2000, 21_000: 3000}),
                                            (34_000, {500: 2000, 2000: 300, 4000: 300, 9000: 300, 15_000: 300, 61_000: 10, 640_001: 2}),
                                            (33_000, {700: 1000, 2500: 9000, 5000: 2000, 9000: 2000, 12_391: 700})])
def test_jaccard_more_parts_than_their_list_beside_other_pairs(nv, orc, filled_memory, copies, others):
    """Columns of at most 131,072 pairs with more parts than have a place on their list (65,536), and more pieces of other work than
    there are CUs: pairs of the largest set, pairs for every set and in global memory, and so many of the smaller ones that the sets have
    kernels of their own."""
    rng = np.random.default_rng(copies)
    times = {23_600: copies, **others}
    rows = [random_text(rng, n).decode() for n in times]
    left, right = [t[: len(t) // 3] for t in rows], [t[len(t) // 4:] for t in rows]
    left[0], right[0] = rows[0][:11_800], rows[0][11_800:]
    exp = orc.jaccard_index(*(HostStringsColumn.from_pylist(side) for side in (left, right)), 4, nthreads=8).values.view(np.uint32)
    order = rng.permutation(np.repeat(np.arange(len(rows)), list(times.values())))
    h1, h2 = (HostStringsColumn.from_pylist([side[i] for i in order]) for side in (left, right))
    got = nv.jaccard_index(dev(nv, h1), dev(nv, h2), 4).to_host()
    assert np.array_equal(got.values.view(np.uint32), exp[order])


@pytest.mark.parametrize("times", [{9000: 1536}, {9000: 1537}, {2500: 4 * 1536}, {2500: 4 * 1536 + 1}, {23_600: 32_768, 15_000: 300, 2500: 10},
                                   {20: 131_000, 2500: 30, 9000: 20, 15_000: 12, 61_000: 9, 640_001: 1}, {20: 131_000, 2500: 30, 9000: 21, 15_000: 12, 61_000: 9, 640_001: 1}])
@pytest.mark.parametrize("nulls", [False, True])
def test_jaccard_where_the_ways_part(nv, orc, filled_memory, times, nulls):
    """Pieces of work up to which the sets share a launch (1,536) and one more, parts of which the last has the last place on their
    list (65,536), pairs up to which the host looks at the lists (131,072) and one more; null rows in one column or the other, and a view."""
    rng = np.random.default_rng(sum(times.values()))
    rows = [random_text(rng, n).decode() for n in times]
    left, right = [t[: len(t) // 3] for t in rows], [t[len(t) // 4:] for t in rows]
    if 23_600 in times:
        left[0], right[0] = rows[0][:11_800], rows[0][11_800:]
    exp = orc.jaccard_index(*(HostStringsColumn.from_pylist(side) for side in (left, right)), 4, nthreads=8).values.view(np.uint32)
    order = rng.permutation(np.repeat(np.arange(len(rows)), list(times.values())))
    valid = np.ones((2, len(order)), bool)
    if nulls:
        valid[0, 3::7] = valid[1, 5::11] = False
    h1, h2 = (HostStringsColumn.from_pylist(["skip", "these"] + [side[i] if v else None for i, v in zip(order, ok)]) for side, ok in zip((left, right), valid))
    n, both = len(order), valid[0] & valid[1]
    got = nv.jaccard_index(*(dev(nv, h).slice(2, n + 2, int((~ok).sum())) for h, ok in zip((h1, h2), valid)), 4).to_host()
    assert got.null_count == int((~both).sum())
    assert np.array_equal(got.values.view(np.uint32)[both], exp[order][both])


def mixed_rows(rng, lens, nulls=()):
    """Rows of these lengths as a column; the rows named in `nulls` are null (and empty)."""
    lens = np.array(lens, np.int64)
    lens[list(nulls)] = 0
    offsets = np.concatenate([[0], np.cumsum(lens)])
    chars = rng.choice(np.frombuffer(b"abcdefgh ", np.uint8), int(offsets[-1]))
    mask = None
    if nulls:
        bits = np.ones((len(lens) + 31) // 32 * 32, np.uint8)
        bits[len(lens):] = 0
        bits[list(nulls)] = 0
        mask = np.packbits(bits, bitorder="little").view(np.uint32)
    return HostStringsColumn(chars, offsets.astype(np.int32), mask, len(lens), 0, len(nulls))


def params(rng, count, bits):
    dtype = np.uint32 if bits == 32 else np.uint64
    return rng.integers(1, 2**bits, count, dtype=np.uint64).astype(dtype), rng.integers(0, 2**bits, count, dtype=np.uint64).astype(dtype)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("count", [1, 33, 64, 128, 260, 700])
def test_minhash_parts_of_rows(nv, orc, bits, count):
    """Rows one byte around one part and several, parts of 256 bytes (little text) and more (33 MB), the parameters in one
    chunk and in several, null and empty rows between them."""
    rng = np.random.default_rng(count)
    edges = [0, 1, 4, 5, 63, 64, 65, 255, 256, 257, 511, 513, 4095, 4096, 4097, 8192, 8193, 20_000]
    call, ref = (nv.minhash, orc.minhash) if bits == 32 else (nv.minhash64, orc.minhash64)
    a, b = params(rng, count, bits)
    for more in ([], [3_000_000] * 11 if count == 64 else []):
        host = mixed_rows(rng, edges + more + [0] + edges[::-1], nulls=(2, 20 + len(more)))
        assert call(dev(nv, host), 5, a, b, 5).to_host().equals(ref(host, 5, a, b, 5, nthreads=8))


@pytest.mark.parametrize("count", [96, 129, 256, 260, 520])
@pytest.mark.parametrize("rows", [100, 450, 700, 1100, 2200])
def test_minhash64_chunks_of_groups(nv, orc, rows, count):
    """Columns in which the wavefronts suffice for two groups of 32 parameters each, for four, and for neither."""
    rng = np.random.default_rng(rows + count)
    a, b = params(rng, count, 64)
    host = mixed_rows(rng, rng.integers(1, 600, rows), nulls=(3,))
    assert nv.minhash64(dev(nv, host), 5, a, b, 5).to_host().equals(orc.minhash64(host, 5, a, b, 5, nthreads=8))


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("count", [1, 64, 130, 260])
def test_minhash_rows_of_thousands_of_parts(nv, orc, bits, count):
    """Rows and lists that are cut into as many parts as look at a slot before they lower it (2048), a few less and twice as many,
    beside short ones."""
    rng = np.random.default_rng(count)
    a, b = params(rng, count, bits)
    call, ref = (nv.minhash, orc.minhash) if bits == 32 else (nv.minhash64, orc.minhash64)
    for lens in ([2048 * 256 - 300, 5], [2048 * 256 + 300], [0, 1_100_000, 40]):
        host = mixed_rows(rng, lens)
        assert call(dev(nv, host), 5, a, b, 5).to_host().equals(ref(host, 5, a, b, 5, nthreads=8))
    call, ref = (nv.minhash_ngrams, orc.minhash_ngrams) if bits == 32 else (nv.minhash64_ngrams, orc.minhash64_ngrams)
    for lens in ([2048 * 64 - 100, 3], [0, 2048 * 128 + 500, 7]):
        offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        lists = HostListStringsColumn(offsets, mixed_rows(rng, rng.integers(0, 9, int(offsets[-1]))), None, len(lens), 0, 0)
        assert call(nv.DeviceListStringsColumn.from_host(lists), 2, 5, a, b).to_host().equals(ref(lists, 2, 5, a, b, nthreads=8))


@pytest.mark.parametrize("rows", [1023, 1024, 1025, 8191, 8192, 8193, 131_071, 131_072, 262_144, 262_145])
@pytest.mark.parametrize("nulls", [False, True])
def test_minhash_row_counts(nv, orc, rows, nulls):
    """Around the tiles of 1024 rows of the plan, the rows from which it takes two launches and those from which its tiles grow."""
    rng = np.random.default_rng(rows)
    lens = rng.integers(0, 12, rows)
    lens[[0, 7, rows // 2, rows - 1]] = [4097, 4096, 30_000, 9000]
    host = mixed_rows(rng, lens, nulls=(1, rows // 3, rows - 2) if nulls else ())
    a, b = params(rng, 3, 32)
    assert nv.minhash(dev(nv, host), 5, a, b, 4).to_host().equals(orc.minhash(host, 5, a, b, 4, nthreads=8))
    a, b = params(rng, 3, 64)
    assert nv.minhash64(dev(nv, host), 5, a, b, 4).to_host().equals(orc.minhash64(host, 5, a, b, 4, nthreads=8))


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("filler, short", [(0, 0), (0, 9000), (20, 0), (20, 9000), (75, 0)])
def test_minhash_even_parts(nv, orc, bits, filler, short):
    """Rows of all lengths up to five parts of 2816 bytes, in columns whose parts are the smallest, larger and the largest
    (20 and 75 MB of other rows), with fewer rows than wavefronts (each part within the length) and with more (the nearest)."""
    rng = np.random.default_rng(filler + short)
    lens = np.concatenate([np.arange(0, 14_500, 97), [1_000_000] * filler, np.full(short, 90)])
    host = mixed_rows(rng, rng.permutation(lens))
    call, ref = (nv.minhash, orc.minhash) if bits == 32 else (nv.minhash64, orc.minhash64)
    a, b = params(rng, 3, bits)
    assert call(dev(nv, host), 5, a, b, 5).to_host().equals(ref(host, 5, a, b, 5, nthreads=8))


@pytest.mark.parametrize("rows", [70_000, 120_000, 300_000])
@pytest.mark.parametrize("bits, count", [(32, 5), (32, 330), (64, 5), (64, 130)])
def test_minhash_units_of_rows(nv, orc, rows, bits, count):
    """Columns whose rows are handed out one and several at a time: rows of a few windows and empty ones, runs of thousands
    of null rows between them (where the rows are not where an even column would have them), long rows first, in the middle
    and last; the parameters in one chunk and in several."""
    if rows * count > 20_000_000:
        rows //= 5
    rng = np.random.default_rng(rows)
    lens = rng.integers(0, 10, rows)
    lens[[0, rows // 2, rows - 1]] = 20_000, 40_001, 9_999
    nulls = np.unique(np.concatenate([np.arange(rows // 8, rows // 8 + rows // 4), np.arange(rows // 2 + 1, rows // 2 + 66), [5, rows - 2]]))
    host = mixed_rows(rng, lens, nulls=tuple(nulls.tolist()))
    call, ref = (nv.minhash, orc.minhash) if bits == 32 else (nv.minhash64, orc.minhash64)
    a, b = params(rng, count, bits)
    assert call(dev(nv, host), 5, a, b, 4).to_host().equals(ref(host, 5, a, b, 4, nthreads=8))


def hard_parameters(kind):
    p = (1 << 61) - 1
    a = {"zero": [0, p, 2 * p], "small": [1, 2, 3, 5], "power": [1 << 60, 1 << 61, 1 << 63, 1 << 44, 1 << 43], "digits of 2": [0xAAAAAAAAAAAAAAAA],
         "digits of 1": [0x5555555555555555], "wraps": [(1 << 64) - 1, p - 1, p + 1], "top": [(1 << 44) - 1, (1 << 64) - (1 << 44)]}[kind]
    b = [0, 1, p - 1, p, p + 7, (1 << 61) - 8, (1 << 64) - 1, 1 << 44, (1 << 44) - 1]
    pairs = np.array([(x, y) for x in a for y in b], np.uint64)
    return pairs[:, 0].copy(), pairs[:, 1].copy()


@pytest.mark.parametrize("kind", ["zero", "small", "power", "digits of 2", "digits of 1", "wraps", "top"])
def test_minhash64_parameters(nv, orc, kind):
    """Parameters for which the fractions that decide what is computed exactly tie, lie at zero or at the wrap, or take their
    sums to the ends of their range; rows of one window, of fewer than a block of 32 and of many, with windows that repeat."""
    rng = np.random.default_rng(7)
    a, b = hard_parameters(kind)
    host = mixed_rows(rng, [5, 6, 30, 36, 37, 300, 3000, 40_000])
    text = HostStringsColumn.from_pylist(["abcdefgh" * 500, "a" * 3000, "the same words " * 400, "naïve 漢字 " * 60])
    for column in (host, text):
        assert nv.minhash64(dev(nv, column), 5, a, b, 5).to_host().equals(orc.minhash64(column, 5, a, b, 5, nthreads=8))


@pytest.mark.parametrize("count", [1, 32, 33, 70, 128, 260])
def test_minhash64_last_blocks(nv, orc, count):
    """Rows of 1 to 130 windows and of some above 256: every fill of a block of 32 hashes, all of them different and with
    one that repeats; the parameters in one group of 32 and in several."""
    rng = np.random.default_rng(count)
    a, b = params(rng, count, 64)
    lens = list(range(5, 135)) + list(range(256, 300))
    rows = [random_text(rng, n).decode() for n in lens] + ["ab" * (n // 2) + "xyz"[: n % 3] for n in lens]
    host = HostStringsColumn.from_pylist(rows)
    assert nv.minhash64(dev(nv, host), 5, a, b, 5).to_host().equals(orc.minhash64(host, 5, a, b, 5, nthreads=8))


@pytest.mark.parametrize("count", [33, 97, 160, 161, 193, 225, 288, 289])
def test_minhash64_gathered_hashes(nv, orc, count):
    """Rows of as many windows as are gathered before they meet the parameters (416) and as a tile of 256 more gives, one
    less and more, whole blocks of 32 or not, in a column long enough that they are not cut; every number of groups of
    parameters that are done two, four or one at a time, and two chunks; windows that repeat within what is remembered."""
    rng = np.random.default_rng(count)
    a, b = params(rng, count, 64)
    windows = [1, 255, 256, 257, 400, 415, 416, 417, 447, 448, 449, 511, 512, 513, 671, 672, 673, 700]
    rows = [random_text(rng, n + 4).decode() for n in windows * 800]
    words = ["ox", "a", "tree", "mill", "saturn", "of"]
    rows += [" ".join(words[i] for i in rng.integers(0, 6, 160)) for _ in range(800)]
    host = HostStringsColumn.from_pylist(rows)
    assert nv.minhash64(dev(nv, host), 5, a, b, 5).to_host().equals(orc.minhash64(host, 5, a, b, 5, nthreads=8))


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("ngrams", [2, 5])
@pytest.mark.parametrize("count", [1, 130])
def test_minhash_ngrams_parts_of_rows(nv, orc, bits, ngrams, count):
    """Lists one element around a trip of 64 positions, around the four that are folded together and around several parts,
    shorter than a run, empty, and among 131,072 others; elements that are null or empty; a view."""
    rng = np.random.default_rng(count)
    call, ref = (nv.minhash_ngrams, orc.minhash_ngrams) if bits == 32 else (nv.minhash64_ngrams, orc.minhash64_ngrams)
    a, b = params(rng, count, bits)
    edges = [0, 1, 2, 5, 6, 7, 63, 64, 65, 68, 69, 255, 256, 260, 261, 1024, 1028, 1029, 2053, 5000]
    for lens in (edges + edges[::-1], edges + [1, 0, 3] * 43_691 if count == 1 else edges):
        offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        n = int(offsets[-1])
        child = mixed_rows(rng, rng.integers(0, 12, n), nulls=range(10, n, 97))
        lists = HostListStringsColumn(offsets, child, None, len(lens), 0, 0)
        d = nv.DeviceListStringsColumn.from_host(lists)
        assert call(d, ngrams, 5, a, b).to_host().equals(ref(lists, ngrams, 5, a, b, nthreads=8))
        assert call(d.slice(2, len(lens) - 1, 0), ngrams, 5, a, b).to_host().equals(
            ref(HostListStringsColumn(offsets, child, None, len(lens) - 3, 2, 0), ngrams, 5, a, b, nthreads=8))


@pytest.mark.parametrize("mean", [3, 113, 115, 420])
@pytest.mark.parametrize("count", [1, 26, 64, 128, 130, 256, 320, 330])
def test_minhash64_ngrams_short_and_long_lists(nv, orc, mean, count):
    """Lists shorter and longer than the average from which products go to the matrix cores (114 elements with 128 parameters
    and fewer, 400 with 256, none with 130 and 320); the parameters in one set, several, with a rest and in two chunks."""
    rng = np.random.default_rng(mean + count)
    lens = np.full(150, mean)
    lens[[3, 60]] += [1, -1]
    lens[[5, 6, 7]] = 0, 1, 2 * mean
    lens[8] -= int(lens.sum()) - 150 * mean if mean > 3 else 0
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    child = mixed_rows(rng, rng.integers(0, 9, int(offsets[-1])), nulls=(4,))
    lists = HostListStringsColumn(offsets, child, None, 150, 0, 0)
    a, b = params(rng, count, 64)
    assert nv.minhash64_ngrams(nv.DeviceListStringsColumn.from_host(lists), 3, 5, a, b).to_host().equals(orc.minhash64_ngrams(lists, 3, 5, a, b, nthreads=8))


@pytest.mark.parametrize("kind", ["zero", "small", "power", "digits of 2", "digits of 1", "wraps", "top"])
def test_minhash64_ngrams_parameters(nv, orc, kind):
    """The same of short lists, whose products are computed whole: sums at p and beyond, which are reduced only where one occurs."""
    rng = np.random.default_rng(8)
    a, b = hard_parameters(kind)
    lens = np.array([1, 2, 3, 6, 7, 8, 64, 66, 70, 100])
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    lists = HostListStringsColumn(offsets, mixed_rows(rng, rng.integers(0, 9, int(offsets[-1]))), None, lens.size, 0, 0)
    assert nv.minhash64_ngrams(nv.DeviceListStringsColumn.from_host(lists), 2, 5, a, b).to_host().equals(orc.minhash64_ngrams(lists, 2, 5, a, b, nthreads=8))


def words_column(rng, lens, vocabulary, oov):
    """Rows of about these many bytes: words of the vocabulary, and `oov` of them random letters."""
    stems = [w for w in vocabulary if not w.startswith("##") and not w.startswith("[")]
    rows = []
    for n in lens:
        parts, size = [], 0
        while size < n:
            w = stems[int(rng.integers(0, len(stems)))] if rng.random() >= oov else "".join(rng.choice(list("abcdefgxyz"), int(rng.integers(1, 26))))
            parts.append(w)
            size += len(w) + 1
        rows.append(" ".join(parts)[:n])
    return HostStringsColumn.from_pylist(rows)


LETTERS = list("abcdefghijklmnopqrstuvwxyz")
VOCABULARY = ["[PAD]", "[UNK]"] + LETTERS[:20] + ["##" + c for c in LETTERS[:20]] + ["hello", "world", "data", "frame", "##ing", "##ed", "abc", "##abc", "internationalization",
                                                                                      "naïve", "漢", "##漢"]


@pytest.mark.parametrize("limit", [0, 1, 9])
@pytest.mark.parametrize("oov", [0.0, 0.2, 1.0])
def test_tokenize_small_columns(nv, orc, limit, oov):
    """Columns that are tokenized in one launch: rows around the 1024-byte tiles and across several of them, words of more
    than sixteen bytes and of more than seven tokens, every word unknown (too many for a tile's records: the passes of a
    large column then), one-letter words and rows, a view."""
    rng = np.random.default_rng(int(10 * oov) + limit)
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    columns = [words_column(rng, [1], VOCABULARY, oov), words_column(rng, [1023, 1, 1024, 0, 1025, 2047, 5000, 3, 16, 17], VOCABULARY, oov),
               words_column(rng, list(rng.integers(0, 90, 3000)), VOCABULARY, oov),
               HostStringsColumn.from_pylist(["a b c d e " * 300, "漢 naïve 漢漢漢漢漢漢漢漢 " * 50, "x" * 199 + " " + "y" * 200 + " " + "a" * 40] + ["a"] * 2000)]
    for host in columns:
        d = dev(nv, host)
        assert nv.wordpiece_tokenize(d, vocabulary, limit).to_host().equals(orc.wordpiece_tokenize(host, reference, limit))
        if host.size > 8:
            view = host.slice(3, host.size - 2)
            assert nv.wordpiece_tokenize(d.slice(3, host.size - 2, 0), vocabulary, limit).to_host().equals(orc.wordpiece_tokenize(view, reference, limit))


def test_tokenize_small_columns_hold_little_memory(nv):
    """32,768 rows of about 120 bytes: the temporaries of a call do not grow to what the largest column of so many rows takes."""
    import torch
    rng = np.random.default_rng(5)
    words = words_column(rng, [120] * 64, VOCABULARY, 0.1)
    n = int(words.offsets[-1])
    offsets = (np.arange(512)[:, None] * n + np.asarray(words.offsets[:-1])).reshape(-1)
    host = HostStringsColumn(np.tile(words.chars[:n], 512), np.append(offsets, 512 * n).astype(np.int32), None, 512 * 64, 0, 0)
    column, vocabulary = dev(nv, host), nv.WordPieceVocabulary(dev(nv, HostStringsColumn.from_pylist(VOCABULARY)))
    nv.wordpiece_tokenize(column, vocabulary, 0)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    held = torch.cuda.memory_allocated()
    nv.wordpiece_tokenize(column, vocabulary, 0)
    assert torch.cuda.max_memory_allocated() - held < 16 * host.chars.size


@pytest.mark.parametrize("limit", [0, 40])
@pytest.mark.parametrize("megabytes", [3, 6, 7.99, 8.01, 20])
@pytest.mark.parametrize("dense", ["", "a b ", "abcq hello world "])
def test_tokenize_small_columns_again(nv, orc, megabytes, dense, limit):
    """Columns of fewer and of more bytes than their rows let one guess (8 MiB), with room for all that a tile is given and
    for half of it; in some a few tiles have more words, or more unknown ones, than that half."""
    rng = np.random.default_rng(int(megabytes))
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    piece = words_column(rng, [200_000], VOCABULARY, 0.1).chars
    total = int(megabytes * (1 << 20))
    chars = np.tile(piece, total // piece.size + 1)[:total].copy()
    if dense:
        patch = np.frombuffer((dense * (5000 // len(dense))).encode(), np.uint8)
        for at in (100_000, total // 2, total - 9000):
            chars[at: at + patch.size] = patch
    offsets = np.linspace(0, total, 4001).astype(np.int32)
    host = HostStringsColumn(chars, offsets, None, 4000, 0, 0)
    assert nv.wordpiece_tokenize(dev(nv, host), vocabulary, limit).to_host().equals(orc.wordpiece_tokenize(host, reference, limit, nthreads=8))


def kernel_launches(call):
    """What call() gives, and the kernels that the library timed for it."""
    import torch
    from cudf_amd import _capi
    _capi.profile_enable(True)
    _capi.profile_read()
    try:
        out = call()
        torch.cuda.synchronize()
        return out, [name for name, _ in _capi.profile_read()]
    finally:
        _capi.profile_enable(False)


@pytest.mark.parametrize("sizes, kilobytes, small, large", [((16,), 7500, 1, 0), ((32, 34), 1000, 1, 0), ((16, 28), 1000, 1, 0), ((8,), 1000, 1, 0),
                                                            ((7, 8, 14, 15, 28), 1000, 1, 0), ((7, 8), 7500, 2, 0), ((2, 3), 1000, 1, 1)])
def test_tokenize_small_columns_of_words_of_many_tokens(nv, orc, sizes, kilobytes, small, large):
    """Columns all of whose words have about eight tokens, or fourteen, and one more: as many as a tile has second records for, more,
    and several times as many; that takes no launch more than what their number takes (a tile of 1000 KB has records for 128 words, of
    7500 KB for 64 in the first launch and for 128 in the second; beyond it is a large column's way)."""
    rng = np.random.default_rng(kilobytes + len(sizes))
    letters = "abcdefgh"
    pairs = [a + b for a in letters for b in letters] if min(sizes) > 15 else []
    hv = HostStringsColumn.from_pylist(["[UNK]"] + list(letters) + ["##" + c for c in letters] + pairs + ["##" + c for c in pairs])
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    text = (" ".join("".join(rng.choice(list(letters), int(rng.choice(sizes)))) for _ in range(20_000)) + " ").encode()
    total = kilobytes * 1000
    chars = np.frombuffer(text * (total // len(text) + 1), np.uint8)[:total].copy()
    host = HostStringsColumn(chars, np.linspace(0, total, 2001).astype(np.int32), None, 2000, 0, 0)
    expected = orc.wordpiece_tokenize(host, reference, 0, nthreads=8)
    for _ in range(2):
        got, names = kernel_launches(lambda: nv.wordpiece_tokenize(dev(nv, host), vocabulary, 0))
        assert got.to_host().equals(expected)
        assert (names.count("wordpiece_word_kernel (small column)"), names.count("wordpiece_word_kernel")) == (small, large)


@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 511, 4095, 4096, 4097, 4105, 8200])
def test_tokenize_blocks_of_tiles(nv, orc, tiles):
    """Columns of so many tiles of 1024 bytes: a block is eight of them, and more where 512 workgroups have more to do; the
    last block is full, has one tile, or all but one.  A second call finds what the first left for it."""
    rng = np.random.default_rng(tiles)
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    text = words_column(rng, [100_000], VOCABULARY, 0.1).chars
    total = 1024 * tiles - 16  # (the first byte may lie up to 15 bytes into a tile)
    chars = np.tile(text, total // text.size + 1)[:total].copy()
    rows = max(total // 400, 1)
    host = HostStringsColumn(chars, np.linspace(0, total, rows + 1).astype(np.int32), None, rows, 0, 0)
    column, expected = dev(nv, host), orc.wordpiece_tokenize(host, reference, 60, nthreads=8)
    for _ in range(2):
        assert nv.wordpiece_tokenize(column, vocabulary, 60).to_host().equals(expected)


@pytest.mark.parametrize("rows", [140_000, 700_000])
@pytest.mark.parametrize("oov", [0.0, 0.003, 0.1, 0.5, 1.0])
def test_tokenize_chunks_of_the_queue(nv, orc, rows, oov):
    """Columns beyond the small ones with no unknown word, a few for some of the wavefronts, a few for each, and so many that
    the queue is handed out in larger chunks; some with words that overflow the first attempt's queue at one end of the column."""
    rng = np.random.default_rng(rows + int(100 * oov))
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    text = words_column(rng, [300_000], VOCABULARY, oov).chars
    total = rows * 60
    chars = np.tile(text, total // text.size + 1)[:total].copy()
    if oov == 0.1:
        chars[total - total // 6:] = np.frombuffer(b"qz " * (total // 18 + 1), np.uint8)[: total // 6]
    host = HostStringsColumn(chars, np.linspace(0, total, rows + 1).astype(np.int32), None, rows, 0, 0)
    assert nv.wordpiece_tokenize(dev(nv, host), vocabulary, 0).to_host().equals(orc.wordpiece_tokenize(host, reference, 0, nthreads=8))


@pytest.mark.parametrize("every", [1, 8, 64])
@pytest.mark.parametrize("megabytes", [64, 144])
def test_tokenize_unknown_words_in_some_ranges(nv, orc, every, megabytes):
    """Ranges of 2048 bytes of unknown words, every one, every eighth and every sixty-fourth, the others of known ones, in columns that
    are done in one part and in two: the queue is handed out evenly, and not much longer than what they fill of it."""
    import torch
    from cudf_amd import _capi
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    tile = lambda text: np.frombuffer((text * (2048 // len(text) + 1)).encode(), np.uint8)[:2047].tolist() + [0x20]
    rng = np.random.default_rng(every)
    known, unknown = tile("hello world data frame "), [tile("".join("".join(rng.choice(LETTERS[:6], 2)) + " " for _ in range(683))) for _ in range(8)]
    block = [unknown[i // every % 8] if i % every == min(3, every - 1) else known for i in range(512)]
    chars = np.tile(np.array(block, np.uint8).reshape(-1), megabytes)
    host = HostStringsColumn(chars, np.linspace(0, chars.size, 150_001).astype(np.int32), None, 150_000, 0, 0)
    column, expected = dev(nv, host), orc.wordpiece_tokenize(host, reference, 0, nthreads=8)
    _capi.set_range_tiles(1)
    try:
        nv.wordpiece_tokenize(column, vocabulary, 0)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        got = nv.wordpiece_tokenize(column, vocabulary, 0)
        # (2.5 bytes of temporaries for a byte and a chunk for a wavefront; what the queue takes of every unknown word; the result)
        words = chars.size // every // 3
        assert torch.cuda.max_memory_allocated() - held < 3 * chars.size + (300 << 20) + 48 * words + 4 * expected.child.size
        assert got.to_host().equals(expected)
    finally:
        _capi.set_range_tiles(0)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("shape", ["first", "last", "middle", "empty between", "even", "short"])
def test_tokenize_rows_of_ranges(nv, orc, shape, wide):
    """Where the rows of every range begin: all bytes in one row of 140,003, runs of empty rows, ranges with no row's beginning and
    ranges with thousands, of a column and of a slice of it."""
    rng = np.random.default_rng(len(shape))
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    rows = 140_003
    lens = {"even": np.full(rows, 9), "short": rng.integers(0, 3, rows), "empty between": np.where(np.arange(rows) % 10_000 < 9_990, 0, 997)}.get(shape)
    if lens is None:
        lens = np.zeros(rows, np.int64)
        lens[{"first": 0, "last": rows - 1, "middle": 70_001}[shape]] = 300_000
    offsets = np.concatenate([[0], np.cumsum(lens)])
    chars = words_column(rng, [int(offsets[-1])], VOCABULARY, 0.1).chars[: int(offsets[-1])]
    host = HostStringsColumn(chars, offsets.astype(np.int64 if wide else np.int32), None, rows, 0, 0)
    for lo in (0, 3):
        part = HostStringsColumn(host.chars, host.offsets, None, rows - lo, lo, 0)
        assert nv.wordpiece_tokenize(dev(nv, host).slice(lo, rows, 0), vocabulary, 5).to_host().equals(orc.wordpiece_tokenize(part, reference, 5, nthreads=8))


@pytest.mark.parametrize("letters", ["ab", "aé", "漢字b", "a\U0001F600"])
@pytest.mark.parametrize("rows", [900, 140_000])
def test_tokenize_words_longer_than_a_window(nv, orc, letters, rows):
    """Words of up to 199 bytes made of pieces of 1 to 60 bytes, some known, some one character off: candidates of 15 to 18 bytes
    and of many more at the beginning of a word and behind other pieces, characters across the sixteenth byte, words of 7, 8,
    14, 15 and more tokens; in a small column and in a large one."""
    rng = np.random.default_rng(rows + len(letters))
    def piece(nbytes):
        out = ""
        while len(out.encode()) < nbytes:
            out += letters[int(rng.integers(0, len(letters)))]
        return out
    sizes = [1, 2, 3, 4, 5, 13, 14, 15, 16, 17, 18, 19, 20, 31, 33, 34, 35, 60]
    keys = sorted({piece(n) for n in sizes for _ in range(4)})
    vocab = ["[UNK]"] + [k for i, k in enumerate(keys) if i % 3 != 1] + ["##" + k for i, k in enumerate(keys) if i % 3 != 2]
    vocab += [w for w in (c for c in letters[:1]) if w not in vocab] + ["##" + c for c in letters if "##" + c not in vocab]
    words = []
    for _ in range(1500):
        parts = [keys[int(rng.integers(0, len(keys)))] for _ in range(int(rng.integers(1, 9)))]
        if rng.random() < 0.3:
            parts = [letters[int(rng.integers(0, len(letters)))] for _ in range(int(rng.choice([6, 7, 8, 13, 14, 15, 16, 30])))]
        if rng.random() < 0.2:
            parts.insert(int(rng.integers(0, len(parts) + 1)), "z")
        words.append("".join(parts)[:199])
    hv = HostStringsColumn.from_pylist(vocab)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    texts = [" ".join(words[int(i)] for i in rng.integers(0, len(words), 3)) for _ in range(900)]
    host = HostStringsColumn.from_pylist([texts[i % 900] for i in range(rows)])
    assert nv.wordpiece_tokenize(dev(nv, host), vocabulary, 0).to_host().equals(orc.wordpiece_tokenize(host, reference, 0, nthreads=8))


def test_tokenize_from_threads_that_come_and_go(nv, orc):
    """Forty host threads, eight at a time, tokenize small columns of different sizes: what a call adds up on the device is its thread's own,
    and is there again for the threads that follow."""
    import threading
    import torch
    rng = np.random.default_rng(3)
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    hosts = [words_column(rng, list(rng.integers(0, 300, 40 * 2 ** k)), VOCABULARY, 0.2) for k in range(8)]
    columns, expected, wrong = [dev(nv, h) for h in hosts], [orc.wordpiece_tokenize(h, reference, 0) for h in hosts], []
    torch.cuda.synchronize()

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                if not nv.wordpiece_tokenize(columns[k], vocabulary, 0).to_host().equals(expected[k]):
                    wrong.append(k)

    for _ in range(5):
        threads = [threading.Thread(target=work, args=(k,)) for k in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not wrong


@pytest.fixture(params=["own", "another", "none"])
def arrivals(request):
    """Calls of a thread that has memory for what workgroups add up, of one whose memory a failed call has made unfit, and of one
    beyond the 1,024 that the library has some for."""
    from cudf_amd import _capi
    if request.param != "own":
        left = _capi.hold_arrivals(0)
        assert (_capi.hold_arrivals(1 << 20) == 0) if request.param == "none" else left > 900
    yield request.param
    _capi.hold_arrivals(0)


def test_a_thread_without_memory_of_its_own(nv, orc, arrivals):
    """A small tokenizer column, one that is sampled and done in two parts, and jaccard_index of pairs that are listed go the
    same way in all three."""
    from cudf_amd import _capi
    rng = np.random.default_rng(11)
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    small = words_column(rng, list(rng.integers(0, 90, 3000)), VOCABULARY, 0.2)
    piece = words_column(rng, [100_000], VOCABULARY, 0.2).chars
    total = 130 << 20
    large = HostStringsColumn(np.tile(piece, total // piece.size + 1)[:total].copy(), np.linspace(0, total, 300_001).astype(np.int32), None, 300_000, 0, 0)
    for host, kernel, launches in ((small, "wordpiece_word_kernel (small column)", 1), (large, "wordpiece_word_kernel", 2)):
        column, expected = dev(nv, host), orc.wordpiece_tokenize(host, reference, 0, nthreads=8)
        for _ in range(2):
            got, names = kernel_launches(lambda: nv.wordpiece_tokenize(column, vocabulary, 0))
            assert got.to_host().equals(expected)
            assert [n for n in names if n.startswith("wordpiece_word_kernel")] == [kernel] * launches
    rows = [random_text(rng, n).decode() for n in (10, 700, 2500, 5000, 9000, 15_000, 61_000)] * 9
    h1, h2 = (HostStringsColumn.from_pylist(side) for side in ([t[: len(t) // 3] for t in rows], [t[len(t) // 4:] for t in rows]))
    expected = orc.jaccard_index(h1, h2, 4, nthreads=8).values.view(np.uint32)
    for _ in range(2):
        got, names = kernel_launches(lambda: nv.jaccard_index(dev(nv, h1), dev(nv, h2), 4))
        assert np.array_equal(got.to_host().values.view(np.uint32), expected)
        assert names == ["jaccard_wave_kernel", "jaccard_teams_kernel"]
    if arrivals == "another":
        left = _capi.hold_arrivals(0)
        nv.wordpiece_tokenize(dev(nv, small), vocabulary, 0)
        assert _capi.hold_arrivals(0) == left - 1


@pytest.mark.parametrize("rows, each", [(4, 65_537), (4, 65_535), (131_072, 10), (131_073, 10), (9000, 3800)])
def test_tokenize_where_small_columns_end(nv, orc, rows, each):
    """Around the bytes (256 KiB; 32 MiB) and the rows up to which a column is put on the stream before its size is known."""
    rng = np.random.default_rng(rows)
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    text = words_column(rng, [rows * each], VOCABULARY, 0.1)
    offsets = np.linspace(0, rows * each, rows + 1).astype(np.int32)
    host = HostStringsColumn(text.chars, offsets, None, rows, 0, 0)
    assert nv.wordpiece_tokenize(dev(nv, host), vocabulary, 50).to_host().equals(orc.wordpiece_tokenize(host, reference, 50, nthreads=8))


@pytest.mark.parametrize("different", [1, 3000, 60_000, 500_000])
@pytest.mark.parametrize("limit, wide", [(0, False), (60, True)])
def test_tokenize_words_met_before(nv, orc, different, limit, wide):
    """Columns around the 128 MiB from which the unknown words of the first ranges are kept: few different ones, many, and
    too many to keep; of 1 to 20 bytes (kept: up to 12), of one token and of more than seven; offsets of 32 and 64 bits."""
    rng = np.random.default_rng(different)
    hv = HostStringsColumn.from_pylist(VOCABULARY)
    vocabulary, reference = nv.WordPieceVocabulary(dev(nv, hv)), orc.Vocabulary(hv)
    cells = np.full((different + 40, 24), 0x20, np.uint8)
    for i in range(40):
        word = VOCABULARY[2 + i % 20] if i % 2 else "hello"
        cells[i, : len(word)] = np.frombuffer(word.encode(), np.uint8)
    size = rng.integers(1, 21, different)
    letters = rng.choice(np.frombuffer(b"abcdefgxyz", np.uint8), (different, 20))
    cells[40:, :20] = np.where(np.arange(20) < size[:, None], letters, 0x20)
    for total in ((128 << 20) - 24 * 64, (128 << 20) + 24 * 64):
        n = total // 24
        chars = cells[np.where(rng.random(n) < 0.5, rng.integers(0, 40, n), rng.integers(40, different + 40, n))].reshape(-1)
        offsets = np.arange(0, n * 24 + 1, 24 * 64, dtype=np.int64 if wide else np.int32)
        host = HostStringsColumn(chars[: offsets[-1]], offsets, None, offsets.size - 1, 0, 0)
        assert nv.wordpiece_tokenize(dev(nv, host), vocabulary, limit).to_host().equals(orc.wordpiece_tokenize(host, reference, limit, nthreads=8))


@pytest.mark.parametrize("rows, each", [(1, 1), (3, 2047), (3, 2048), (61, 300), (4, 65_535), (4, 65_537), (131_072, 9), (131_073, 9), (30_000, 2300)])
@pytest.mark.parametrize("brackets", [True, False])
def test_normalize_where_small_columns_end(nv, rows, each, brackets):
    """Tiles of 2048 bytes and their remainders, and the bytes (256 KiB; 20 MiB) and rows up to which a column is worked on
    before its size is known; a view of it too.  With a special token in every tile, which is then written the long way, and
    without."""
    from oracle import normalize_py
    rng = np.random.default_rng(rows)
    text = "Héllo Wörld, [CLS] naïve 漢字! ΑΒΓ don't [sep] plain words and more plain words of text "
    if not brackets:
        text = text.replace("[", "\u200b").replace("]", "\u0301")
    chars = np.frombuffer((text * (rows * each // len(text) + 1)).encode(), np.uint8).copy()
    cuts = np.sort(rng.integers(0, chars.size, rows - 1)) if rows > 1 else np.zeros(0, np.int64)
    while True:  # whole characters
        inside = (cuts > 0) & ((chars[np.minimum(cuts, chars.size - 1)] & 0xC0) == 0x80)
        if not inside.any():
            break
        cuts[inside] -= 1
    host = HostStringsColumn(chars, np.concatenate([[0], cuts, [chars.size]]).astype(np.int32), None, rows, 0, 0)
    special = HostStringsColumn.from_pylist(["[CLS]", "[SEP]"])
    normalizer = nv.CharacterNormalizer(True, dev(nv, special))
    d = dev(nv, host)
    for lo, hi in ((0, rows), (1, rows - 1)) if rows > 4 else ((0, rows),):
        got = nv.normalize_characters(d.slice(lo, hi, 0), normalizer).to_host()
        exp = normalize_py.normalize_characters_native(host.slice(lo, hi), True, [b"[CLS]", b"[SEP]"], nthreads=8)
        assert np.array_equal(got.chars, exp.chars) and np.array_equal(got.offsets, exp.offsets)


@pytest.mark.parametrize("width", [2, 5, 17])
@pytest.mark.parametrize("lead", [0, 1, 3])
def test_characters_of_a_tile(nv, orc, width, lead):
    """Rows of several scripts and of bytes that are no UTF-8 (continuation bytes in front, in the middle and alone, characters
    cut off by the end of the row), of lengths around the tiles of 256 bytes, with any alignment of the first byte."""
    rng = np.random.default_rng(10 * width + lead)
    pieces = [b"a", b"xyz", "é".encode(), "漢字".encode(), "\U0001F600".encode(), b"\x80", b"\xbf\x80\x80\x80\x80", b"\xe6\xbc", b"\xff", b"\xf0\x9f"]
    rows = []
    for shares in ([8, 8, 8, 8, 8, 0, 0, 0, 0, 0], [4, 2, 8, 1, 1, 1, 0, 0, 0, 0], [1, 1, 1, 1, 1, 1, 1, 1, 1, 1], [0, 0, 1, 9, 0, 0, 0, 0, 0, 0], [0, 0, 0, 0, 0, 4, 1, 0, 0, 0]):
        p = np.array(shares) / np.sum(shares)
        for size in [1, 7, 63, 64, 65, 127, 128, 129, 250, 255, 256, 257, 258, 261, 383, 384, 385, 511, 512, 513, 767, 768, 769, 1500]:
            rows.append(b"".join(pieces[i] for i in rng.choice(len(pieces), size, p=p))[:size])
    chars = np.frombuffer(b"#" * lead + b"".join(rows), np.uint8).copy()
    offsets = np.concatenate([[0], lead + np.concatenate([[0], np.cumsum([len(r) for r in rows])])]).astype(np.int32)
    host = HostStringsColumn(chars, offsets, None, len(rows) + 1, 0, 0).slice(1, len(rows) + 1)
    for bits in (32, 64):
        a, b = params(rng, 40, bits)
        call, ref = (nv.minhash, orc.minhash) if bits == 32 else (nv.minhash64, orc.minhash64)
        assert call(dev(nv, host), 5, a, b, width).to_host().equals(ref(host, 5, a, b, width, nthreads=8))
    h1, h2 = host.slice(0, len(rows) - 1), host.slice(1, len(rows))
    got, exp = nv.jaccard_index(dev(nv, h1), dev(nv, h2), width).to_host(), orc.jaccard_index(h1, h2, width, nthreads=8)
    assert np.array_equal(got.values.view(np.uint32), exp.values.view(np.uint32))


@pytest.mark.parametrize("elements, count", [(n, c) for c in (26, 64, 100, 260) for n in (199_999, 200_000)] + [(122_070, 1024), (122_071, 1024)])
def test_minhash64_ngrams_few_elements(nv, orc, count, elements):
    """Lists of so many elements (200,000), or of so many products of them and the parameters (125,000,000), that these are found on the
    matrix cores, and one element less; the last group of parameters full or not."""
    rng = np.random.default_rng(count)
    a, b = params(rng, count, 64)
    lens = [700] * (elements // 714)
    lens += [elements - sum(lens)]
    offsets = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    child = mixed_rows(rng, rng.integers(0, 12, elements))
    lists = HostListStringsColumn(offsets, child, None, len(lens), 0, 0)
    got = nv.minhash64_ngrams(nv.DeviceListStringsColumn.from_host(lists), 3, 5, a, b).to_host()
    assert got.equals(orc.minhash64_ngrams(lists, 3, 5, a, b, nthreads=8))


@pytest.mark.parametrize("rows", [3, 40, 700])
@pytest.mark.parametrize("count", [1, 26, 33, 65, 100, 129, 260, 300])
def test_minhash64_few_units(nv, orc, rows, count):
    """Columns of fewer parts than wavefronts, done by chunks of two groups of parameters, and of some more; the last group
    full or not."""
    rng = np.random.default_rng(count)
    a, b = params(rng, count, 64)
    host = HostStringsColumn.from_pylist([random_text(rng, n).decode() for n in rng.integers(0, 200_000 // rows, rows)])
    assert nv.minhash64(dev(nv, host), 5, a, b, 8).to_host().equals(orc.minhash64(host, 5, a, b, 8, nthreads=8))
