"""The sizes at which a kernel hands over to another, or a loop to its remainder, against the host oracle, bit for bit."""
import numpy as np
import pytest

from cudf_amd.arrow_host import HostStringsColumn

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


@pytest.mark.parametrize("width", [2, 7, 40])
def test_jaccard_pair_sizes(nv, orc, width):
    """Pairs one byte around the most that each set takes (4/5 of 1024, 4096, 8064, 14336 and 29440 slots), around one
    and several parts of 20,000 bytes, and around the most parts (16); no window repeats, so the sets are as full as they get."""
    rng = np.random.default_rng(width)
    sizes = [n * 4 // 5 + d for n in (1024, 4096, 8064, 14336, 29440) for d in (0, 1)]
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
