"""The device-wide scan behind the sizes of normalize_characters and wordpiece_tokenize, which no column that a test can hold takes
through all of its ways: one launch, two, and three for more values than 4 GB of text have tiles."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIBRARY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "libscan_test.so")


@pytest.fixture(scope="module")
def scan():
    import torch
    assert torch.cuda.is_available(), "these tests need the MI355X"
    assert os.path.exists(LIBRARY), "build it with __graft_entry__.build() or make -C tests/cpp"
    lib = C.CDLL(LIBRARY)
    lib.scan_test.argtypes = [C.c_void_p, C.c_int64, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p]
    lib.scan_test_temp_bytes.restype, lib.scan_test_temp_bytes.argtypes = C.c_size_t, [C.c_int64]
    lib.scan_test_lines.restype, lib.scan_test_lines.argtypes = C.c_int64, [C.c_int]
    return lib


@pytest.mark.parametrize("tiles", ["one", "small", "direct", "beyond"])
@pytest.mark.parametrize("extra", [-1, 0, 1, 700])
def test_scan_of_so_many_tiles(scan, tiles, extra):
    """One value around a tile of the scan, the tiles that one launch does, those that two do, and more than twice those; values of up
    to 32 bits, whose sums have more."""
    import torch
    tile, small, direct = (scan.scan_test_lines(i) for i in range(3))
    n = tile * {"one": 1, "small": small, "direct": direct, "beyond": 2 * direct + 300}[tiles] + extra
    rng = np.random.default_rng(n)
    values = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    values[rng.random(n) < 0.3] = 0
    d = torch.from_numpy(values.view(np.int32)).cuda()
    out = torch.full((n + 2,), -7, dtype=torch.int64, device="cuda")
    temp_words = scan.scan_test_temp_bytes(n) // 8
    temp = torch.full((temp_words + 1,), -7, dtype=torch.int64, device="cuda")
    total = torch.full((1,), -7, dtype=torch.int64, device="cuda")
    assert scan.scan_test(d.data_ptr(), n, out.data_ptr(), temp.data_ptr(), total.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    expected = np.concatenate([[0], np.cumsum(values.astype(np.int64))])
    assert np.array_equal(out[: n + 1].cpu().numpy(), expected) and int(out[n + 1]) == -7
    assert int(total) == expected[-1] and int(temp[-1]) == -7
    assert int(temp[temp_words - 1]) == expected[-1]
