"""The sorted dedup at the sizes where its work is cut anew: the single
workgroup's 1 and 4 keys per thread (1,024 and 4,096 keys) and the
first size past them, the radix sort's tiles of 2,048 keys (up to 229,376 keys) and
of 4,096, its 64 count groups and the launch that adds counts up (beyond 256
tiles), the run outputs' tiles of 4,096 positions and 64 of them looked back
over at a time; with keys whose
digits pile up in one bin, all equal (one run over every tile), descending, or
spread over all 64 bits."""
import ctypes

import numpy as np
import pytest

from nve_helpers import stream_ptr, to_dev, vp
from pynve import _lib

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TILE = 4096


def make(kind, n, rng):
    if kind == "table":  # rows of a table: the 27-bit passes
        return (rng.random(n) ** 4 * 5e7).astype(np.int64)
    if kind == "wide":  # every bit, both signs: sorted again on the exact bits
        return rng.integers(-2**63, 2**63 - 1, size=n, dtype=np.int64)
    if kind == "one":
        return np.full(n, 12345, np.int64)
    if kind == "descending":
        return np.arange(n, 0, -1).astype(np.int64)
    hot = np.where(rng.random(n) < 0.9, 7, rng.integers(0, 1 << 20, size=n))
    return hot.astype(np.int64)


@pytest.mark.parametrize("n", [100, 1024, 3000, 8192, 8193, 20000])
def test_int32_keys(n):
    rng = np.random.default_rng(n)
    keys = rng.integers(-2**31, 2**31 - 1, size=n).astype(np.int32)
    keys[rng.random(n) < 0.4] = -5
    need = ctypes.c_uint64()
    _lib.call("nve_amd_dedup_workspace_size", n, ctypes.byref(need))
    ws = torch.empty(need.value, dtype=torch.uint8, device="cuda")
    out = [torch.zeros(n + 1, dtype=torch.int32, device="cuda") for _ in range(4)]
    num, d_keys = ctypes.c_int64(), to_dev(keys)
    _lib.call("nve_amd_dedup", _lib.KEY_INT32, n, vp(d_keys), vp(out[0]), vp(out[1]), vp(out[2]), vp(out[3]),
              ctypes.byref(num), vp(ws), need.value, stream_ptr())
    unique, counts = np.unique(keys, return_counts=True)
    got = [t.cpu().numpy() for t in out]
    assert num.value == unique.size
    assert np.array_equal(got[0][:num.value], unique) and np.array_equal(got[1][:num.value], counts)
    assert np.array_equal(got[2][:n], np.argsort(keys, kind="stable"))


@pytest.mark.parametrize("kind", ["table", "wide", "one", "descending", "hot"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, TILE - 1, TILE, TILE + 1, 2 * TILE - 1, 2 * TILE,
                               2 * TILE + 1, 3 * TILE + 17, 16 * TILE, 16 * TILE + 1025, 63 * TILE + 1, 64 * TILE,
                               65 * TILE + 5, 128 * TILE, 128 * TILE + 1, 256 * TILE, 256 * TILE + 1, 300 * TILE + 9])
def test_dedup_equals_numpy(kind, n):
    if n > 65 * TILE + 5 and kind in ("wide", "descending"):
        n = 129 * TILE + 3
    rng = np.random.default_rng(n)
    keys = make(kind, n, rng)
    need = ctypes.c_uint64()
    _lib.call("nve_amd_dedup_workspace_size", n, ctypes.byref(need))
    ws = torch.full((need.value,), 0xEE, dtype=torch.uint8, device="cuda")
    out = [torch.zeros(n + 1, dtype=torch.int64, device="cuda") for _ in range(4)]
    num, d_keys = ctypes.c_int64(), to_dev(keys)
    for _ in range(2):  # the second call finds the first one's state in its workspace
        _lib.call("nve_amd_dedup", _lib.KEY_INT64, n, vp(d_keys), vp(out[0]), vp(out[1]), vp(out[2]), vp(out[3]),
                  ctypes.byref(num), vp(ws), need.value, stream_ptr())
        unique, start, counts = np.unique(keys, return_index=True, return_counts=True)
        u = num.value
        assert u == unique.size
        got = [t.cpu().numpy() for t in out]
        assert np.array_equal(got[0][:u], unique)
        assert np.array_equal(got[1][:u], counts)
        assert np.array_equal(got[2][:n], np.argsort(keys, kind="stable"))
        assert np.array_equal(got[3][:u], np.cumsum(counts) - counts)


@pytest.mark.parametrize("kind", ["table", "wide", "hot"])
@pytest.mark.parametrize("n", [4097, 6143, 6144, 6145, 8191, 131072, 131073, 229376 - 2048, 229375, 229376, 229377, 233473,
                               262144 - 2048, 262143, 262144, 262145, 266241])
def test_two_round_tiles(kind, n):
    test_dedup_equals_numpy(kind, n)


def test_workspace_of_more_keys_serves_fewer():
    """A workspace sized for n keys is taken for every smaller batch, also across a change of tile size."""
    need, last = ctypes.c_uint64(), 0
    for n in [1, 4096, 4097, 8192, 131072, 229375, 229376, 229377, 229400, 240000, 262143, 262144, 262145, 262200,
              280000, 458752, 524288, 600000]:
        _lib.call("nve_amd_dedup_workspace_size", n, ctypes.byref(need))
        assert need.value >= last, n
        last = need.value
