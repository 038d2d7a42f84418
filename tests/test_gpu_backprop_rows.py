"""Training backprop where the bag of every key position is found anew: batches
of one workgroup and of several 4,096-key tiles, one bag to more bags than keys,
bags that end at a tile's edge or span tiles, empty bags at either end,
positions before the first bag and after the last one, more bags in a tile than
its threads mark (8 each), and keys that need the sort on their exact bits.
Against the oracle, bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_backprop import gpu_backprop

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

TILE = 4096


def offsets_of(kind, n, rng):
    if kind == "one":
        cut = [0, n]
    elif kind == "edges":  # every bag ends at a multiple of a quarter tile
        cut = list(range(0, n, TILE // 4)) + [n]
    elif kind == "many":  # more bags than keys, most of them empty
        cut = np.sort(rng.integers(0, n + 1, size=2 * n + 3))
        cut[0], cut[-1] = 0, n
    elif kind == "marked":  # as many bags as are marked start at the last key
        cut = [0] + [n - 1] * (8 * 1024) + [n]
    elif kind == "searched":  # and one more
        cut = [0] + [n - 1] * (8 * 1024 + 1) + [n]
    elif kind == "sparse":  # many times more bags than keys, some keys outside them
        cut = np.sort(rng.integers(3, n - 2, size=70001))
    elif kind == "front":  # a key in each of the first bags, all others empty
        cut = np.concatenate([np.arange(n), np.full(50000, n)])
    elif kind == "outside":  # keys before the first bag and after the last
        cut = np.sort(rng.integers(n // 5, n - n // 5 + 1, size=70))
    else:  # 64 and 1,024 are the widths of a search step
        cut = np.sort(rng.integers(0, n + 1, size=int(kind) + 1))
        cut[0], cut[-1] = 0, n
        cut[1:4] = 0
        cut[-3:] = n
    return np.asarray(cut, np.int64)


@pytest.mark.parametrize("pooling", [O.SUM, O.MEAN, O.WSUM, O.WMEAN])
@pytest.mark.parametrize("kind", ["one", "edges", "many", "outside", "63", "64", "65", "1023", "1024", "1025",
                                  "marked", "searched", "sparse", "front"])
@pytest.mark.parametrize("n,wide", [(900, False), (TILE, False), (TILE + 1, False), (3 * TILE + 50, False),
                                    (2 * TILE + 7, True)])
def test_rows_of_every_position(n, wide, kind, pooling):
    rng = np.random.default_rng(n + 17 * pooling + len(kind))
    off = offsets_of(kind, n, rng)
    keys = (rng.zipf(1.2, size=n) % 3000).astype(np.int64)
    if wide:  # keys that differ above the bits the sort assumes
        keys = keys * (1 << 30) - (1 << 40)
    w = rng.uniform(0.1, 1.0, size=n).astype(np.float32) if pooling in (O.WSUM, O.WMEAN) else None
    g = rng.normal(0, 1, size=(off.size - 1, 20)).astype(np.float32)
    uq, out = gpu_backprop(keys, pooling, O.CSR, off, 0, w, O.F32, g, O.F32, 20)
    ruq, rout = O.pooling_backprop(keys, pooling, O.CSR, off, off.size - 1, 0, w, O.F32, g, O.F32, 20)
    assert np.array_equal(uq, ruq)
    assert np.array_equal(out, rout.view(np.uint32))


@pytest.mark.parametrize("pooling", [O.SUM, O.WMEAN])
@pytest.mark.parametrize("n,wide", [(200001, False), (262145, False), (600000, False), (1060000, False), (270000, True)])
def test_rows_of_many_tiles(n, wide, pooling):
    """A counting workgroup finds the rows of several tiles, of 2,048 and of 4,096 keys, and a first pass over either
    (behind the launch that adds counts up at 1,060,000 keys) carries them: bags over several tiles, thousands of
    empty ones between two keys, keys outside every bag."""
    rng = np.random.default_rng(n + pooling)
    cut = np.sort(np.concatenate([rng.integers(5000, n - 3000, size=n // 40), np.full(30000, 7 * TILE + 5),
                                  np.full(3000, 64 * TILE // 2 - 1)]))
    cut = cut[(cut < 20 * TILE) | (cut > 27 * TILE + 9)]  # a bag of seven tiles
    off = cut.astype(np.int64)
    keys = (rng.zipf(1.2, size=n) % 50000).astype(np.int64)
    if wide:
        keys = keys * (1 << 30) - (1 << 40)
    w = rng.uniform(0.1, 1.0, size=n).astype(np.float32) if pooling == O.WMEAN else None
    g = rng.normal(0, 1, size=(off.size - 1, 4)).astype(np.float32)
    uq, out = gpu_backprop(keys, pooling, O.CSR, off, 0, w, O.F32, g, O.F32, 4)
    ruq, rout = O.pooling_backprop(keys, pooling, O.CSR, off, off.size - 1, 0, w, O.F32, g, O.F32, 4)
    assert np.array_equal(uq, ruq)
    assert np.array_equal(out, rout.view(np.uint32))
