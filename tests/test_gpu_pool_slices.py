"""Pooled lookups over rows cut into 16-, 8- and 4-byte slices at any alignment
(odd widths, quantized rows with their scale behind the values, rows of several
64-lane columns): the widths where a slice count, a slice width or the choice of
kernel changes, against the oracle.  Short bags are added in key order and must
equal it bit for bit; long bags are split, within the fp32 tolerance of their
order.  Tables and outputs start at odd element offsets and bytes around the
output must stay as they were."""
import numpy as np
import pytest

from nve_helpers import (csr_offsets, float_table, oracle_pool, pooled_f16_close, quant_table, rel_close, to_dev, vp,
                         stream_ptr)
from oracle import oracle as O
from pynve import _lib

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CDT = {O.F32: _lib.DT_F32, O.F16: _lib.DT_F16, O.QI8_F32: _lib.DT_QI8_F32, O.QI8_F16: _lib.DT_QI8_F16,
       O.QU8_F32: _lib.DT_QU8_F32, O.QU8_F16: _lib.DT_QU8_F16, O.XI8A_F32: _lib.DT_XI8A_F32,
       O.XE4M3_F32: _lib.DT_XE4M3_F32}
GUARD = 64

# (type, values per row): 31 / 32 / 33 bytes and 64 / 65, 128 / 129 (slice widths), 8 to 64 slices and one more
# (lane groups, columns), 4,096 bytes (the widest row of these kernels) and wider; of the byte rows past 512 those of
# whole 16-byte slices, whose 16 values a lane are stored through LDS, the second column's too
FLOATS = [(O.F16, d) for d in (15, 16, 17, 32, 33, 63, 65, 100, 129, 256, 512, 513, 2048, 2050)] + \
         [(O.F32, d) for d in (7, 8, 9, 16, 17, 31, 50, 65, 128, 255, 257, 600, 1024, 1025)]
QUANT = [(t, d) for t in (O.QI8_F32, O.QI8_F16, O.QU8_F32, O.QU8_F16, O.XI8A_F32, O.XE4M3_F32)
         for d in (30, 32, 34, 66, 128, 136, 300, 512, 514, 528, 1030, 2048)]


def pooled(tb, dtype, count, keys, pooling, off, w, out_dtype, shift):
    """The kernel-level pooled lookup with table and output `shift` elements past an aligned address."""
    rows, width = tb.shape
    es, oes = O.value_bytes(dtype), 2 if out_dtype == O.F16 else 4
    buf = torch.zeros(tb.size + 64, dtype=torch.uint8, device="cuda")
    table = buf[shift * es:shift * es + tb.size]
    table.copy_(torch.from_numpy(tb.reshape(-1)))
    bags = off.size - 1
    nb = bags * count * oes
    raw = torch.full((nb + 2 * GUARD,), 0xA5, dtype=torch.uint8, device="cuda")
    start = GUARD - 16 + shift * oes
    out = raw[start:start + nb]
    d_keys, d_off, d_w = to_dev(keys), to_dev(off), None if w is None else to_dev(w)
    _lib.call("nve_amd_find_and_pool", _lib.KEY_INT64, keys.size, vp(d_keys), vp(table), rows, width, CDT[dtype],
              pooling, _lib.SPARSE_CSR, vp(d_off), off.size, 0, vp(d_w), 0 if w is None else _lib.DT_F32,
              CDT[out_dtype], vp(out), count * oes, 0, 0, stream_ptr())
    torch.cuda.synchronize()
    raw = raw.cpu().numpy()
    assert np.all(raw[:start] == 0xA5) and np.all(raw[start + nb:] == 0xA5), "bytes around the output changed"
    return raw[start:start + nb].view(np.uint16 if out_dtype == O.F16 else np.float32).reshape(bags, count)


def check(dtype, count, pooling, lens, shift, exact, seed, out_dtype=None):
    rng = np.random.default_rng(seed)
    rows = 3000
    quant = O.meta_bytes(dtype) > 0
    tb = quant_table(rng, rows, count, dtype) if quant else float_table(rng, rows, count, dtype, dyadic_values=False)
    if out_dtype is None:
        out_dtype = dtype if not quant else O.F16 if dtype in (O.QI8_F16, O.QU8_F16) else O.F32
    off = np.zeros(len(lens) + 1, np.int64)
    off[1:] = np.cumsum(lens)
    keys = rng.integers(0, rows, size=int(off[-1])).astype(np.int64)
    keys[:: 5] = np.where(rng.uniform(size=keys[:: 5].size) < 0.5, rows - 1, 0)  # the table's first and last row
    absent = rng.uniform(size=keys.size) < 0.02
    weighted = pooling in (_lib.POOL_WSUM, _lib.POOL_WMEAN)
    w = rng.uniform(0, 1, size=keys.size).astype(np.float32) if weighted else None
    if weighted and pooling == _lib.POOL_WSUM:
        w[absent] = np.inf  # the weight of a key outside the table does not reach the sum
    asked = np.where(absent, rows + 7, keys)
    got = pooled(tb, dtype, count, asked, pooling, off, w, out_dtype, shift)
    padded = np.concatenate([tb, np.zeros((1, tb.shape[1]), np.uint8)])
    mapped = np.where(absent, rows, keys)
    w_ref = None if w is None else np.where(np.isfinite(w), w, 0).astype(np.float32)
    ref = oracle_pool(padded, mapped, dtype, count, O.CSR, pooling, off, len(lens), 0, w_ref, O.F32, out_dtype)
    if exact:
        bits = np.uint16 if out_dtype == O.F16 else np.uint32
        assert np.array_equal(got.view(bits), ref.view(bits))
    elif out_dtype == O.F16:
        assert pooled_f16_close(got.view(np.uint16), ref.view(np.uint16))
    else:
        # fp32 sums of n terms in another order differ by at most about n ulps of the largest partial sum;
        # 1e-5 of the row's magnitude is the repository's bound for the split order at these lengths
        assert rel_close(got, ref, 1e-5)


@pytest.mark.parametrize("shift", [0, 3])
@pytest.mark.parametrize("pooling", [_lib.POOL_SUM, _lib.POOL_WSUM, _lib.POOL_WMEAN])
@pytest.mark.parametrize("dtype,count", FLOATS + QUANT)
def test_short_bags_equal_the_oracle_bitwise(dtype, count, pooling, shift):
    rng = np.random.default_rng(count)
    lens = np.diff(csr_offsets(rng, 70, 40))
    check(dtype, count, pooling, lens, shift, True, 31 * count + pooling)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("dtype", [O.XI8A_F32, O.XE4M3_F32])
@pytest.mark.parametrize("count", [34, 136, 300, 528, 1024, 1030, 2048])
def test_fp32_scaled_bytes_to_fp16(dtype, count, shift):
    lens = np.diff(csr_offsets(np.random.default_rng(count), 70, 40))
    check(dtype, count, _lib.POOL_WMEAN, lens, shift, True, count, O.F16)


@pytest.mark.parametrize("pooling", [_lib.POOL_MEAN, _lib.POOL_WMEAN])
@pytest.mark.parametrize("dtype,count", FLOATS + QUANT)
def test_long_bags_within_tolerance(dtype, count, pooling):
    lens = np.array([0, 700, 33, 1, 90, 1024, 64, 257])
    check(dtype, count, pooling, lens, 1, False, 17 * count + pooling)


@pytest.mark.parametrize("out", [O.F16, O.F32])
@pytest.mark.parametrize("dtype,count", [(O.F16, 100), (O.F16, 128), (O.F32, 36), (O.F16, 33), (O.F16, 520),
                                         (O.F16, 1024), (O.F32, 300)])
def test_several_tables_of_bags_that_fill_no_workgroup(dtype, count, out):
    """Bags per table that are no multiple of a workgroup's, tables at odd offsets: each output column bitwise."""
    rng = np.random.default_rng(count)
    tables, bags = [float_table(rng, r, count, dtype, dyadic_values=False) for r in (50, 1, 700)], 37
    lens = rng.integers(0, 30, size=3 * bags)
    off = np.zeros(lens.size + 1, np.int64)
    off[1:] = np.cumsum(lens)
    keys = np.concatenate([rng.integers(0, tables[t].shape[0], size=int(off[(t + 1) * bags] - off[t * bags]))
                           for t in range(3)]).astype(np.int64)
    es, oes = O.value_bytes(dtype), 2 if out == O.F16 else 4
    dev = []
    for t in tables:
        buf = torch.zeros(t.size + 64, dtype=torch.uint8, device="cuda")
        v = buf[es:es + t.size]
        v.copy_(torch.from_numpy(t.reshape(-1)))
        dev.append(v)
    d_out = torch.zeros(bags * 3 * count * oes, dtype=torch.uint8, device="cuda")
    ptrs = (_lib.P * 3)(*[t.data_ptr() for t in dev])
    rows = (_lib.I64 * 3)(*[t.shape[0] for t in tables])
    d_keys, d_off = to_dev(keys), to_dev(off)
    _lib.call("nve_amd_find_and_pool_multi", _lib.KEY_INT64, 3, ptrs, rows, tables[0].shape[1], CDT[dtype], bags,
              keys.size, vp(d_keys), vp(d_off), None, 0, _lib.POOL_MEAN, CDT[out], vp(d_out), stream_ptr())
    torch.cuda.synchronize()
    bits = np.uint16 if out == O.F16 else np.uint32
    got = d_out.cpu().numpy().view(bits).reshape(bags, 3, count)
    for t in range(3):
        s, e = off[t * bags], off[(t + 1) * bags]
        ref = oracle_pool(tables[t], keys[s:e], dtype, count, O.CSR, O.MEAN, off[t * bags:(t + 1) * bags + 1] - s, bags,
                          0, None, 0, out)
        assert np.array_equal(got[:, t], ref.view(bits))


# rows under 32 bytes (the general kernel) in groups of 1, 2, 4, 8 and 16 lanes; numbers of bags on both sides of the
# lines where such a bag's share of a wave changes
@pytest.mark.parametrize("bags", [300, 3100, 6200, 12300, 33000])
@pytest.mark.parametrize("dtype,count", [(O.F16, 4), (O.F16, 12), (O.F32, 4), (O.F32, 7), (O.QI8_F32, 8), (O.QU8_F32, 30)])
def test_narrow_rows_in_bags_of_a_few_dozen_keys(dtype, count, bags):
    lens = np.random.default_rng(bags).integers(20, 60, size=bags)
    check(dtype, count, _lib.POOL_WMEAN if count % 8 else _lib.POOL_SUM, lens, 0, False, bags + count)


@pytest.mark.parametrize("dtype,count,bags,pooling,whole", [
    (O.F16, 64, 16384, _lib.POOL_WSUM, True), (O.F16, 64, 16383, _lib.POOL_WSUM, False),
    (O.F32, 64, 8192, _lib.POOL_SUM, True), (O.F32, 64, 8191, _lib.POOL_SUM, False),
    (O.QI8_F32, 130, 4096, _lib.POOL_WMEAN, True),
    (O.QI8_F32, 130, 4095, _lib.POOL_WMEAN, False), (O.F16, 256, 50, _lib.POOL_WMEAN, True),
    (O.F16, 256, 50, _lib.POOL_MEAN, False), (O.F16, 256, 4096, _lib.POOL_MEAN, True)])
def test_bags_of_a_few_dozen_keys(dtype, count, bags, pooling, whole):
    """Bags of 33 to 64 keys on both sides of the lines where a wave shares a bag: one added by a single group equals
    the oracle bit for bit, one that is cut stays within the tolerance of its order."""
    lens = np.random.default_rng(bags).integers(25, 70, size=bags)
    check(dtype, count, pooling, lens, 1, whole, bags + count)


@pytest.mark.parametrize("lens,bags", [((0, 5), 3000), ((10, 40), 8192), ((8, 20), 33000), ((50, 70), 8192)],
                         ids=["up_to_4_keys", "more_bytes", "more_waves", "past_48_keys"])
@pytest.mark.parametrize("dtype,count", [(t, d) for t in (O.QI8_F32, O.QI8_F16, O.QU8_F32, O.QU8_F16, O.XI8A_F32, O.XE4M3_F32)
                                         for d in (130, 514)] + [(O.F16, 66)])
def test_metadata_loaded_with_the_row(dtype, count, lens, bags):
    """Launches whose rows pass the size up to which metadata is loaded ahead, in every number of rows in flight; keys
    outside the table and slots past the end of a bag read the zero row's metadata."""
    if count == 514:
        bags //= 2
    lens = np.random.default_rng(bags).integers(lens[0], lens[1], size=bags)
    check(dtype, count, _lib.POOL_WSUM, lens, 1, lens.mean() < 50 or count != 514, bags + count)
