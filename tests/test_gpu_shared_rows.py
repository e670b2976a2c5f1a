"""Runs of different codecs that share rows, columns that share an output, columns
that share a null mask: the codec whose first run comes later (in a batch, in the
order bit-packed, RLE, uncompressed, constant), or the later column, wins, as when
each is a launch of its own, however many segments there are."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import fixed_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
N = 4_000_000


def _encoded(codec, values, base, rg):
    """(codec, segments of rows [base, base + len(values))) and what they keep alive."""
    if codec == A.CONSTANT:
        d = torch.from_numpy(np.concatenate([values[:1].view(np.uint8), np.zeros(64, np.uint8)])).cuda()
        return [A.Segment(d.data_ptr(), values.dtype.itemsize, base, values.size, 0)], [d]
    encode = {A.BITPACKING: E.encode_bitpacking, A.RLE: E.encode_rle, A.UNCOMPRESSED: E.encode_uncompressed}[codec]
    enc = encode(values, rg_rows=rg)
    d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
    segs = enc.segments(d.data_ptr())
    for g in segs:
        g.row_offset += base
    return segs, [d, enc]


def _runs(order, rg):
    """Runs of the codecs in this order, each over fewer rows than the one before, and the values that remain."""
    rng = np.random.default_rng(len(order))
    want, runs, keep = np.zeros(N, np.int32), [], []
    for i, codec in enumerate(order):
        lo, hi = i * (N // 10), N - i * (N // 9)
        v = rng.integers(1000 * i, 1000 * i + 900, hi - lo).astype(np.int32)
        if codec == A.RLE:
            v = np.repeat(v, 5)[:hi - lo]
        if codec == A.CONSTANT:
            v[:] = v[0]
        segs, k = _encoded(codec, v, lo, rg)
        runs.append((codec, segs))
        keep += k
        want[lo:hi] = v
    return runs, want, keep


def _decode(how, cols):
    """Decode the list of columns and wait."""
    lib, s = L.load(), torch.cuda.current_stream().cuda_stream
    arr = (A.Column * len(cols))(*cols)
    if how == "batch":
        b = C.c_void_p()
        L.check(lib.sdr_batch_create(C.byref(b)))
        for col in arr:
            L.check(lib.sdr_batch_add_table(b, C.byref(col), 1))
        L.check(lib.sdr_batch_launch(b, s))
        L.check(lib.sdr_batch_finish(b, s))
        lib.sdr_batch_destroy(b)
    elif how == "plan":
        p = C.c_void_p()
        L.check(lib.sdr_plan_create(arr, len(cols), A.LAUNCH_BATCHED, s, C.byref(p)))
        L.check(lib.sdr_plan_launch(p, s))
        counts = (C.c_int64 * len(cols))()
        L.check(lib.sdr_plan_null_counts(p, counts, len(cols), s))
        lib.sdr_plan_destroy(p)
        return list(counts)
    else:
        L.check(lib.sdr_decode_table(arr, len(cols), s))
    torch.cuda.synchronize()
    return [c.null_count for c in arr]


ORDERS = {"up": [A.BITPACKING, A.RLE, A.UNCOMPRESSED, A.CONSTANT], "down": [A.CONSTANT, A.UNCOMPRESSED, A.RLE, A.BITPACKING],
          "mixed": [A.RLE, A.CONSTANT, A.BITPACKING, A.UNCOMPRESSED]}


@pytest.mark.parametrize("rg", [2_000_000, 8192], ids=["few", "many"])
@pytest.mark.parametrize("order", ["up", "down", "mixed"])
@pytest.mark.parametrize("how", ["table", "plan", "batch"])
def test_later_codec_wins(how, order, rg):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if how == "batch" and order != "up":
        pytest.skip("a batch takes codecs in its own order")
    runs, want, keep = _runs(ORDERS[order], rg)
    out = torch.zeros(N, dtype=torch.int32, device="cuda")
    col, k = fixed_column(runs, 4, N, out.data_ptr())
    print(f"[gpu] shared rows {how} {order} rg={rg}", flush=True)
    _decode(how, [col])
    np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("how", ["table", "plan", "batch"])
def test_columns_that_share_outputs(how):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(3)
    a, b = rng.integers(0, 500, N).astype(np.int32), rng.integers(500, 900, N // 2).astype(np.int32)
    sa, ka = _encoded(A.BITPACKING, a, 0, 122_880)
    sb, kb = _encoded(A.UNCOMPRESSED, b, 0, 122_880)
    out = torch.zeros(N, dtype=torch.int32, device="cuda")
    mask = torch.zeros(N // 8, dtype=torch.uint8, device="cuda")
    bits = [rng.integers(0, 256, n // 8, dtype=np.uint8) for n in (N, N // 2)]
    vs = [torch.from_numpy(x).cuda() for x in bits]
    cols, keep = [], []
    for segs, codec, n, v in ((sa, A.BITPACKING, N, vs[0]), (sb, A.UNCOMPRESSED, N // 2, vs[1])):
        col, k = fixed_column([(codec, segs)], 4, N, out.data_ptr(),
                              [(A.UNCOMPRESSED, [A.Segment(v.data_ptr(), n // 8, 0, n, 0)])], mask.data_ptr())
        cols.append(col)
        keep.append(k)
    print(f"[gpu] shared outputs {how}", flush=True)
    counts = _decode(how, cols)
    np.testing.assert_array_equal(out.cpu().numpy(), np.concatenate([b, a[N // 2:]]))
    # a column's mask is all valid where no validity segment lies
    np.testing.assert_array_equal(mask.cpu().numpy(), np.concatenate([bits[1], np.full(N // 16, 0xFF, np.uint8)]))
    assert counts == [int((~np.unpackbits(x).astype(bool)).sum()) for x in bits]
