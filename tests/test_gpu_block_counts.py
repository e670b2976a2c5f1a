"""Tables whose codec groups take more blocks than one grid may have (2^32 threads),
because one long segment stands beside many short ones: what one launch can not
hold is split."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import fixed_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _constant():
    """int64: a segment of 2^23 rows (1024 blocks of output) beside 16,384 of one row each."""
    n0, n1 = 1 << 23, 16_384
    vals = np.arange(n1 + 1, dtype=np.int64) + 7
    d = torch.from_numpy(vals).cuda()
    segs = [A.Segment(d.data_ptr(), 8, 0, n0, 0)]
    segs += [A.Segment(d.data_ptr() + 8 * (i + 1), 8, n0 + i, 1, 0) for i in range(n1)]
    return A.CONSTANT, segs, np.concatenate([np.full(n0, 7), vals[1:]]).astype(np.int64), [d]


def _rle():
    """int8: a segment of 2^26 rows (8192 slices) beside 2,100 of two rows each."""
    n0, n1 = 1 << 26, 2_100
    long = E.encode_rle(np.full(n0, 3, np.int8), rg_rows=n0)
    short = E.encode_rle(np.repeat(np.arange(n1) % 100, 2).astype(np.int8), rg_rows=2)
    assert len(long.segs) == 1 and len(short.segs) == n1
    keep, segs = [], []
    for enc, base in ((long, 0), (short, n0)):
        d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
        for g in enc.segments(d.data_ptr()):
            g.row_offset += base
            segs.append(g)
        keep += [d, enc]
    return A.RLE, segs, np.concatenate([np.full(n0, 3), np.repeat(np.arange(n1) % 100, 2)]).astype(np.int8), keep


@pytest.mark.parametrize("beside", [False, True], ids=["alone", "beside"])
@pytest.mark.parametrize("make", [_constant, _rle], ids=["constant", "rle"])
@pytest.mark.parametrize("how", ["table", "batch"])
def test_more_blocks_than_a_grid(how, make, beside):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    codec, segs, want, keep = make()
    lib, s = L.load(), torch.cuda.current_stream().cuda_stream
    out = torch.zeros(want.size, dtype=getattr(torch, str(want.dtype)), device="cuda")
    cols = [fixed_column([(codec, segs)], want.dtype.itemsize, want.size, out.data_ptr())]
    small = torch.zeros(10, dtype=torch.int16, device="cuda")
    if beside:  # a second group shares the launch
        v = torch.tensor([5], dtype=torch.int16, device="cuda")
        cols.append(fixed_column([(A.CONSTANT, [A.Segment(v.data_ptr(), 2, 0, 10, 0)])], 2, want.size, small.data_ptr()))
    arr = (A.Column * len(cols))(*[c for c, _ in cols])
    print(f"[gpu] block counts {how} {make.__name__} beside={beside}", flush=True)
    if how == "table":
        L.check(lib.sdr_decode_table(arr, len(cols), s))
    else:
        b = C.c_void_p()
        L.check(lib.sdr_batch_create(C.byref(b)))
        L.check(lib.sdr_batch_add_table(b, arr, len(cols)))
        L.check(lib.sdr_batch_launch(b, s))
        L.check(lib.sdr_batch_finish(b, s))
        lib.sdr_batch_destroy(b)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), want)
    if beside:
        assert (small.cpu().numpy() == 5).all()
