"""Chunks whose lengths take long, ahead of short ones that wait for them: rows of
many kilobytes (walked by one thread), rows that fill several runs, each in the
first chunk, in one in the middle and in the last, in every launch mode and beside
another stream's decode.  Bit for bit as they were encoded."""
import ctypes as C
import threading

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import string_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
ROWS = 60_000


def _column(row, rows, length):
    """ROWS short strings of which `rows` from `row` on have `length` random bytes."""
    rng = np.random.default_rng(row + length)
    lens = rng.integers(0, 12, ROWS)
    lens[row:row + rows] = length
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    chars = rng.integers(0, 256, int(offs[-1]), dtype=np.uint8)
    enc = E.encode_fsst(chars, offs)
    d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
    o = torch.full((ROWS + 1,), -7, dtype=torch.int32, device="cuda")
    c = torch.full((chars.size + 32,), 0xCC, dtype=torch.uint8, device="cuda")
    col, k = string_column([(A.FSST, enc.segments(d.data_ptr()))], ROWS, o.data_ptr(), c.data_ptr(), chars.size + 32)

    def check():
        assert col.chars_used == chars.size
        np.testing.assert_array_equal(o.cpu().numpy(), offs.astype(np.int32))
        np.testing.assert_array_equal(c.cpu().numpy()[:chars.size], chars)
        assert (c.cpu().numpy()[chars.size:] == 0xCC).all()
        o.fill_(-7)
        c.fill_(0xCC)

    return col, check, [d, enc, k, o, c]


@pytest.mark.parametrize("rows,length", [(1, 40_000), (1000, 90)], ids=["one", "runs"])
@pytest.mark.parametrize("row", [0, 30_000, ROWS - 1000], ids=["first", "middle", "last"])
def test_long_rows(row, rows, length):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib, s = L.load(), torch.cuda.current_stream().cuda_stream
    col, check, keep = _column(row, rows, length)
    for mode in (A.LAUNCH_BATCHED, A.LAUNCH_PER_SEGMENT, A.LAUNCH_PERSISTENT):
        print(f"[gpu] long strings row={row} length={length} mode={mode}", flush=True)
        L.check(lib.sdr_decode_strings_column_mode(C.byref(col), s, mode))
        check()


def test_two_streams():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib = L.load()
    parts = [_column(30_000 * i, 1, 30_000) for i in range(2)]
    streams = [torch.cuda.Stream() for _ in parts]
    torch.cuda.synchronize()
    errors, start = [], threading.Barrier(2)

    def work(i):
        torch.cuda.set_device(0)
        start.wait()
        for _ in range(20):
            errors.append(lib.sdr_decode_strings_column(C.byref(parts[i][0]), streams[i].cuda_stream))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    print("[gpu] long strings on two streams", flush=True)
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert errors == [A.SDR_OK] * 40
    for _, check, _ in parts:
        check()
