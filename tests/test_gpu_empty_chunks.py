"""FSST chunks without a byte: in the first, a middle and the last place of a column,
all of it, and beside segments with a bad header and rows of no segment.  The
offsets run on through them in every launch mode."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import string_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
ROWS = 9_000


@pytest.mark.parametrize("empty", [(0, 2048), (3000, 6000), (7000, ROWS), (0, ROWS), (1, ROWS), (0, ROWS - 1)], ids=str)
@pytest.mark.parametrize("bad", [False, True], ids=["sound", "bad"])
def test_empty_chunks(empty, bad):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(empty[0] + 1)
    lens = rng.integers(1, 30, ROWS)
    lens[empty[0]:empty[1]] = 0
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    chars = rng.integers(97, 123, int(offs[-1]), dtype=np.uint8)
    enc = E.encode_fsst(chars, offs)
    d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(256, np.uint8)])).cuda()
    segs = enc.segments(d.data_ptr())
    gap = 1500 if bad else 0  # before the rows: some of no segment, some of one whose header is all zero
    for g in segs:
        g.row_offset += gap
    if bad:
        segs.insert(0, A.Segment(d.data_ptr() + enc.blob.size, 64, 300, 1100, 0))
    total = ROWS + gap
    want = np.concatenate([np.zeros(gap), offs]).astype(np.int32)
    o = torch.full((total + 1,), -7, dtype=torch.int32, device="cuda")
    c = torch.full((chars.size + 32,), 0xCC, dtype=torch.uint8, device="cuda")
    col, keep = string_column([(A.FSST, segs)], total, o.data_ptr(), c.data_ptr(), chars.size + 32)
    for mode in (A.LAUNCH_BATCHED, A.LAUNCH_PER_SEGMENT, A.LAUNCH_PERSISTENT):
        print(f"[gpu] empty chunks {empty} bad={bad} mode={mode}", flush=True)
        L.check(L.load().sdr_decode_strings_column_mode(C.byref(col), torch.cuda.current_stream().cuda_stream, mode))
        assert col.chars_used == chars.size
        np.testing.assert_array_equal(o.cpu().numpy(), want)
        np.testing.assert_array_equal(c.cpu().numpy()[:chars.size], chars)
        assert (c.cpu().numpy()[chars.size:] == 0xCC).all()
        o.fill_(-7)
        c.fill_(0xCC)
