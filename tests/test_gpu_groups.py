"""Tables whose codec groups and null masks share a launch: every codec and
width beside the others, as many segments as one launch's arguments hold, a few
more (the groups are cut between launches) and so many that they are uploaded.
Equal to the encoded values; the masks and null counts to the validity bits."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import fixed_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
SEG = 2048


def _columns(rows, rng):
    f32, f64 = np.round(rng.random(rows) * 900, 2).astype(np.float32), np.round(rng.random(rows) * 90_000, 2)
    runs = np.repeat(rng.integers(0, 99, rows), rng.integers(1, 40, rows))[:rows]
    return [(A.BITPACKING, rng.integers(0, 100, rows).astype(t), E.encode_bitpacking)
            for t in (np.int8, np.int16, np.int32, np.int64)] + \
           [(A.RLE, runs.astype(t), E.encode_rle) for t in (np.int8, np.int16, np.int32, np.int64)] + \
           [(A.ALP, f32, E.encode_alp), (A.ALP, f64, E.encode_alp),
            (A.ALPRD, rng.random(rows).astype(np.float32), E.encode_alprd), (A.ALPRD, rng.random(rows), E.encode_alprd),
            (A.UNCOMPRESSED, rng.integers(-9, 9, rows), E.encode_uncompressed), (A.CONSTANT, np.full(rows, 77, np.int32), None)]


@pytest.mark.parametrize("segs", [1, 9, 10, 300])
@pytest.mark.parametrize("mode", [A.LAUNCH_BATCHED, A.LAUNCH_PER_SEGMENT], ids=["batched", "plain"])
def test_all_groups(mode, segs):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(segs)
    rows = segs * SEG - 5
    cols, keep, checks = [], [], []
    for i, (codec, values, encode) in enumerate(_columns(rows, rng)):
        ts = values.dtype.itemsize
        if encode:
            enc = encode(values, rg_rows=SEG)
            d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
            table = enc.segments(d.data_ptr())
        else:
            d = torch.from_numpy(np.concatenate([values[:1].view(np.uint8), np.zeros(64, np.uint8)])).cuda()
            table = [A.Segment(d.data_ptr(), ts, r, min(SEG, rows - r), 0) for r in range(0, rows, SEG)]
        assert len(table) >= segs
        out = torch.full((rows * ts + 64,), 0xCC, dtype=torch.uint8, device="cuda")
        nb, bits, m, validity = (rows + 7) // 8, None, None, None
        if i % 3 == 0:
            bits = rng.integers(0, 256, nb, dtype=np.uint8)
            v = torch.from_numpy(bits).cuda()
            m = torch.full((nb + 32,), 0xA5, dtype=torch.uint8, device="cuda")
            validity = [(A.UNCOMPRESSED, [A.Segment(v.data_ptr() + r // 8, (min(SEG, rows - r) + 7) // 8, r,
                                                    min(SEG, rows - r), 0) for r in range(0, rows, SEG)])]
            keep.append(v)
        col, k = fixed_column([(codec, table)], ts, rows, out.data_ptr(), validity, m.data_ptr() if validity else None)
        cols.append(col)
        keep += [d, k, out]
        checks.append((values, out, bits, m))
    arr = (A.Column * len(cols))(*cols)
    print(f"[gpu] groups segs={segs} mode={mode}", flush=True)
    L.check(L.load().sdr_decode_table_mode(arr, len(cols), torch.cuda.current_stream().cuda_stream, mode))
    torch.cuda.synchronize()
    for c, (values, out, bits, m) in enumerate(checks):
        got = out.cpu().numpy()
        np.testing.assert_array_equal(got[:values.nbytes], values.view(np.uint8).reshape(-1), err_msg=str(c))
        assert (got[values.nbytes:] == 0xCC).all()
        if bits is not None:
            got = m.cpu().numpy()
            np.testing.assert_array_equal(got[:bits.size], bits)
            assert (got[bits.size:] == 0xA5).all()
            assert arr[c].null_count == rows - int(np.unpackbits(bits, bitorder="little")[:rows].sum())


@pytest.mark.parametrize("segs", [1023, 1024, 1025, 1300])
@pytest.mark.parametrize("which", ["alp4", "alp8", "alprd8", "copy8"])
def test_blocks_of_one_group(which, segs):
    """One segment less, as many and one more than the blocks a launch takes in
    the order of the dies, and some past its last whole turn."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(segs)
    rows = segs * SEG - 5
    i = {"alp4": 8, "alp8": 9, "alprd8": 11, "copy8": 12}[which]
    codec, values, encode = _columns(rows, rng)[i]
    ts = values.dtype.itemsize
    enc = encode(values, rg_rows=SEG)
    d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
    out = torch.full((rows * ts + 64,), 0xCC, dtype=torch.uint8, device="cuda")
    col, keep = fixed_column([(codec, enc.segments(d.data_ptr()))], ts, rows, out.data_ptr())
    print(f"[gpu] one group {which} segs={segs}", flush=True)
    L.check(L.load().sdr_decode_table(C.byref(col), 1, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:values.nbytes], values.view(np.uint8).reshape(-1))
    assert (got[values.nbytes:] == 0xCC).all()
