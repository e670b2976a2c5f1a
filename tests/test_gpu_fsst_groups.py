"""FSST chunks at the edges of the 16-byte-group decode: rows shorter than a
group, chunks at the most compressed bytes the groups hold and past it, output
past one window, escapes on group and row boundaries, last chunks of every
size.  Offsets and chars equal the oracle's, byte for byte."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from oracle import oracle as O
from sirius_amd import lib as L
from tests.helpers import string_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
MODES = [A.LAUNCH_BATCHED, A.LAUNCH_PERSISTENT]


def _rows(name, rng):
    """Row lengths and a char source of one shape."""
    if name == "tiny":  # up to 16 rows in a group, empty rows among them
        return rng.integers(0, 4, 9_000), np.frombuffer(b"ab cde", np.uint8)
    if name == "empty_runs":
        return rng.integers(1, 30, 5_000) * (rng.random(5_000) < 0.05), np.frombuffer(b"xyz01", np.uint8)
    if name == "escapes":  # two compressed bytes per char, literal 255s among them
        return rng.integers(0, 24, 6_000), np.arange(256, dtype=np.uint8)
    if name == "brim":  # chunks of 16 KiB of compressed bytes, give or take some tens
        return 16 - (rng.random(41_000) < np.linspace(0.02, 0.10, 41_000)), np.arange(256, dtype=np.uint8)
    if name == "windows":  # a chunk decodes to several windows, cut inside rows and symbols
        return rng.integers(20, 160, 5_000), np.frombuffer(b"01234567", np.uint8)
    if name == "runs":  # a chunk's rows take several runs, one of them empty rows alone
        return np.where((np.arange(6_000) % 1024 < 700) & (np.arange(6_000) % 1024 > 500), 0, rng.integers(10, 120, 6_000)), \
            np.arange(64, 120, dtype=np.uint8)
    if name == "wide_row":  # a row longer than any run holds
        return np.where(np.arange(2_500) == 1200, 30_000, rng.integers(10, 60, 2_500)), np.arange(64, 120, dtype=np.uint8)
    if name == "long_row":
        return np.where(np.arange(3_000) == 1500, 60_000, rng.integers(0, 9, 3_000)), np.frombuffer(b"01234567", np.uint8)
    return rng.integers(5, 25, int(name)), np.frombuffer(b"the quick brown fox ", np.uint8)


def _encode(name):
    rng = np.random.default_rng(sum(map(ord, name)))
    lens, source = _rows(name, rng)
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    n = int(offs[-1])
    chars = rng.choice(source, n) if source.size > 8 or name == "tiny" else np.resize(source, n)
    return E.encode_fsst(chars.astype(np.uint8), offs)


def _check(enc, mode, skew):
    o_offs, o_chars = O.decode_strings(enc)
    dev = torch.device("cuda:0")
    d = torch.zeros(enc.blob.size + skew + 256, dtype=torch.uint8, device=dev)
    d[skew:skew + enc.blob.size] = torch.from_numpy(enc.blob).to(dev)
    n, cap = enc.n_rows, o_chars.size
    offs = torch.full((n + 1,), -7, dtype=torch.int32, device=dev)
    chars = torch.full((cap + skew + 64,), 0xCC, dtype=torch.uint8, device=dev)
    col, keep = string_column([(A.FSST, enc.segments(d.data_ptr() + skew))], n, offs.data_ptr(),
                              chars.data_ptr() + skew, cap)
    print(f"[gpu] fsst groups rows={n} mode={mode} skew={skew}", flush=True)
    L.check(L.load().sdr_decode_strings_column_mode(C.byref(col), torch.cuda.current_stream().cuda_stream, mode))
    torch.cuda.synchronize()
    got = chars.cpu().numpy()
    np.testing.assert_array_equal(offs.cpu().numpy(), o_offs)
    np.testing.assert_array_equal(got[skew:skew + cap], o_chars)
    assert (got[:skew] == 0xCC).all() and (got[skew + cap:] == 0xCC).all()  # nothing written around them


@pytest.mark.parametrize("mode", MODES, ids=["batched", "persistent"])
@pytest.mark.parametrize("name", ["tiny", "empty_runs", "escapes", "brim", "windows", "runs", "wide_row", "long_row",
                                  "1", "2", "63", "1023", "1025", "2049"])
def test_shapes(name, mode):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    enc = _encode(name)
    for skew in (0, 1, 6, 11, 15):
        _check(enc, mode, skew)


@pytest.mark.parametrize("share", [0.003, 0.1, 0.6])
def test_bytes_turned_into_escapes(share):
    """Compressed bytes overwritten with 255: escapes that end rows, runs of
    them across rows and groups."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    enc = _encode("5000")
    rng = np.random.default_rng(7)
    for s in enc.segs:
        head = enc.blob[int(s["offset"]):int(s["offset"]) + 16].view("<u4")
        width, end, rows = int(head[2]), int(head[1]), int(s["row_count"])
        bits = enc.blob[int(s["offset"]) + 16:int(s["offset"]) + 16 + (rows * width + 7) // 8]
        bits = np.unpackbits(bits, bitorder="little")[:rows * width].reshape(rows, width)
        total = int((bits << np.arange(width)).sum())  # compressed bytes: the last `total` before dict_end
        data = enc.blob[int(s["offset"]) + end - total:int(s["offset"]) + end]
        data[rng.random(total) < share] = 255
    for mode in MODES:
        _check(enc, mode, 5)
