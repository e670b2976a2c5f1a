"""DICTIONARY, UNCOMPRESSED and DICT_FSST rows at the edges of the word-wise
copy: every alignment of a row's source and of its place in the output, rows
of 0 to 40 bytes, rows cut by the output window and longer than it, segments
and chars at odd addresses.  Equal to the oracle, byte for byte."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import (StringBlob, dictionary_string_segment, duckdb_segments, oracle_string_runs, string_column,
                           uncompressed_string_segment)

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
MODES = [A.LAUNCH_BATCHED, A.LAUNCH_PERSISTENT]


def _strings(name):
    rng = np.random.default_rng(sum(map(ord, name)))
    if name == "lengths":
        lens = rng.integers(0, 41, 5_000)
    elif name == "windows":  # a chunk's output passes the window several times
        lens = rng.integers(0, 400, 2_500)
    elif name == "long":  # rows longer than the window
        lens = np.where(rng.random(1_500) < 0.004, rng.integers(39_000, 90_000, 1_500), rng.integers(0, 5, 1_500))
    else:
        lens = rng.integers(1, 9, int(name))
    return [rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in lens]


def _decode(segs_of, total, cap, mode, skew):
    offs = torch.full((total + 1,), -7, dtype=torch.int32, device="cuda")
    chars = torch.full((cap + skew + 64,), 0xCC, dtype=torch.uint8, device="cuda")
    mask = torch.zeros((total + 7) // 8, dtype=torch.uint8, device="cuda")
    col, keep = string_column(segs_of, total, offs.data_ptr(), chars.data_ptr() + skew, cap)
    col.d_null_mask = mask.data_ptr()  # DICT_FSST's NULL slot needs one
    L.check(L.load().sdr_decode_strings_column_mode(C.byref(col), torch.cuda.current_stream().cuda_stream, mode))
    torch.cuda.synchronize()
    got = chars.cpu().numpy()
    assert (got[:skew] == 0xCC).all() and (got[skew + cap:] == 0xCC).all()
    return offs.cpu().numpy(), got[skew:skew + cap]


@pytest.mark.parametrize("name", ["lengths", "windows", "long", "1", "1024", "1025"])
@pytest.mark.parametrize("codec", ["dictionary", "uncompressed"])
def test_rows(codec, name):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    strings = _strings(name)
    if codec == "dictionary":  # entries drawn again, some of them NULL
        rng = np.random.default_rng(3)
        strings = [None if k % 17 == 3 else strings[k] for k in rng.integers(0, len(strings), len(strings))]
    b = StringBlob()
    cid = A.DICTIONARY if codec == "dictionary" else A.UNCOMPRESSED
    enc = dictionary_string_segment if codec == "dictionary" else uncompressed_string_segment
    b.add(cid, enc(strings), 0, len(strings))
    table = np.array(b.table, np.int64)
    o_offs, o_chars = oracle_string_runs(b.blob, table, len(strings))
    for skew in (0, 1, 2, 3, 13):
        d = torch.zeros(b.blob.size + skew + 64, dtype=torch.uint8, device="cuda")
        d[skew:skew + b.blob.size] = torch.from_numpy(b.blob)
        print(f"[gpu] plain rows {codec} {name} skew={skew}", flush=True)
        for mode in MODES:
            offs, chars = _decode(duckdb_segments(table, d.data_ptr() + skew), len(strings), o_chars.size, mode, 15 - skew)
            np.testing.assert_array_equal(offs, o_offs)
            np.testing.assert_array_equal(chars, o_chars)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_dict_fsst_rows(mode):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    strings = _strings("lengths")
    offs = np.concatenate([[0], np.cumsum([len(s) for s in strings])]).astype(np.uint64)
    chars = np.frombuffer(b"".join(strings), np.uint8)
    enc = E.encode_dict_fsst(chars, offs, mode, seg_rows=3000)
    for skew in (0, 5):
        d = torch.zeros(enc.blob.size + skew + 64, dtype=torch.uint8, device="cuda")
        d[skew:skew + enc.blob.size] = torch.from_numpy(enc.blob)
        print(f"[gpu] plain rows dict_fsst mode={mode} skew={skew}", flush=True)
        g_offs, g_chars = _decode([(A.DICT_FSST, enc.segments(d.data_ptr() + skew))], len(strings), chars.size,
                                  A.LAUNCH_BATCHED, skew)
        np.testing.assert_array_equal(g_offs.astype(np.uint64), offs)
        np.testing.assert_array_equal(g_chars, chars)


def _label_segment(words, sel):
    """A DICTIONARY segment of the rows words[sel] (entry 0 is NULL)."""
    width = len(words).bit_length()
    bits = np.packbits(((sel[:, None] >> np.arange(width)) & 1).astype(np.uint8).reshape(-1), bitorder="little")
    ends = np.cumsum([0] + [len(x) for x in words[1:]]).astype("<u4")
    ibo = 20 + bits.size + (-bits.size) % 4
    body = b"".join(reversed(words[1:]))
    head = np.array([len(body), ibo + ends.nbytes + len(body), ibo, ends.size, width], "<u4")
    return head.tobytes() + bits.tobytes() + bytes(ibo - 20 - bits.size) + ends.tobytes() + body


@pytest.mark.parametrize("longest", [9, 60], ids=["one_window", "windows"])
@pytest.mark.parametrize("rows", [1_048_575, 1_049_601, 2_097_151, 2_097_153])
def test_label_chunk_widths(rows, longest):
    """Columns on either side of the sizes where a chunk of labels gets wider,
    in segments that end inside chunks; rows past a window as well."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(rows + longest)
    words = [None] + [rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in range(0, longest, 1 + longest // 12)]
    b = StringBlob()
    for lo, hi in ((0, 123_457), (123_457, rows)):
        b.add(A.DICTIONARY, _label_segment(words, rng.integers(0, len(words), hi - lo)), lo, hi - lo)
    table = np.array(b.table, np.int64)
    o_offs, o_chars = oracle_string_runs(b.blob, table, rows)
    for skew in (0, 3):
        d = torch.zeros(b.blob.size + skew + 64, dtype=torch.uint8, device="cuda")
        d[skew:skew + b.blob.size] = torch.from_numpy(b.blob)
        offs, chars = _decode(duckdb_segments(table, d.data_ptr() + skew), rows, o_chars.size, A.LAUNCH_BATCHED, 4 * skew)
        np.testing.assert_array_equal(offs, o_offs)
        np.testing.assert_array_equal(chars, o_chars)


@pytest.mark.parametrize("rows", [1_500, 1_100_003, 2_200_001])
@pytest.mark.parametrize("entries,longest", [(2, 32), (255, 31), (256, 32), (257, 32), (256, 33), (9, 0), (40, 17)])
def test_labels_in_lds(entries, longest, rows):
    """Dictionaries on either side of what a workgroup keeps in LDS, output of
    less and of more than a window, entries with bad ends among them."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(entries * 64 + longest)
    lens = [longest if k == 1 else int(rng.integers(0, longest + 1)) for k in range(1, entries)]
    words = [None] + [rng.integers(0, 256, n, dtype=np.uint8).tobytes() for n in lens]
    seg = bytearray(_label_segment(words, rng.integers(0, entries, rows)))
    ibo = int.from_bytes(seg[8:12], "little")
    for k in (2, entries // 2):  # an end below its start, and one past dict_end
        if 1 < k < entries - 1:
            at = ibo + 4 * k
            seg[at:at + 4] = int(0 if k == 2 else 1 << 30).to_bytes(4, "little")
    b = StringBlob()
    b.add(A.DICTIONARY, bytes(seg), 0, rows)
    table = np.array(b.table, np.int64)
    o_offs, o_chars = oracle_string_runs(b.blob, table, rows)
    for skew in (0, 1):
        d = torch.zeros(b.blob.size + skew + 64, dtype=torch.uint8, device="cuda")
        d[skew:skew + b.blob.size] = torch.from_numpy(b.blob)
        print(f"[gpu] labels entries={entries} longest={longest} rows={rows} skew={skew}", flush=True)
        offs, chars = _decode(duckdb_segments(table, d.data_ptr() + skew), rows, o_chars.size, A.LAUNCH_BATCHED, 7 * skew)
        np.testing.assert_array_equal(offs, o_offs)
        np.testing.assert_array_equal(chars, o_chars)
