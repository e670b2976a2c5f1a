"""DICT_FSST's passes where their words and tiles are cut: entries of 0 to 60
bytes with escapes at every alignment, segments that share bytes of the null
mask, more rows than a tile.  Offsets, chars, mask and null count equal the
oracle's."""
import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from oracle import oracle as O
from sirius_amd import lib as L
from tests.test_gpu_dict_fsst import gpu_decode, upload

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dmode,source", [(0, "bytes"), (1, "bytes"), (1, "text"), (2, "bytes")])
@pytest.mark.parametrize("seg_rows", [1, 1001, 6000])
def test_cuts(seg_rows, dmode, source):
    rng = np.random.default_rng(seg_rows + dmode)
    n = 40 if seg_rows == 1 else 9_000
    lens = rng.integers(0, 61, n)
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    letters = np.arange(256, dtype=np.uint8) if source == "bytes" else np.frombuffer(b"the rain in spain ", np.uint8)
    chars = rng.choice(letters, int(offs[-1])) if source == "bytes" else np.resize(letters, int(offs[-1]))
    valid = None if dmode == 2 else (rng.random(n) > 0.2).astype(np.uint8)
    enc = E.encode_dict_fsst(chars.astype(np.uint8), offs, dmode, valid=valid, seg_rows=seg_rows)
    o_offs, o_chars, o_valid, o_nulls = O.decode_strings_masked(enc, threads=8)
    for skew in range(4):
        d, base = upload(enc.blob, skew=skew)
        print(f"[gpu] dict_fsst passes seg_rows={seg_rows} mode={dmode} skew={skew}", flush=True)
        rc, col, g_offs, g_chars, g_valid = gpu_decode([(A.DICT_FSST, enc.segments(base))], n, len(chars) + 64)
        L.check(rc)
        np.testing.assert_array_equal(g_offs, o_offs)
        assert col.chars_used == len(o_chars) and col.null_count == o_nulls
        np.testing.assert_array_equal(g_chars[:len(o_chars)], o_chars)
        np.testing.assert_array_equal(g_valid, o_valid)
