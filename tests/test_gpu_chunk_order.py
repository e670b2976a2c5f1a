"""String decodes whose first attempt, with chunks in workgroup order, gives up
(its share of a bound of 1024 is one wait): done again by ticket, they are right
in every mode, masks, totals and inline NULLs included; with a bound below that,
by ticket at once."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from oracle import oracle as O
from sirius_amd import lib as L
from tests.helpers import StringBlob, dictionary_string_segment, duckdb_segments, oracle_string_runs
from tests.test_gpu_dict_fsst import gpu_decode, upload

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _column(codec):
    rng = np.random.default_rng(5)
    n = 200_000
    if codec == "dictionary":
        words = [None] + [rng.integers(0, 256, k, dtype=np.uint8).tobytes() for k in range(1, 13)]
        b = StringBlob()
        b.add(A.DICTIONARY, dictionary_string_segment([words[k] for k in rng.integers(0, 13, n)]), 0, n)
        table = np.array(b.table, np.int64)
        offs, chars = oracle_string_runs(b.blob, table, n)
        d, base = upload(b.blob)
        return duckdb_segments(table, base), n, offs, chars, None, [d]
    chars, offs = E.gen_zipf_strings(77, n)
    if codec == "fsst":
        enc, valid = E.encode_fsst(chars, offs), None
        offs, chars = O.decode_strings(enc)
    else:
        enc = E.encode_dict_fsst(chars, offs, 1, valid=(np.arange(n) % 17 != 3).astype(np.uint8), seg_rows=9001)
        offs, chars, valid, _ = O.decode_strings_masked(enc, threads=8)
    d, base = upload(enc.blob)
    return [(getattr(A, codec.upper()), enc.segments(base))], n, offs, chars, valid, [d, enc]


@pytest.mark.parametrize("codec", ["fsst", "dictionary", "dict_fsst"])
@pytest.mark.parametrize("bound", [1 << 24, 1024, 1023])
def test_second_attempt(bound, codec):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib = L.load()
    runs, n, offs, chars, valid, keep = _column(codec)
    old = lib.sdr_tune_get(A.TUNE_FSST_SPIN_LIMIT)
    try:
        L.check(lib.sdr_tune_set(A.TUNE_FSST_SPIN_LIMIT, bound))
        for mode in (A.LAUNCH_BATCHED, A.LAUNCH_PER_SEGMENT, A.LAUNCH_PERSISTENT):
            print(f"[gpu] chunk order {codec} bound={bound} mode={mode}", flush=True)
            rc, col, g_offs, g_chars, g_valid = gpu_decode(runs, n, len(chars) + 64, mode)
            L.check(rc)
            assert col.chars_used == len(chars)
            np.testing.assert_array_equal(g_offs, offs)
            np.testing.assert_array_equal(g_chars[:len(chars)], chars)
            if valid is not None:
                np.testing.assert_array_equal(g_valid, valid)
                assert col.null_count == n - int(valid.sum())
    finally:
        L.check(lib.sdr_tune_set(A.TUNE_FSST_SPIN_LIMIT, old))
