"""The RLE slice knob: until it is set, and set to 0, launches choose by their size;
every other value that it takes, the reported default among them, is taken as it is."""
import sirius_amd._abi as A
from sirius_amd import lib as L


def test_zero_and_the_default_are_values():
    lib = L.load()
    key = A.TUNE_RLE_SLICE_ROWS
    before = [lib.sdr_tune_get_width(key, w) for w in A.TUNE_WIDTHS]
    try:
        for value in (16384, 0, 1024, 0):
            assert lib.sdr_tune_set(key, value) == A.SDR_OK
            assert [lib.sdr_tune_get_width(key, w) for w in A.TUNE_WIDTHS] == [value] * 4
        assert lib.sdr_tune_set_width(key, 8, 4096) == A.SDR_OK
        assert [lib.sdr_tune_get_width(key, w) for w in A.TUNE_WIDTHS] == [0, 0, 0, 4096]
        assert lib.sdr_tune_set(key, 64) == A.SDR_E_INVALID_ARG
        assert lib.sdr_tune_set(A.TUNE_BP_CHUNK_ROWS, 0) == A.SDR_E_INVALID_ARG
    finally:
        for w, v in zip(A.TUNE_WIDTHS, before):
            assert lib.sdr_tune_set_width(key, w, v if v != 16384 else 0) == A.SDR_OK
