"""Bit-packed groups staged in chunks of 512, 1024 and 2048 rows, fewer than a step
of a wavefront takes where values are a byte: every mode and width over whole
groups, a group cut short and one row, alone and beside other groups.  Bit for bit as
the oracle decodes them."""
import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from oracle import oracle as O
from sirius_amd import lib as L
from tests.helpers import fixed_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
MODES = [0, 4, 5]  # the encoder's choice, DELTA_FOR, FOR


def _modes(enc):
    """The modes of the first segment's groups (an entry for each, back to front before the metadata's end)."""
    g = enc.segs[0]
    seg = enc.blob[int(g["offset"]):]
    end, n = int(seg[:8].view(np.uint64)[0]), (int(g["row_count"]) + 2047) // 2048
    return {int(x) >> 24 for x in seg[end - 4 * n:end].view(np.uint32)}


@pytest.mark.parametrize("chunk", [512, 1024, 2048])
@pytest.mark.parametrize("rows", [1, 511, 2048, 4096 + 700, 10 * 2048])
def test_chunk_rows(chunk, rows):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib, s = L.load(), torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(rows)
    cols, keep, checks = [], [], []
    for t in (np.int8, np.int16, np.int32, np.int64):
        for mode in MODES:
            # rises slowly and starts again with each group of 2048, so that its deltas fit every type
            v = np.concatenate([np.cumsum(rng.random(2048) < 0.09) - 100 for _ in range(rows // 2048 + 1)])[:rows].astype(t)
            enc = E.encode_bitpacking(v, force_mode=mode)
            assert mode == 0 or rows < 2048 or _modes(enc) == {mode}
            d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
            out = torch.full((rows * v.itemsize,), 0xCC, dtype=torch.uint8, device="cuda")
            col, k = fixed_column([(A.BITPACKING, enc.segments(d.data_ptr()))], v.itemsize, rows, out.data_ptr())
            cols.append(col)
            keep += [d, k]
            checks.append((out, O.decode_encoded(enc)))
    saved = [lib.sdr_tune_get_width(A.TUNE_BP_CHUNK_ROWS, w) for w in A.TUNE_WIDTHS]
    try:
        L.check(lib.sdr_tune_set(A.TUNE_BP_CHUNK_ROWS, chunk))
        for group in ([c] for c in cols), [cols]:
            for part in group:
                print(f"[gpu] bp chunks {chunk} rows={rows} columns={len(part)}", flush=True)
                arr = (A.Column * len(part))(*part)
                L.check(lib.sdr_decode_table(arr, len(part), s))
            torch.cuda.synchronize()
            for out, want in checks:
                np.testing.assert_array_equal(out.cpu().numpy(), want)
                out.fill_(0xCC)
    finally:
        for w, x in zip(A.TUNE_WIDTHS, saved):
            L.check(lib.sdr_tune_set_width(A.TUNE_BP_CHUNK_ROWS, w, x))
