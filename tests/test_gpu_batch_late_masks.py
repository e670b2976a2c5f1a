"""A nullable column added to a batch between a launch and its finish is not that
launch's: finish leaves its null count alone, whatever earlier launches of the batch
had counted, and reports those of the columns launched."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
from sirius_amd import lib as L
from tests.helpers import fixed_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _column(rows, nulls):
    """A constant column; `nulls` (None: not nullable) rows of it are NULL."""
    value = torch.tensor([7], dtype=torch.int32, device="cuda")
    out = torch.zeros(rows, dtype=torch.int32, device="cuda")
    keep, validity, m = [value, out], None, None
    if nulls is not None:
        bits = np.ones(rows, np.uint8)
        bits[:nulls] = 0
        v = torch.from_numpy(np.packbits(bits, bitorder="little")).cuda()
        m = torch.zeros(v.numel(), dtype=torch.uint8, device="cuda")
        validity = [(A.UNCOMPRESSED, [A.Segment(v.data_ptr(), v.numel(), 0, rows, 0)])]
        keep += [v, m]
    col, k = fixed_column([(A.CONSTANT, [A.Segment(value.data_ptr(), 4, 0, rows, 0)])], 4, rows, out.data_ptr(), validity,
                          m.data_ptr() if m is not None else None)
    return col, keep + [k]


@pytest.mark.parametrize("launched", ["plain", "nullable"])
def test_added_before_finish(launched):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib, s, b = L.load(), torch.cuda.current_stream().cuda_stream, C.c_void_p()
    L.check(lib.sdr_batch_create(C.byref(b)))
    try:
        first, k0 = _column(5000, 4321)  # an earlier launch's masks
        L.check(lib.sdr_batch_add_table(b, C.byref(first), 1))
        L.check(lib.sdr_batch_launch(b, s))
        L.check(lib.sdr_batch_finish(b, s))
        assert first.null_count == 4321
        L.check(lib.sdr_batch_clear(b))
        col, k1 = _column(6000, 77 if launched == "nullable" else None)
        late, k2 = _column(7000, 5)
        print(f"[gpu] late masks, launched {launched}", flush=True)
        L.check(lib.sdr_batch_add_table(b, C.byref(col), 1))
        L.check(lib.sdr_batch_launch(b, s))
        L.check(lib.sdr_batch_add_table(b, C.byref(late), 1))
        L.check(lib.sdr_batch_finish(b, s))
        assert col.null_count == (77 if launched == "nullable" else 0)
        assert late.null_count == 0
        L.check(lib.sdr_batch_launch(b, s))
        L.check(lib.sdr_batch_finish(b, s))
        assert late.null_count == 5 and col.null_count == (77 if launched == "nullable" else 0)
    finally:
        lib.sdr_batch_destroy(b)
