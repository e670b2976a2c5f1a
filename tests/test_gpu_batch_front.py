"""A batch's first launches: from nothing but masks to string columns beside
fixed-width ones and masks, the same batch used again with another layout before
its last one is collected, columns of no rows among them.  Chars used, null
counts and outputs are those of each layout, with and without a graph."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import fixed_column, string_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _strings(rows, seed):
    rng = np.random.default_rng(seed)
    offs = np.concatenate([[0], np.cumsum(rng.integers(0, 20, rows))]).astype(np.uint64)
    chars = np.resize(np.frombuffer(b"batches of rows ", np.uint8), int(offs[-1]))
    keep = []
    if rows:
        enc = E.encode_fsst(chars, offs)
        d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
        runs, keep = [(A.FSST, enc.segments(d.data_ptr()))], [d, enc]
    else:
        runs = []
    o = torch.full((rows + 1,), -7, dtype=torch.int32, device="cuda")
    c = torch.zeros(chars.size + 32, dtype=torch.uint8, device="cuda")
    col, k = string_column(runs, rows, o.data_ptr(), c.data_ptr(), chars.size + 32)

    def check():
        assert col.chars_used == chars.size
        np.testing.assert_array_equal(o.cpu().numpy(), offs.astype(np.int32))
        np.testing.assert_array_equal(c.cpu().numpy()[:chars.size], chars)

    return "add_strings", col, check, [keep, k, o, c]


def _fixed(rows, seed, nullable):
    rng = np.random.default_rng(seed)
    v = rng.integers(0, 1000, rows).astype(np.int32)
    enc = E.encode_bitpacking(v)
    d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
    out = torch.zeros(rows, dtype=torch.int32, device="cuda")
    bits = rng.integers(0, 256, (rows + 7) // 8, dtype=np.uint8)
    vb = torch.from_numpy(bits).cuda()
    m = torch.zeros(bits.size, dtype=torch.uint8, device="cuda")
    col, k = fixed_column([(A.BITPACKING, enc.segments(d.data_ptr()))], 4, rows, out.data_ptr(),
                          [(A.UNCOMPRESSED, [A.Segment(vb.data_ptr(), bits.size, 0, rows, 0)])] if nullable else None,
                          m.data_ptr() if nullable else None)

    def check():
        np.testing.assert_array_equal(out.cpu().numpy(), v)
        if nullable:
            np.testing.assert_array_equal(m.cpu().numpy(), bits)
            assert col.null_count == rows - int(np.unpackbits(bits, bitorder="little")[:rows].sum())

    return "add_table", col, check, [d, out, vb, m, k]


LAYOUTS = {
    "masks": lambda: [_fixed(3_000, 1, True)],
    "strings": lambda: [_strings(0, 2), _strings(40_000, 3), _strings(1, 4), _strings(0, 5)],
    "all": lambda: [_strings(130_000, 6), _fixed(200_001, 7, True), _fixed(9, 8, False), _strings(0, 9), _strings(777, 10)],
    "empty": lambda: [_strings(0, 11)],
}


@pytest.mark.parametrize("graph", [1, 0], ids=["graph", "nograph"])
def test_layouts_in_turn(graph):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib, s, b = L.load(), torch.cuda.current_stream().cuda_stream, C.c_void_p()
    L.check(lib.sdr_batch_create(C.byref(b)))
    try:
        L.check(lib.sdr_batch_set_option(b, A.BATCH_USE_GRAPH, graph))
        for name in ("strings", "all", "masks", "all", "empty", "strings", "masks"):
            for finish in (False, True):  # the first of two launches is never collected
                parts = LAYOUTS[name if finish else "all"]()
                print(f"[gpu] batch front {name} graph={graph} finish={finish}", flush=True)
                L.check(lib.sdr_batch_clear(b))
                for kind, col, _, _ in parts:
                    if kind == "add_strings":
                        L.check(lib.sdr_batch_add_strings(b, C.byref(col)))
                    else:
                        L.check(lib.sdr_batch_add_table(b, C.byref(col), 1))
                L.check(lib.sdr_batch_launch(b, s))
                if finish:
                    L.check(lib.sdr_batch_finish(b, s))
                    for _, _, check, _ in parts:
                        check()
                else:
                    kept = parts  # its outputs stay alive until the next launch has finished
            del kept
    finally:
        lib.sdr_batch_destroy(b)
