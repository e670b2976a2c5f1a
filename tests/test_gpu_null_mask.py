"""Null masks against a byte-by-byte overlay: pieces at the edges of a block's
8 KiB, segments out of order, overlapping and with gaps, any alignment of the
source and the mask, few pieces (kernel arguments) and many (pinned list),
through every entry that builds a mask."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _segments(name, rng):
    """(total rows, [(row_offset, row_count)...]): the segments in the order given."""
    if name.isdigit():
        n = int(name)
        return n, [(0, n)]
    if name == "gaps":
        return 300_011, [(8, 100), (4096, 65536), (200_000, 99_000)]
    if name == "reversed":
        return 245_760, [(122_880, 122_880), (0, 122_880)]
    if name == "overlaps":  # a later one wins where two share a byte
        return 90_001, [(0, 70_001), (64, 9), (69_992, 20_009), (800, 40_000), (1000, 64), (840, 8), (0, 16)]
    starts = np.arange(0, 1_000_000, 4096)  # many pieces
    return 1_000_003, [(int(s), int(min(4096, 1_000_003 - s))) for s in rng.permutation(starts)]


def _case(name, skew):
    rng = np.random.default_rng(len(name) + skew)
    total, segs = _segments(name, rng)
    want = np.full((total + 7) // 8, 0xFF, np.uint8)
    blob, table, at = [], [], 0
    for off, rows in segs:
        nb = (rows + 7) // 8
        b = rng.integers(0, 256, nb, dtype=np.uint8)
        want[off // 8:off // 8 + nb] = b
        pad = np.zeros((-(nb + skew) % 16) + skew, np.uint8)
        blob += [np.zeros(skew, np.uint8), b, pad]
        table.append((at + skew, nb, off, rows))
        at += nb + skew + pad.size
    d = torch.from_numpy(np.concatenate(blob)).cuda()
    vsegs = [A.Segment(d.data_ptr() + o, nb, off, rows, 0) for o, nb, off, rows in table]
    runs, keep = A.make_runs([(A.UNCOMPRESSED, vsegs)])
    nulls = total - int(np.unpackbits(want, bitorder="little")[:total].sum())
    return total, want, nulls, runs, [d, keep]


def _mask(total, skew):
    m = torch.full(((total + 7) // 8 + skew + 32,), 0xA5, dtype=torch.uint8, device="cuda")
    return m, m.data_ptr() + skew


def _same(m, skew, want):
    got = m.cpu().numpy()
    np.testing.assert_array_equal(got[skew:skew + want.size], want)
    assert (got[:skew] == 0xA5).all() and (got[skew + want.size:] == 0xA5).all()


NAMES = ["1", "7", "9", "65535", "65536", "65537", "524291", "gaps", "reversed", "overlaps", "many"]


@pytest.mark.parametrize("skew", [0, 3, 6])
@pytest.mark.parametrize("name", NAMES)
def test_masks(name, skew):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    total, want, nulls, runs, keep = _case(name, skew)
    lib, stream = L.load(), torch.cuda.current_stream().cuda_stream
    value = torch.tensor([7], dtype=torch.int32, device="cuda")
    data, keep2 = A.make_runs([(A.CONSTANT, [A.Segment(value.data_ptr(), 4, 0, total, 0)])])
    out = torch.empty(total, dtype=torch.int32, device="cuda")
    print(f"[gpu] null masks {name} rows={total} skew={skew}", flush=True)

    def column(d_mask):
        c = A.Column()
        c.type_size, c.total_rows, c.data, c.n_data, c.d_out = 4, total, data, 1, out.data_ptr()
        c.has_nulls, c.validity, c.n_validity, c.d_null_mask = 1, runs, 1, d_mask
        return c

    for mode in (A.LAUNCH_BATCHED, A.LAUNCH_PERSISTENT):
        masks = [_mask(total, s) for s in (0, skew)]
        cols = (A.Column * 2)(*[column(p) for _, p in masks])
        L.check(lib.sdr_decode_table_mode(cols, 2, stream, mode))
        for (m, _), s, c in zip(masks, (0, skew), cols):
            _same(m, s, want)
            assert c.null_count == nulls

    m, p = _mask(total, skew)
    cols = (A.Column * 1)(column(p))
    plan, count = C.c_void_p(), (C.c_int64 * 1)()
    L.check(lib.sdr_plan_create(cols, 1, A.LAUNCH_BATCHED, stream, C.byref(plan)))
    for _ in range(2):
        m.fill_(0xA5)
        L.check(lib.sdr_plan_launch(plan, stream))
        L.check(lib.sdr_plan_null_counts(plan, count, 1, stream))
        _same(m, skew, want)
        assert count[0] == nulls
    lib.sdr_plan_destroy(plan)

    chars, offs = np.frombuffer(b"x", np.uint8), np.minimum(np.arange(total + 1), 1).astype(np.uint64)
    enc = E.encode_fsst(chars, offs) if total <= 70_000 else None
    if enc is not None:  # the string entries, the allocation-free one among them
        blob = torch.from_numpy(enc.blob).cuda()
        sruns, keep3 = A.make_runs([(A.FSST, enc.segments(blob.data_ptr()))])
        d_offs = torch.empty(total + 1, dtype=torch.int32, device="cuda")
        d_chars = torch.empty(64, dtype=torch.uint8, device="cuda")
        for entry in (lib.sdr_decode_strings_column, lib.sdr_decode_strings_column_noalloc):
            m, p = _mask(total, skew)
            col = A.StringColumn()
            col.total_rows, col.data, col.n_data = total, sruns, 1
            col.d_offsets, col.d_chars, col.chars_capacity = d_offs.data_ptr(), d_chars.data_ptr(), 64
            col.has_nulls, col.validity, col.n_validity, col.d_null_mask = 1, runs, 1, p
            L.check(entry(C.byref(col), stream))
            _same(m, skew, want)
            assert col.null_count == nulls
