"""A batch's string columns are right once the stream has passed the launch: copies
enqueued behind it, before sdr_batch_finish or with none at all, hold the decoded
offsets and chars, also where waits for other chunks are as short as the bound on
them allows; a launch that nobody collects leaves nothing to the next."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import string_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _columns(rows_of):
    out = []
    for i, n in enumerate(rows_of):
        # the first chunk's rows are long, so the chunks after it wait for its length
        lens = np.where(np.arange(n) < 1024, 150, np.arange(n) % 3)
        offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
        chars = np.random.default_rng(31 + i).integers(97, 123, int(offs[-1]), dtype=np.uint8)
        enc = E.encode_fsst(chars, offs)
        offs = offs.astype(np.int32)
        d = torch.from_numpy(np.concatenate([enc.blob, np.zeros(64, np.uint8)])).cuda()
        o = torch.full((n + 1,), -7, dtype=torch.int32, device="cuda")
        c = torch.full((len(chars) + 32,), 0xCC, dtype=torch.uint8, device="cuda")
        col, k = string_column([(A.FSST, enc.segments(d.data_ptr()))], n, o.data_ptr(), c.data_ptr(), len(chars) + 32)
        out.append((col, offs, chars, o, c, [d, enc, k]))
    return out


def _add(lib, b, cols):
    L.check(lib.sdr_batch_clear(b))
    for col, *_ in cols:
        L.check(lib.sdr_batch_add_strings(b, C.byref(col)))


@pytest.mark.parametrize("graph", [0, 1], ids=["nograph", "graph"])
@pytest.mark.parametrize("bound", [1 << 24, 1024, 1023])
def test_copies_behind_the_launch(bound, graph):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib, s, b = L.load(), torch.cuda.current_stream().cuda_stream, C.c_void_p()
    old = lib.sdr_tune_get(A.TUNE_FSST_SPIN_LIMIT)
    L.check(lib.sdr_batch_create(C.byref(b)))
    try:
        L.check(lib.sdr_tune_set(A.TUNE_FSST_SPIN_LIMIT, bound))
        L.check(lib.sdr_batch_set_option(b, A.BATCH_USE_GRAPH, graph))
        first, second = _columns([300_000, 1, 90_000]), _columns([1024, 200_000, 1025])
        for finish in (True, False):
            for cols in (first, second):
                print(f"[gpu] batch stream order bound={bound} graph={graph} finish={finish}", flush=True)
                for *_, o, c, _ in cols:
                    o.fill_(-7)
                    c.fill_(0xCC)
                _add(lib, b, cols)
                L.check(lib.sdr_batch_launch(b, s))
                copies = [(o.clone(), c.clone()) for *_, o, c, _ in cols]  # on the launch's stream
                torch.cuda.synchronize()
                for (_, offs, chars, *_), (o, c) in zip(cols, copies):
                    np.testing.assert_array_equal(o.cpu().numpy(), offs)
                    np.testing.assert_array_equal(c.cpu().numpy()[:len(chars)], chars)
                    assert (c.cpu().numpy()[len(chars):] == 0xCC).all()
                if finish:
                    L.check(lib.sdr_batch_finish(b, s))
                    assert [col.chars_used for col, *_ in cols] == [len(chars) for _, _, chars, *_ in cols]
    finally:
        L.check(lib.sdr_tune_set(A.TUNE_FSST_SPIN_LIMIT, old))
        lib.sdr_batch_destroy(b)
