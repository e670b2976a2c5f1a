"""RLE where runs are cut: windows of 64 runs longer than a wave's rows, slices
of every size the launch chooses, counts that end inside and on a step of the
walk.  Equal to the rows that were encoded."""
import ctypes as C

import numpy as np
import pytest

import sirius_amd._abi as A
from sirius_amd import lib as L
from tests.helpers import fixed_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _segment(values, counts):
    """u64 offset of the counts, the values, the u16 counts."""
    head = np.array([8 + values.nbytes], "<u8")
    return np.concatenate([head.view(np.uint8), values.view(np.uint8), counts.astype("<u2").view(np.uint8)])


@pytest.mark.parametrize("dtype", ["u1", "u2", "u4", "u8"])
@pytest.mark.parametrize("n_segs,entries,longest", [
    (1, 1, 65_535), (1, 128, 900), (3, 129, 400), (10, 600, 400), (1, 511, 64), (1, 513, 66), (40, 700, 130),
    (2, 8_192, 14), (2, 8_193, 15),
])
def test_long_runs(n_segs, entries, longest, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(entries + longest)
    blobs, want, segs, at, row = [], [], [], 0, 0
    for _ in range(n_segs):
        counts = rng.integers(max(1, longest // 2), longest + 1, entries)
        values = rng.integers(0, 256, (entries, int(dtype[1])), dtype=np.uint8).view("<" + dtype)[:, 0].copy()
        b = _segment(values, counts)
        want.append(np.repeat(values, counts))
        segs.append((at, b.size, row, int(counts.sum())))
        blobs.append(np.concatenate([b, np.zeros(-b.size % 4 + 3, np.uint8)]))  # odd addresses follow
        at += blobs[-1].size
        row += int(counts.sum())
    blob, want = np.concatenate(blobs), np.concatenate(want)
    d = torch.from_numpy(np.concatenate([blob, np.zeros(64, np.uint8)])).cuda()
    out = torch.zeros(want.nbytes + 64, dtype=torch.uint8, device="cuda")
    out.fill_(0xCC)
    col, keep = fixed_column([(A.RLE, [A.Segment(d.data_ptr() + o, n, r, c, 0) for o, n, r, c in segs])],
                             int(dtype[1]), row, out.data_ptr())
    L.check(L.load().sdr_decode_table(C.byref(col), 1, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:want.nbytes].view("<" + dtype), want)
    assert (got[want.nbytes:] == 0xCC).all()


@pytest.mark.parametrize("n_segs,rows", [(7, 16_000), (8, 16_384), (9, 16_385), (63, 100), (64, 2_048), (65, 2_048),
                                         (32, 4_096), (43, 4_097), (129, 100)])
def test_launch_edges(n_segs, rows):
    """Launches of one slice less, as many and one more than whole turns of 64."""
    test_long_runs(n_segs, rows // 10, 10, "u4")
