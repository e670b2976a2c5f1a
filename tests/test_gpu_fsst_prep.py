"""The FSST segment pre-pass at its edges: length streams of one and of many
staged pieces, narrow and wide fields, and the number of ranges at which they
stop travelling with the launch.  Offsets and chars equal the oracle's."""
import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from tests.test_gpu_fsst_groups import _check

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("mode", [A.LAUNCH_BATCHED, A.LAUNCH_PERSISTENT], ids=["batched", "persistent"])
@pytest.mark.parametrize("rows,seg_rows,longest", [
    (130_000, 130_000, 3),   # one segment, two-bit lengths: more than one staged piece
    (70_000, 35_000, 700),   # seven-bit lengths: the last piece a remainder
    (26_201, 26_201, 200),   # five-bit lengths: the stream ends a byte past a piece's bytes
    (1_000, 10, 30),         # 100 ranges
    (1_001, 10, 30),         # 101 ranges
])
def test_staged_lengths(rows, seg_rows, longest, mode):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    rng = np.random.default_rng(rows)
    lens = rng.integers(0, 3 if longest < 10 else 16, rows)
    lens[::4_001] = longest
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    chars = np.resize(np.frombuffer(b"row by row ", np.uint8), int(offs[-1]))
    enc = E.encode_fsst(chars, offs, rg_rows=seg_rows, block=1 << 22)
    assert len(enc.segs) == -(-rows // seg_rows)
    for skew in (0, 7):
        _check(enc, mode, skew)
