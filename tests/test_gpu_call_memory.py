"""The memory that calls take from each other: a call that waits for its own result
does not wait for other streams' queued work first, and of the device memory of many
string calls at once little is kept after them."""
import ctypes as C
import threading

import numpy as np
import pytest

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L
from tests.helpers import dictionary_string_segment, fixed_column, string_column

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _sleep(ms):
    """Enqueue a kernel of about `ms` on the current stream."""
    t = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t[0].record()
    torch.cuda._sleep(1_000_000)
    t[1].record()
    torch.cuda.synchronize()
    cycles = int(1_000_000 * ms / max(t[0].elapsed_time(t[1]), 1e-3))
    return lambda: torch.cuda._sleep(cycles)


def _table():
    """A column of 300 constant segments: more descriptors than travel in kernel arguments."""
    v = torch.arange(300, dtype=torch.int32, device="cuda")
    out = torch.zeros(300 * 64, dtype=torch.int32, device="cuda")
    segs = [A.Segment(v.data_ptr() + 4 * i, 4, 64 * i, 64, 0) for i in range(300)]
    col, k = fixed_column([(A.CONSTANT, segs)], 4, 300 * 64, out.data_ptr())
    return (A.Column * 1)(col), out, [v, k]


def _strings(n, segs):
    """A DICTIONARY column of `segs` segments of n rows each, one word."""
    blob = np.frombuffer(dictionary_string_segment([b"word"] * n), np.uint8)
    d = torch.from_numpy(np.concatenate([blob, np.zeros(64, np.uint8)])).cuda()
    o = torch.zeros(n * segs + 1, dtype=torch.int32, device="cuda")
    c = torch.zeros(4 * n * segs + 32, dtype=torch.uint8, device="cuda")
    col, k = string_column([(A.DICTIONARY, [A.Segment(d.data_ptr(), blob.size, n * i, n, 0) for i in range(segs)])],
                           n * segs, o.data_ptr(), c.data_ptr(), 4 * n * segs + 32)
    return col, o, c, [d, k]


def test_waits_for_its_own_stream_alone():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib = L.load()
    busy, mine = torch.cuda.Stream(), torch.cuda.Stream()
    sleep = _sleep(400)
    tables = [_table() for _ in range(32)]
    col, o, c, keep = _strings(100, 3)
    bits = torch.zeros(8, dtype=torch.uint8, device="cuda")
    mask, value, out = torch.zeros_like(bits), torch.ones(1, dtype=torch.int32, device="cuda"), torch.zeros(64, device="cuda")
    nullable, k = fixed_column([(A.CONSTANT, [A.Segment(value.data_ptr(), 4, 0, 64, 0)])], 4, 64, out.data_ptr(),
                               [(A.UNCOMPRESSED, [A.Segment(bits.data_ptr(), 8, 0, 64, 0)])], mask.data_ptr())
    nullable = (A.Column * 1)(nullable)
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    with torch.cuda.stream(busy):
        sleep()
        for arr, _, _ in tables:
            L.check(lib.sdr_decode_table(arr, 1, busy.cuda_stream))
        done.record()
    print("[gpu] a string call and a nullable table beside 32 queued tables", flush=True)
    assert not done.query()
    L.check(lib.sdr_decode_strings_column(C.byref(col), mine.cuda_stream))
    L.check(lib.sdr_decode_table(nullable, 1, mine.cuda_stream))
    waited = done.query()
    torch.cuda.synchronize()
    assert not waited, "the calls waited for the other stream's work"
    assert col.chars_used == 1200 and nullable[0].null_count == 64
    want = np.repeat(np.arange(300, dtype=np.int32), 64)
    for _, out, _ in tables:
        np.testing.assert_array_equal(out.cpu().numpy(), want)


def _pool(attr):
    """An attribute of the device's default memory pool, in bytes."""
    hip, pool, v = C.CDLL("libamdhip64.so"), C.c_void_p(), C.c_uint64()
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert hip.hipMemPoolGetAttribute(pool, attr, C.byref(v)) == 0
    return v.value


def _held():
    """Device memory that is neither free nor the pool's to hand out again."""
    reserved, used = 5, 7
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free - (_pool(reserved) - _pool(used))


def test_little_is_kept():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib, threads = L.load(), 12
    sleep = _sleep(30)
    parts = [_strings(1, 8_000) for _ in range(threads)]  # 19 MB of descriptors, mostly symbol tables
    streams = [torch.cuda.Stream() for _ in range(threads)]
    L.check(lib.sdr_decode_strings_column(C.byref(_strings(1, 2)[0]), streams[0].cuda_stream))
    torch.cuda.synchronize()
    before, errors, start = _held(), [], threading.Barrier(threads)

    def work(i):
        torch.cuda.set_device(0)
        start.wait()
        with torch.cuda.stream(streams[i]):
            sleep()
        errors.append(lib.sdr_decode_strings_column(C.byref(parts[i][0]), streams[i].cuda_stream))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    print(f"[gpu] {threads} string calls at once", flush=True)
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert errors == [A.SDR_OK] * threads
    kept = _held() - before
    print(f"[gpu] kept {kept >> 20} MiB", flush=True)
    for col, o, c, _ in parts:
        assert col.chars_used == 32_000
        np.testing.assert_array_equal(o.cpu().numpy(), 4 * np.arange(8_001, dtype=np.int32))
        assert bytes(c.cpu().numpy()[:32_000]) == b"word" * 8_000
    assert kept <= (8 * 32 + 32) << 20  # at most 8 calls' memory, of 32 MiB at most, and slack
