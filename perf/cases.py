"""Decode calls as programs make them, for timing on one MI355X.

Every case decodes DuckDB-format segments that are resident in device memory
into flat device columns, through the C ABI (include/sdr/decode.h):

  table    sdr_decode_table: fixed-width columns of one table, with or
           without NULLs (validity segments, one per row group)
  strings  sdr_decode_strings_column: one VARCHAR column of one string codec
  batch    sdr_batch_*: the columns of many requests in one launch, as the
           decode server collects them

Columns come in the shapes that scans meet: 122,880-row row groups cut into
segments of at most one 256 KiB block, a partly filled last row group, and
the value distributions of keys, quantities, dates, prices, flags, names and
labels.  The encoded rows of a large column are a base of whole row groups,
laid out again at addresses of their own until the column is full.
"""
import ctypes as C
import math

import numpy as np
import torch

import sirius_amd._abi as A
import sirius_amd.encode as E
from sirius_amd import lib as L

RG = E.ROW_GROUP_ROWS  # 122,880 rows

# kind -> (numpy type of a value, compressed bytes per row, base row groups).
# The compressed bytes are what these distributions encode to.
FIXED = {
    "bp_flag": ("int8", 0.26, 32),     # a flag of four values
    "bp_small": ("int16", 1.13, 32),   # a line number or a small code
    "bp_qty": ("int32", 0.76, 32),     # quantities 1..50
    "bp_date": ("int32", 0.51, 32),    # dates over seven years, sorted by group
    "bp_key": ("int64", 0.39, 32),     # an ascending key with small steps
    "bp_price": ("int64", 3.01, 32),   # decimal(15,2) prices
    "rle_key": ("int64", 0.62, 32),    # keys in runs of 16 on average
    "rle_day": ("int32", 0.03, 32),    # a clustered date, runs of 200
    "alp_price": ("float64", 3.12, 32),  # two decimals, 1% of full precision
    "alp_rate": ("float32", 1.65, 32),   # float rates of two decimals
    "alprd_unit": ("float64", 6.9, 16),  # doubles without a decimal form
    "unc_hash": ("int64", 8.0, 16),    # hashes, stored uncompressed
    "const_year": ("int32", 0.0001, 32),  # a constant per row group
}
# codec -> (compressed bytes per row, decoded chars per row, base row groups, longest text)
STRINGS = {
    "fsst": (12.9, 27.0, 4, 44),      # comments: words of a 2000-word vocabulary, 10-44 bytes
    "dictionary": (0.50, 5.9, 4, 17),  # labels: a handful of names
    "plain": (31.0, 27.0, 2, 44),     # text that DuckDB left uncompressed
    "dict_fsst": (2.3, 27.0, 1, 44),  # repeated texts under a compressed dictionary
}
# what the decode server's stream asks for, and its shares
MIX = (("bp_qty", 0.40), ("rle_key", 0.20), ("alp_price", 0.25), ("fsst", 0.15))
LARGEST = 1.3e9  # bytes of the largest listed case


def listed():
    return [
        # a point query's column: one row group of one column, where the call's own cost counts
        {"name": "row_group_date", "what": "table", "cols": "bp_date", "rows": RG, "nulls": 0.0},
        # one scan split: ten row groups of a table's usual columns, some of them NULL
        {"name": "split_with_nulls", "what": "table", "cols": "bp_key bp_price bp_date rle_day alp_price",
         "rows": 10 * RG, "nulls": 0.03},
        # a full scan of integer and date columns (the integer/date workload of the benchmark)
        {"name": "int_date_scan", "what": "table", "cols": "rle_key bp_qty bp_date", "rows": 64 << 20, "nulls": 0.0},
        # a scan of measures: doubles with and without a decimal form (the benchmark's ALP workload)
        {"name": "double_scan", "what": "table", "cols": "alp_price alprd_unit", "rows": 16 << 20, "nulls": 0.0},
        # the other widths and codecs at a ragged row count
        {"name": "all_widths", "what": "table", "cols": "bp_flag bp_small rle_day alp_rate unc_hash const_year",
         "rows": 10_000_019, "nulls": 0.0},
        # a nullable measure over a whole table: values, mask and null count
        {"name": "nullable_scan", "what": "table", "cols": "bp_price", "rows": 32 << 20, "nulls": 0.1},
        # a comment column over a whole table (the benchmark's FSST workload)
        {"name": "comments_scan", "what": "strings", "codec": "fsst", "rows": 16 << 20, "nulls": 0.0},
        # the same for one row group, as a filtered scan reads it
        {"name": "comments_row_group", "what": "strings", "codec": "fsst", "rows": RG, "nulls": 0.0},
        # a label column (ship mode, status) with some NULLs
        {"name": "labels_scan", "what": "strings", "codec": "dictionary", "rows": 8 << 20, "nulls": 0.02},
        # text that was not worth compressing, at a ragged row count
        {"name": "plain_text", "what": "strings", "codec": "plain", "rows": 2_000_003, "nulls": 0.0},
        # repeated texts under a compressed dictionary
        {"name": "dict_fsst_text", "what": "strings", "codec": "dict_fsst", "rows": 2_000_003, "nulls": 0.0},
        # what one launch of the decode server holds: 128 requests of mixed codecs and sizes
        {"name": "served_batch", "what": "batch", "requests": 128, "min_rows": 2048, "max_rows": 4 << 20},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    what = rng.choice(("table", "table", "table", "strings", "strings", "batch"))
    if what == "table":
        cols = [rng.choice(sorted(FIXED)) for _ in range(rng.randint(1, 6))]
        per_row = sum(np.dtype(FIXED[c][0]).itemsize + FIXED[c][1] for c in cols)
        return {"what": what, "cols": " ".join(cols), "rows": _log_int(rng, 2048, min(64 << 20, int(LARGEST / per_row))),
                "nulls": rng.choice((0.0, 0.0, 0.01, 0.2))}
    if what == "strings":
        codec = rng.choice(("fsst", "fsst", "dictionary", "plain", "dict_fsst"))
        most = {"fsst": 16 << 20, "dictionary": 16 << 20, "plain": 4 << 20, "dict_fsst": 4 << 20}[codec]
        return {"what": what, "codec": codec, "rows": _log_int(rng, 2048, most),
                "nulls": 0.0 if codec == "dict_fsst" else rng.choice((0.0, 0.0, 0.05))}
    return {"what": what, "requests": _log_int(rng, 8, 128), "min_rows": 2048, "max_rows": _log_int(rng, 65536, 4 << 20)}


# ---- values and their segments ------------------------------------------------


def _values(kind, rng, n):
    """Host values of a fixed-width column."""
    if kind == "bp_flag":
        return rng.integers(0, 4, n, dtype=np.int8)
    if kind == "bp_small":
        return rng.integers(1, 500, n, dtype=np.int16)
    if kind == "bp_qty":
        return rng.integers(1, 51, n, dtype=np.int32)
    if kind == "bp_date":
        v = rng.integers(8035, 8035 + 7 * 365, n, dtype=np.int32)
        whole = n // 2048 * 2048
        v[:whole] = np.sort(v[:whole].reshape(-1, 2048), axis=1).reshape(-1)
        return v
    if kind == "bp_key":
        return np.cumsum(rng.integers(1, 9, n, dtype=np.int64))
    if kind == "bp_price":
        return rng.integers(90_000, 10_500_000, n, dtype=np.int64)
    if kind == "rle_key":
        runs = n // 16 + 64
        v = np.repeat(rng.integers(0, 1 << 40, runs, dtype=np.int64), rng.geometric(1 / 16, runs))
        return np.resize(v, n)
    if kind == "rle_day":
        runs = n // 200 + 64
        v = np.repeat(rng.integers(8035, 10590, runs, dtype=np.int32), rng.geometric(1 / 200, runs))
        return np.resize(v, n)
    if kind == "alp_price":
        v = rng.integers(90_000, 10_500_000, n).astype(np.float64) / 100.0
        odd = rng.integers(0, n, n // 100)
        v[odd] = rng.random(odd.size) * 1e6
        return v
    if kind == "alp_rate":
        return (rng.integers(0, 2000, n).astype(np.float32) / np.float32(100.0)).astype(np.float32)
    if kind == "alprd_unit":
        return rng.random(n)
    if kind == "unc_hash":
        return rng.integers(-(1 << 62), 1 << 62, n, dtype=np.int64)
    groups = -(-n // RG)
    return np.repeat(rng.integers(1992, 1999, groups, dtype=np.int32), RG)[:n]


def _constant_segments(values):
    """One 16-byte slot per row group, holding its value."""
    groups = -(-values.size // RG)
    blob = np.zeros((groups, 16), np.uint8)
    blob[:, :4] = values[::RG].astype("<i4").view(np.uint8).reshape(groups, 4)
    rows = np.arange(groups) * RG
    segs = np.zeros(groups, E.SEG_DTYPE)
    segs["offset"], segs["bytes_size"] = np.arange(groups) * 16, 4
    segs["row_offset"], segs["row_count"] = rows, np.minimum(RG, values.size - rows)
    return blob.reshape(-1), segs


def _encode_fixed(kind, values):
    if kind == "const_year":
        return (A.CONSTANT,) + _constant_segments(values)
    enc = {"bp": E.encode_bitpacking, "rl": E.encode_rle, "un": E.encode_uncompressed}.get(kind[:2])
    if enc is None:
        enc = E.encode_alprd if kind.startswith("alprd") else E.encode_alp
    e = enc(values)
    return e.codec, e.blob, e.segs


def _text(seed, n):
    """n texts of 10-44 bytes: words of a vocabulary, Zipf-distributed."""
    return E.gen_zipf_strings(seed, n)


def _reversed_bytes(chars, lo, hi):
    """The texts [lo[i], hi[i]) of `chars`, last text first, in one array."""
    lo, length = lo[::-1].astype(np.int64), (hi - lo)[::-1].astype(np.int64)
    start = np.cumsum(length) - length
    return chars[np.arange(length.sum()) + np.repeat(lo - start, length)]


def _join(parts):
    """Segments (bytes, rows, longest text) -> blob, segment table."""
    segs = np.zeros(len(parts), E.SEG_DTYPE)
    at = row = 0
    chunks = []
    for i, (b, rows, longest) in enumerate(parts):
        segs[i] = (at, b.size, row, rows, longest)
        pad = np.zeros(-b.size % 16, np.uint8)
        chunks += [b, pad]
        at += b.size + pad.size
        row += rows
    return np.concatenate(chunks), segs


def _plain_segments(chars, offs):
    """UNCOMPRESSED text: {dict_size, dict_end}, an int32 end per row, then the
    bytes, last row first; as many rows as fit a block."""
    n, parts, r = offs.size - 1, [], 0
    while r < n:
        last = int(np.searchsorted(offs + 4 * np.arange(n + 1, dtype=np.uint64), offs[r] + np.uint64(4 * r + E.BLOCK_SIZE - 64)))
        last = max(r + 1, min(last - 1, n, r // RG * RG + RG))
        ends = (offs[r + 1:last + 1] - offs[r]).astype("<i4")
        size = 8 + 4 * ends.size + int(ends[-1])
        head = np.array([int(ends[-1]), size], "<u4")
        body = _reversed_bytes(chars, offs[r:last], offs[r + 1:last + 1])
        parts.append((np.concatenate([head.view(np.uint8), ends.view(np.uint8), body]), last - r,
                      int((offs[r + 1:last + 1] - offs[r:last]).max())))
        r = last
    return _join(parts)


LABELS = (b"REG AIR", b"AIR", b"RAIL", b"SHIP", b"TRUCK", b"MAIL", b"FOB", b"DELIVER IN PERSON")


def _label_segments(rng, n):
    """DICTIONARY labels: 20-byte header, bit-packed selections (0 is NULL), an
    index buffer of cumulative ends, the entries back to front."""
    ends = np.concatenate([[0, 0], np.cumsum([len(x) for x in LABELS])])[1:].astype("<u4")
    body = np.frombuffer(b"".join(LABELS[::-1]), np.uint8)
    width, parts = 4, []
    for r in range(0, n, RG):
        rows = min(RG, n - r)
        pick = rng.integers(1, len(LABELS) + 1, rows, dtype=np.uint8)
        pick = np.concatenate([pick, np.zeros(-rows % 32, np.uint8)])
        sel = (pick[0::2] | (pick[1::2] << 4)).astype(np.uint8)
        ibo = 20 + sel.size
        end = ibo + 4 * ends.size + body.size
        head = np.array([body.size, end, ibo, ends.size, width], "<u4")
        parts.append((np.concatenate([head.view(np.uint8), sel, ends.view(np.uint8), body]), rows,
                      max(len(x) for x in LABELS)))
    return _join(parts)


def _repeated(rng, seed, n):
    """n texts out of 2,000 different ones."""
    chars, offs = _text(seed, 2000)
    pick = rng.integers(0, 2000, n)
    length = (offs[1:] - offs[:-1])[pick].astype(np.int64)
    o = np.concatenate([[0], np.cumsum(length)])
    at = np.arange(o[-1]) + np.repeat(offs[:-1][pick].astype(np.int64) - o[:-1], length)
    return chars[at], o.astype(np.uint64)


def _encode_strings(codec, rng, seed, n):
    if codec == "fsst":
        e = E.encode_fsst(*_text(seed, n))
        return A.FSST, e.blob, e.segs
    if codec == "dictionary":
        return (A.DICTIONARY,) + _label_segments(rng, n)
    if codec == "plain":
        return (A.UNCOMPRESSED,) + _plain_segments(*_text(seed, n))
    e = E.encode_dict_fsst(*_repeated(rng, seed, n), mode=1, seg_rows=32768)
    return A.DICT_FSST, e.blob, e.segs


def _resident(blob, segs, base_rows, copies, tail):
    """`copies` of the base's blob and then the tail's in device memory, with
    one segment table over all of them."""
    d = torch.from_numpy(np.concatenate([blob, np.zeros(-blob.size % 16, np.uint8)])).cuda()
    size, tables = d.numel(), []
    for i in range(copies):
        t = segs.copy()
        t["offset"] += np.uint64(i * size)
        t["row_offset"] += np.uint32(i * base_rows)
        tables.append(t)
    d = d.repeat(copies)
    if tail is not None:
        t = tail[1].copy()
        t["offset"] += np.uint64(copies * size)
        t["row_offset"] += np.uint32(copies * base_rows)
        tables.append(t)
        d = torch.cat([d, torch.from_numpy(tail[0]).cuda()])
    table = np.concatenate(tables)
    table["offset"] += np.uint64(d.data_ptr())  # the descriptor's d_bytes
    return d, table


def _runs(codec, table):
    """An sdr_run over a segment table (whose records are sdr_segments)."""
    segs = (A.Segment * len(table)).from_buffer_copy(table.tobytes())
    run = (A.Run * 1)()
    run[0].codec, run[0].n_segments, run[0].segments = codec, len(table), C.cast(segs, C.POINTER(A.Segment))
    return run, [segs, run]


def _split(rows, base_groups):
    """(rows of the base, how often it is laid out, rows of the tail)."""
    base = min(base_groups, max(1, rows // RG)) * RG
    if rows < RG:
        return rows, 1, 0
    return base, rows // base, rows % base


def _fixed_column(kind, seed, rows):
    base, copies, rest = _split(rows, FIXED[kind][2])
    codec, blob, segs = _encode_fixed(kind, _values(kind, np.random.default_rng([seed, 1]), base))
    tail = _encode_fixed(kind, _values(kind, np.random.default_rng([seed, 2]), rest))[1:] if rest else None
    return (codec,) + _resident(blob, segs, base, copies, tail)


def _string_column(codec, seed, rows):
    base, copies, rest = _split(rows, STRINGS[codec][2])
    cid, blob, segs = _encode_strings(codec, np.random.default_rng([seed, 1]), 2 * seed + 1, base)
    tail = _encode_strings(codec, np.random.default_rng([seed, 2]), 2 * seed + 2, rest)[1:] if rest else None
    return (cid,) + _resident(blob, segs, base, copies, tail)


def _validity(seed, rows, nulls):
    """Validity bits in device memory, one segment per row group."""
    base = min(rows, 16 * RG)
    bits = np.packbits(np.random.default_rng([seed, 3]).random(base) >= nulls, bitorder="little")
    bits = np.resize(bits, -(-rows // 8) + 16)
    d = torch.from_numpy(bits).cuda()
    start = np.arange(0, rows, RG)
    table = np.zeros(start.size, E.SEG_DTYPE)
    table["offset"] = d.data_ptr() + start // 8
    table["row_offset"], table["row_count"] = start, np.minimum(RG, rows - start)
    table["bytes_size"] = (table["row_count"] + 7) // 8
    run, keep = _runs(A.UNCOMPRESSED, table)
    return run, torch.empty(-(-rows // 8), dtype=torch.uint8, device="cuda"), keep + [d]


# ---- prepare, run --------------------------------------------------------------


def _torch_type(kind):
    return getattr(torch, FIXED[kind][0])


def _prepare_table(case, seed):
    kinds, rows = case["cols"].split(), case["rows"]
    cols, outs, masks, keep = (A.Column * len(kinds))(), [], [], []
    for i, kind in enumerate(kinds):
        codec, d, table = _fixed_column(kind, 1000 * seed + i, rows)
        run, k = _runs(codec, table)
        out = torch.empty(rows, dtype=_torch_type(kind), device="cuda")
        keep += [d, k]
        outs.append(out)
        c = cols[i]
        c.type_size, c.total_rows, c.data, c.n_data, c.d_out = out.element_size(), rows, run, 1, out.data_ptr()
        if case["nulls"]:
            vrun, mask, k = _validity(1000 * seed + i, rows, case["nulls"])
            keep.append(k)
            masks.append(mask)
            c.has_nulls, c.validity, c.n_validity, c.d_null_mask = 1, vrun, 1, mask.data_ptr()
    return {"what": "table", "lib": L.load(), "cols": cols, "outs": outs, "masks": masks, "keep": keep}


def _prepare_strings(case, seed):
    rows = case["rows"]
    codec, d, table = _string_column(case["codec"], 1000 * seed, rows)
    run, keep = _runs(codec, table)
    cap = rows * STRINGS[case["codec"]][3]
    offs = torch.empty(rows + 1, dtype=torch.int32, device="cuda")
    chars = torch.zeros(cap, dtype=torch.uint8, device="cuda")
    col = A.StringColumn()
    col.total_rows, col.data, col.n_data = rows, run, 1
    col.d_offsets, col.d_chars, col.chars_capacity = offs.data_ptr(), chars.data_ptr(), cap
    mask = None
    if case["nulls"]:
        vrun, mask, k = _validity(1000 * seed, rows, case["nulls"])
        keep.append(k)
        col.has_nulls, col.validity, col.n_validity, col.d_null_mask = 1, vrun, 1, mask.data_ptr()
    elif case["codec"] == "dict_fsst":  # its NULL slot needs a mask buffer
        mask = torch.empty(-(-rows // 8), dtype=torch.uint8, device="cuda")
        col.d_null_mask = mask.data_ptr()
    return {"what": "strings", "lib": L.load(), "col": col, "offs": offs, "chars": chars, "mask": mask, "keep": [d, keep]}


def _prepare_batch(case, seed):
    """Requests of log-uniform sizes: consecutive row groups of a resident
    source column from a random start, then a partial one from a ladder.
    The stream of sizes and codecs belongs to the case, the rows to the seed."""
    rng = np.random.default_rng([case["requests"], case["max_rows"]])
    kinds = rng.choice(len(MIX), case["requests"], p=[m[1] for m in MIX])
    sizes = np.exp(rng.uniform(math.log(case["min_rows"]), math.log(case["max_rows"]), case["requests"])).astype(np.int64)
    ladder = np.unique(np.geomspace(2048, RG - 1, 8).astype(np.int64))
    lib, keep, requests, total = L.load(), [], [], {}
    for ki, (kind, _) in enumerate(MIX):
        mine = sizes[kinds == ki]
        groups = max(1, -(-int(mine.max()) // RG)) if mine.size else 1
        column = _string_column if kind == "fsst" else _fixed_column
        codec, d, source = column(kind, 1000 * seed + 16 * ki, groups * RG)
        keep.append(d)
        firsts = np.flatnonzero(source["row_offset"] % RG == 0)  # first segment of each row group
        tails = []
        for ti, n in enumerate(ladder):
            _, d, t = column(kind, 1000 * seed + 16 * ki + 1 + ti, int(n))
            keep.append(d)
            tails.append(t)
        for n in mine:
            g = min(int(n) // RG, groups)
            parts, rows = [], 0
            if g:
                f = int(rng.integers(0, groups - g + 1))
                end = firsts[f + g] if f + g < len(firsts) else len(source)
                part = source[firsts[f]:end].copy()
                part["row_offset"] -= part["row_offset"][0]
                parts.append(part)
                rows = g * RG
            i = int(np.searchsorted(ladder, int(n) - rows, side="right")) - 1
            if i >= 0 or not parts:
                part = tails[max(i, 0)].copy()
                part["row_offset"] += np.uint32(rows)
                rows += int(ladder[max(i, 0)])
                parts.append(part)
            requests.append((kind, codec, np.concatenate(parts), rows))
            total[kind] = total.get(kind, 0) + rows
    rng.shuffle(requests)
    outs = {k: torch.zeros(n + (case["requests"] if k == "fsst" else 0) + 64 * case["requests"],
                           dtype=torch.int32 if k == "fsst" else _torch_type(k), device="cuda") for k, n in total.items()}
    longest = STRINGS["fsst"][3]
    chars = torch.zeros(max(1, sum(longest * rows + 16 for k, _, _, rows in requests if k == "fsst")), dtype=torch.uint8,
                        device="cuda")
    at, chars_at, tables, strings = {k: 0 for k in outs}, 0, [], []
    for kind, codec, table, rows in requests:
        run, k = _runs(codec, table)
        keep.append(k)
        out, o = outs[kind], at[kind]
        if kind == "fsst":
            cap = longest * rows
            col = A.StringColumn()
            col.total_rows, col.data, col.n_data = rows, run, 1
            col.d_offsets, col.d_chars, col.chars_capacity = out.data_ptr() + 4 * o, chars.data_ptr() + chars_at, cap
            chars_at += -(-cap // 16) * 16
            strings.append(col)
            rows += 1
        else:
            col = A.Column()
            col.type_size, col.total_rows, col.data, col.n_data = out.element_size(), rows, run, 1
            col.d_out = out.data_ptr() + out.element_size() * o
            tables.append(col)
        at[kind] = o + -(-rows // 16) * 16
    batch = C.c_void_p()
    L.check(lib.sdr_batch_create(C.byref(batch)))
    return {"what": "batch", "lib": lib, "batch": batch, "tables": tables, "strings": strings, "outs": outs,
            "chars": chars, "keep": keep}


def prepare(case, seed):
    return {"table": _prepare_table, "strings": _prepare_strings, "batch": _prepare_batch}[case["what"]](case, seed)


def run(state):
    lib, stream = state["lib"], torch.cuda.current_stream().cuda_stream
    if state["what"] == "table":
        cols = state["cols"]
        L.check(lib.sdr_decode_table(cols, len(cols), stream))
        return [state["outs"], state["masks"], [c.null_count for c in cols]]
    if state["what"] == "strings":
        col = state["col"]
        L.check(lib.sdr_decode_strings_column(C.byref(col), stream))
        return [state["offs"], state["chars"], col.chars_used, state["mask"], col.null_count]
    b = state["batch"]
    L.check(lib.sdr_batch_clear(b))
    for col in state["tables"]:
        L.check(lib.sdr_batch_add_table(b, col, 1))
    for col in state["strings"]:
        L.check(lib.sdr_batch_add_strings(b, col))
    L.check(lib.sdr_batch_launch(b, stream))
    L.check(lib.sdr_batch_finish(b, stream))
    return [state["outs"], state["chars"], [int(sum(col.chars_used for col in state["strings"]))]]


# ---- what a pass cannot do without ---------------------------------------------


def work(case):
    if case["what"] == "table":
        per = sum(np.dtype(FIXED[k][0]).itemsize + FIXED[k][1] + (0.25 if case["nulls"] else 0.0)
                  for k in case["cols"].split())
        return {"bytes": case["rows"] * per, "flops": 0}
    if case["what"] == "strings":
        comp, chars = STRINGS[case["codec"]][:2]
        return {"bytes": case["rows"] * (comp + chars + 4 + (0.25 if case["nulls"] else 0.0)), "flops": 0}
    lo, hi = case["min_rows"], case["max_rows"]
    mean = (hi - lo) / math.log(hi / lo)  # of a log-uniform size
    per = sum(share * (np.dtype(FIXED[k][0]).itemsize + FIXED[k][1] if k in FIXED else sum(STRINGS[k][:2]) + 4)
              for k, share in MIX)
    return {"bytes": case["requests"] * mean * per, "flops": 0}


def exact(case, seed):
    """The doubles and floats as they were before encoding (ALP and ALP-RD are
    lossless); the other outputs are whole numbers and bytes."""
    if case["what"] != "table":
        return None
    outs = []
    for i, kind in enumerate(case["cols"].split()):
        if not FIXED[kind][0].startswith("float"):
            outs.append(None)
            continue
        base, copies, rest = _split(case["rows"], FIXED[kind][2])
        v = np.tile(_values(kind, np.random.default_rng([1000 * seed + i, 1]), base), copies)
        if rest:
            v = np.concatenate([v, _values(kind, np.random.default_rng([1000 * seed + i, 2]), rest)])
        outs.append(v.astype(np.float64))
    if all(o is None for o in outs):
        return None
    return [outs, [None] * (len(outs) if case["nulls"] else 0), [None] * len(outs)]
