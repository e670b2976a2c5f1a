// sdr_fsst.hpp — descriptors shared by the FSST kernels and their host drivers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/sdr/decode.h"

namespace sdr {

struct MaskUnit;

constexpr uint32_t FSST_CHUNK_ROWS = 1024;        // rows per workgroup
constexpr uint32_t WIDE_CHUNK_ROWS = 4096;        // ... at most, in columns of DICTIONARY segments
constexpr uint32_t FSST_GAP        = 0xFFFFFFFFu;  // chunk of rows no segment covers
constexpr uint32_t FSST_SPIN_LIMIT = 1u << 24;     // look-back wait bound (never reached)
// A chunk waits on the chunks before it, so these must be running or done.  A
// decode first takes each workgroup's number for its chunk's, the order in which
// workgroups are in fact started, and waits a 1024th of the bound, 1024 sleeps or
// about a millisecond at most; if that was not enough the decode is done again with chunks in the order of a ticket that
// workgroups draw as they start, which needs no assumption but costs each of
// them one of a queue of atomics on one word, 13 ns apart (16 Mi rows 293 us,
// without 274; 2 M rows of 27 chars 44 us, 35 us; a batch's strings 182 us, 168 us).
// A call that waits for its result before it returns looks at it and decodes again
// (with a bound below 1024, for tests, by ticket at once); behind a batch's chunks, whose
// outputs are to be complete in stream order, a kernel does (k_batch_again).
//
// It is not enough where the XCDs, each of which starts its share of a launch by
// itself, are full of workgroups that wait: of two string launches on two streams,
// one that came first on some XCDs and the other on the others, or beside a long
// kernel that holds some of them.  That costs the wait, and the decode twice.
constexpr uint32_t FSST_UNORDERED_SHARE = 1024;
constexpr uint32_t FSST_UNORDERED_MOST  = 1024;
__host__ __device__ inline uint32_t fsst_unordered_spins(uint32_t bound)
{
  return bound / FSST_UNORDERED_SHARE < FSST_UNORDERED_MOST ? bound / FSST_UNORDERED_SHARE : FSST_UNORDERED_MOST;
}
inline bool fsst_unordered(uint32_t spin_limit) { return spin_limit >= FSST_UNORDERED_SHARE; }

// A row range of a column: a segment, or (bytes == nullptr) rows no
// segment covers, which decode to empty strings.  Its rows are chunks
// first_chunk, first_chunk + 1, ... of the column's chunk list, which the
// segment pre-pass writes; the range starts at column row col_row.  codec
// is the segment's sdr_codec (FSST, DICTIONARY or UNCOMPRESSED; 0 for a gap).
struct FsstSeg {
  const uint8_t* bytes;
  uint32_t bytes_size;
  uint32_t row_count;
  uint32_t first_chunk;
  uint32_t col_row;
  uint16_t codec;
  uint16_t chunk_rows;  // of its chunks but the last; FSST_CHUNK_ROWS but in columns of DICTIONARY segments
  uint32_t pad;
};
static_assert(sizeof(FsstSeg) == 32, "FsstSeg layout");

// Rows per chunk of a column of DICTIONARY segments alone: of 4096, 2048 and
// 1024 the widest that still gives each of the 256 CUs two chunks.  A chunk's
// descriptors and look-back are round trips that more rows share (8 Mi labels: a
// call of 103 us in chunks of 1024 rows, 71 of 2048, 54 of 4096), but fewer chunks
// leave CUs idle (a row group: 23, 23, 25 us; 512 Ki rows: 26, 26, 28; 1 Mi: 33,
// 28, 29; 2 Mi: 43, 35, 32).
inline uint32_t label_chunk_rows(uint32_t total_rows)
{
  uint32_t r = WIDE_CHUNK_ROWS;
  while (r > FSST_CHUNK_ROWS && total_rows / r < 512u) r /= 2u;
  return r;
}

// Chunks covering a range.
inline uint32_t fsst_chunk_count(const FsstSeg& sg)
{
  return sg.row_count / sg.chunk_rows + (sg.row_count % sg.chunk_rows ? 1u : 0u);
}

// A chunk: `rows` rows starting at segment row `row_begin` (column row
// `col_row`).  Chunks are listed in column row order.
struct FsstChunk {
  uint32_t seg;
  uint32_t row_begin;
  uint32_t rows;
  uint32_t col_row;
};

// What the segment pre-pass (k_fsst_prep) leaves for each chunk: the
// segment's header fields and the chunk's compressed-length prefix bounds,
// so a chunk decode issues all of its loads at once.
constexpr uint32_t FI_WIDTH = 0xFFu;      // bits 0-7: length-stream bit width
constexpr uint32_t FI_OK    = 1u << 8;    // header valid, symbol table imported
constexpr uint32_t FI_LFAST = 1u << 9;    // the chunk's length fields lie inside the segment
constexpr uint32_t FI_HUGE  = 1u << 10;   // a row of the chunk has >= 1 MiB of compressed bytes
constexpr uint32_t FI_DICT  = 1u << 11;   // a DICTIONARY segment (bits 0-7: selection width)
constexpr uint32_t FI_UNC   = 1u << 12;   // an UNCOMPRESSED string segment
constexpr uint32_t FI_DFSST = 1u << 13;   // a DICT_FSST segment (bytes: its DictFsstSeg)

struct FsstChunkInfo {
  const uint8_t* bytes;  // the segment
  uint32_t c_lo;         // compressed bytes of the segment's rows before the chunk
                         // (DICTIONARY: index_buffer_offset)
  uint32_t c_hi;         // ... up to and including the chunk's last row
                         // (DICTIONARY: index_buffer_count)
  uint32_t dict_end;
  uint32_t flags;        // width and FI_* bits
  uint32_t bytes_size;
  uint32_t pad;
};
static_assert(sizeof(FsstChunkInfo) == 32, "FsstChunkInfo layout");

// A segment's symbol table as the decoder reads it: symbol bytes (zero
// above the length) and lengths, 256 codes (255, the escape, has length 0).
struct FsstSymTab {
  uint64_t sym[256];
  uint8_t len[256];
};
static_assert(sizeof(FsstSymTab) == 2304, "FsstSymTab layout");

// A DICT_FSST segment (strings/dict_fsst.cu:17-38): the host fills the
// region offsets from the 16-byte header (:64-72, :516-525), the dictionary
// pre-pass the entry offsets, and `src` is the raw dict region (mode 0, or
// a dictionary of at most one entry) or the entries the predecode pass
// wrote.  Entry k of the segment is [e[k], e[k + 1]) of src.
struct DictFsstSeg {
  const uint8_t* bytes;  // the segment
  const uint32_t* e;     // dict_count + 1 entry offsets into src
  const uint8_t* src;
  uint64_t src_size;     // readable bytes at src
  uint32_t bytes_size;
  uint32_t dict_count;
  uint32_t off_dict, off_symtab, off_slens, off_didx;
  uint32_t range;        // its row range: index of its symbol table
  uint8_t mode, slw, diw, valid;
  uint32_t e_byte;       // offset of its byte_off entries in the pre-pass array
  uint32_t pad;
};
static_assert(sizeof(DictFsstSeg) == 72, "DictFsstSeg layout");

// Device memory of a column's DICT_FSST passes.
struct DfsstWork {
  DictFsstSeg* desc;   // the descriptors
  uint32_t* pre_size;  // bytes of each segment's predecoded entries
  uint32_t* e_byte;    // entry offsets: compressed ...
  uint32_t* e_dec;     // ... and decoded
  uint8_t* pre;        // the predecoded entries, segment by segment (null: none)
};

// DICT_FSST passes (k_fsst.hip): the 16-byte headers of the DICT_FSST
// ranges into hdr[4 * i] (ranges of other codecs are skipped); the
// per-segment dictionary pre-pass (byte and decoded entry offsets, symbol
// table, per-segment decoded total and inline-NULL flag into out[2 * j]);
// the predecode of FSST-mode entries, beside the segment pre-pass
// (launch_fsst_prep); and the inline-NULL marking of a column's mask (`fresh`: all
// valid, not written yet), with the rows it clears in each of
// dfsst_null_counts() counts.  Ranges, descriptors, headers, `out` and `counts`
// are pinned host memory, which the passes read and write in place; the last pass
// takes the ranges from the copy that the segment pre-pass left on the device.
constexpr uint32_t DFSST_NULL_COUNTS = 2048;  // at most
inline uint32_t dfsst_null_counts(uint32_t total_rows)
{
  const uint32_t tiles = (total_rows - 1u) / 2048u + 1u;
  return tiles < DFSST_NULL_COUNTS ? tiles : DFSST_NULL_COUNTS;
}
hipError_t launch_dfsst_headers(const FsstSeg* segs, uint32_t n_ranges, uint32_t* hdr, hipStream_t s);
hipError_t launch_dfsst_prep(const DictFsstSeg* dseg, uint32_t n_dseg, const DfsstWork& wk, FsstSymTab* d_tabs,
                             uint32_t* out, hipStream_t s);
hipError_t launch_dfsst_nulls(const FsstSeg* d_segs, uint32_t n_ranges, uint8_t* d_mask, uint32_t total_rows,
                              bool fresh, uint32_t* counts, hipStream_t s);

// What a column decode reports to the host, in pinned memory.
struct FsstResult {
  uint64_t total;  // decoded chars
  uint64_t error;  // the look-back did not complete
};

// Device state of one column decode: ticket counter, look-back status per
// chunk, error flag and the decoded chars total, which the last chunk also
// writes to `result` when that is set.
struct FsstState {
  uint32_t ticket;
  uint32_t error;
  uint64_t total;
  FsstResult* result;
  uint32_t* failed;    // a batch's: where a failure is told as well (may be null)
  uint64_t status[1];  // n_chunks entries
};
constexpr uint32_t FSST_STATE_WORDS = 4;  // 8-byte words before status

// Segment pre-pass over n_segs ranges: writes the chunk list, the chunks'
// FsstChunkInfo and the segments' symbol tables, and sets up the state (its
// result may be null).  With `host` the ranges are pinned host memory: a few
// travel in the kernel arguments, each of many is read by its block.  With `wk` the
// n_dseg DICT_FSST segments' entries are predecoded in the same launch, and
// `copy`, if set, receives the ranges in device memory; without it the column's
// n_units mask pieces (memory the device reads) are built in the same launch, with
// their null counts.
hipError_t launch_fsst_prep(const FsstSeg* segs, uint32_t n_segs, FsstChunk* d_chunks, FsstChunkInfo* d_info,
                            FsstSymTab* d_tabs, FsstState* d_state, FsstResult* result, hipStream_t s, bool host,
                            const DfsstWork* wk, uint32_t n_dseg, FsstSeg* copy, const MaskUnit* units,
                            uint32_t n_units, uint32_t* counts);
// `chunk_rows`: 0 for a column with FSST segments, else the rows of its chunks.
// `ordered`: by ticket, see FSST_UNORDERED_SHARE.
hipError_t launch_fsst(bool ordered, uint32_t chunk_rows, const FsstChunk* d_chunks, uint32_t first, uint32_t n,
                       uint32_t n_chunks_total, const FsstChunkInfo* d_info, const FsstSymTab* d_tabs,
                       FsstState* d_state, int32_t* d_offsets, uint8_t* d_chars, uint64_t chars_cap,
                       uint32_t total_rows, hipStream_t s);

}  // namespace sdr
