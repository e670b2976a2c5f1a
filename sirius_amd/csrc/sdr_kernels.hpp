// sdr_kernels.hpp — host-side launch wrappers of the decode kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sdr {

// One fixed-width segment as the kernels see it.  `out` already points at
// the segment's first output row (d_out + row_offset * type_size).
struct FixedSeg {
  const uint8_t* bytes;
  uint8_t* out;
  uint32_t bytes_size;
  uint32_t row_count;
};
static_assert(sizeof(FixedSeg) == 24, "FixedSeg layout");

// Rows of one RLE slice (one 256-thread block decodes a slice) where nothing else
// is said: in a batch's queue entries.  Launches of their own choose by size.
constexpr uint32_t RLE_SLICE_ROWS = 16384;

// Descriptors a launch can carry in its kernel arguments.
constexpr uint32_t SEGS_INLINE = 128;

// Launch the decode of segments [seg_base, seg_base + n) of `segs`: a device
// array, or with `host` a host array whose descriptors travel in the kernel
// arguments (SEGS_INLINE per launch, no upload).  `max_rows` is the largest
// row_count among them (sizes the grid).
hipError_t launch_bitpacking(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows,
                             uint32_t type_size, hipStream_t s, bool host = false);
hipError_t launch_rle(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t type_size,
                      hipStream_t s, bool host = false);
hipError_t launch_alp(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t type_size,
                      bool rd, hipStream_t s, bool host = false);
hipError_t launch_uncompressed(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows,
                               uint32_t type_size, hipStream_t s, bool host = false);
hipError_t launch_constant(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows,
                           uint32_t type_size, hipStream_t s, bool host = false);

// Row ids: out[r.out_offset + i] = r.first_row + i for each range r (i < r.count).
struct RowRange {
  int64_t first_row;
  uint64_t out_offset;
  uint32_t count;
  uint32_t reserved;
};
hipError_t launch_rowids(const RowRange* d_ranges, uint32_t n, uint32_t max_count, int64_t* out, hipStream_t s);

hipError_t launch_fill_u8(uint8_t* p, uint8_t v, uint64_t n, hipStream_t s);

// Validity: a piece of a null mask, copied from a validity segment (src null:
// set to all valid) with its zero bits counted.  `past` has the bits of the
// piece's last byte that are past the column's rows.
struct MaskUnit {
  const uint8_t* src;
  uint8_t* dst;
  uint32_t bytes;
  uint32_t past;
};
static_assert(sizeof(MaskUnit) == 24, "MaskUnit layout");
constexpr uint32_t MASK_UNIT_BYTES = 8192;  // the largest piece: one 256-thread block
constexpr uint32_t MASKS_INLINE    = 120;   // pieces a launch can carry in its kernel arguments
// Build n pieces, one block each; piece i's null count is stored at counts[i],
// or (counts null) added to *total.  `units`: memory the device reads, or
// with `host` host memory whose pieces travel in the kernel arguments.
hipError_t launch_null_mask(const MaskUnit* units, uint32_t n, uint32_t* counts, unsigned long long* total,
                            hipStream_t s, bool host);

// Descriptors [first, first + count) of one codec and value width, or a call's
// mask pieces (codec MASK_GROUP, counted from 0).
constexpr uint32_t MASK_GROUP = 0xFFFFFFFFu;
struct FixedGroup {
  uint32_t codec, ts;
  uint32_t first, count;
  uint32_t max_rows;
};
// The groups in one launch (or as few as carry their descriptors in the kernel
// arguments, with `host`), *done set; or nothing, where a single group or the
// number of blocks asks for the codecs' own launches.  Null counts of `units` go
// to counts[i]; units and, without `host`, segs are memory the device reads,
// host_units (may be null) the pieces in host memory.
hipError_t launch_groups(const FixedGroup* groups, uint32_t n_groups, const FixedSeg* segs, const MaskUnit* units,
                         const MaskUnit* host_units, uint32_t* counts, hipStream_t s, bool host, bool* done);

}  // namespace sdr
