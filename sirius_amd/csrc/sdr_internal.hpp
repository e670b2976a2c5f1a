// sdr_internal.hpp — host-side helpers shared by the C ABI translation units.
#pragma once

#include "../../include/sdr/decode.h"
#include "sdr_kernels.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

namespace sdr {

int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();
const char* last_error();

#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t _e = (expr);                                                             \
    if (_e != hipSuccess) return ::sdr::fail(SDR_E_HIP, "%s: %s", #expr, hipGetErrorString(_e)); \
  } while (0)

void ensure_pool(int dev);
int device_alloc(void** p, size_t bytes, hipStream_t s);
void device_free(void* p, hipStream_t s);
// Per-call descriptors in a reused slot (pinned + device buffer): copies
// h_src to the slot's device buffer on s and returns it; desc_release marks
// the slot free once the work enqueued on s so far has completed.
int desc_acquire(const void* h_src, size_t bytes, hipStream_t s, void** d_out, void** token);
int desc_release(void* token, hipStream_t s);
// The same without a copy: h_src in a slot's pinned buffer, which kernels read in
// place.  For descriptors of which a workgroup reads one: its 24 bytes over the
// bus cost a launch less than the copy before it and the event between them (64
// Mi rows in 1641 segments 238 -> 234 us, 32 Mi nullable rows in 547 97 -> 93 us).
// `waits`: the call waits for its result.
int desc_pinned(const void* h_src, size_t bytes, hipStream_t s, bool waits, void** p, void** token);
// A slot's pinned (device-accessible) and device buffers of at least these
// sizes, nothing copied, for a call that waits for its result on `s`; given back
// with desc_release, or, when no work on them can be pending (the stream was
// synchronised), slot_release_idle.
int slot_acquire(size_t h_bytes, size_t d_bytes, hipStream_t s, void** h_out, void** d_out, void** token);
void slot_release_idle(void* token, hipStream_t s);

bool type_ok_for(uint32_t codec, uint32_t ts);
bool codec_fixed(uint32_t codec);
int check_runs(const sdr_run* runs, uint32_t n, uint32_t total_rows, const char* what);
int check_validity_runs(const sdr_run* runs, uint32_t n, uint32_t total_rows);
// Append the pieces of a column's null mask: its validity segments (a later
// one wins where two share a byte) and all-valid rows where none lies.
void add_mask_units(const sdr_run* runs, uint32_t n, uint32_t total_rows, uint8_t* d_mask, std::vector<MaskUnit>& out);
// The launch of a call's pieces.  counts[i] is piece i's null count once `s`
// has been synchronised; desc_release(token, s) then ends the use of counts.
int masks_launch(const std::vector<MaskUnit>& units, hipStream_t s, const uint32_t** counts, void** token);

// A call's null-mask pieces: `units` in memory the device reads, and (null for a
// plan) `host`, from which they may travel in kernel arguments; piece i's null
// count goes to counts[i].
struct MaskLaunch {
  const MaskUnit* host  = nullptr;
  const MaskUnit* units = nullptr;
  uint32_t* counts      = nullptr;
  uint32_t n            = 0;
  const uint32_t* ends  = nullptr;  // a call's: where each of n_cols columns' pieces end
  uint32_t n_cols       = 0;
};
// Pieces and counts in pinned memory, to be launched; `token` as for masks_launch.
int masks_prepare(const std::vector<MaskUnit>& units, hipStream_t s, MaskLaunch* m, void** token);

// Bytes that a call's launches write.  Segments may share rows, and columns outputs
// and masks: the codec or the column that comes later wins, launch after launch.
// Blocks of one launch have no order, so what shares a byte may not share a launch.
class WrittenBytes {
 public:
  void add(const void* p, uint64_t bytes)
  {
    const uintptr_t lo = reinterpret_cast<uintptr_t>(p);
    if (bytes == 0) return;
    if (!spans_.empty() && spans_.back().second == lo) spans_.back().second = lo + bytes;
    else spans_.push_back({lo, lo + bytes});
  }
  bool any_twice()
  {
    std::sort(spans_.begin(), spans_.end());
    for (size_t i = 1; i < spans_.size(); ++i)
      if (spans_[i].first < spans_[i - 1].second) return true;
    return false;
  }

 private:
  std::vector<std::pair<uintptr_t, uintptr_t>> spans_;  // one for a column whose segments come in row order
};

// One fixed-width run and where its rows go.
struct RunTarget {
  const sdr_run* run;
  void* d_out;
  uint32_t type_size;
};
int decode_runs(const std::vector<RunTarget>& targets, hipStream_t s, uint32_t mode, const MaskLaunch& masks = {});
int validate_fixed_columns(const sdr_column* cols, uint32_t n_cols);
int validate_string_column(const sdr_string_column* col);
// The column has DICT_FSST segments (decoded only by the per-column passes).
bool has_dict_fsst(const sdr_string_column* col);
// SDR_LAUNCH_PERSISTENT: one persistent launch through a thread-local batch.
int decode_table_persistent(sdr_column* cols, uint32_t n_cols, hipStream_t s);
int decode_strings_persistent(sdr_string_column* col, hipStream_t s);
// Batch internals used by the server (sdr_serve.cpp); the caller validates.
int batch_add_fixed(sdr_batch* b, sdr_column* cols, uint32_t n_cols);
int batch_add_strings(sdr_batch* b, sdr_string_column* col);
int batch_launch(sdr_batch* b, hipStream_t s);
int batch_ready(sdr_batch* b);    // 1 finished, 0 running, < 0 error
int batch_collect(sdr_batch* b);  // after batch_ready: write back totals and null counts
int batch_column_status(const sdr_batch* b, const sdr_string_column* col);

// Segments grouped by (codec, type size); [first, first + count) in the
// descriptor array.
struct Batch {
  uint32_t codec, ts;
  uint32_t first, count;
  uint32_t max_rows;
};

}  // namespace sdr

struct sdr_plan {
  uint32_t mode   = 0;
  uint32_t n_cols = 0;
  std::vector<sdr::Batch> batches;
  std::vector<sdr::FixedSeg> all;
  sdr::FixedSeg* d_segs = nullptr;
  bool shared = false;  // outputs share bytes
  std::vector<sdr_column> masked;  // columns with a null mask, in column order
  std::vector<bool> col_masked;
  std::vector<uint32_t> mask_ends;  // per masked column: its pieces end here in the list of all
  sdr::MaskUnit* d_units = nullptr;
  uint32_t* d_counts     = nullptr;  // null count of each piece
  ~sdr_plan();
};
