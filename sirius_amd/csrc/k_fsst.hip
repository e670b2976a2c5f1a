// k_fsst.hip — per-column FSST decode kernel (one launch decodes every chunk
// of a VARCHAR column; see dec_fsst.hpp for the chunk decoder).
#include "dec_fsst.hpp"
#include "dec_groups.hpp"
#include "sdr_tune.hpp"

#include <cstring>

namespace sdr {

// The chunk of this workgroup of a launch over chunks [first, first + grid), of
// which all before `first` are done: by its own number, or by ticket.
__device__ __forceinline__ uint32_t chunk_number(FsstState* st, uint32_t first, uint32_t ordered)
{
  __shared__ uint32_t s_ticket;
  if (!ordered) return first + blockIdx.x;
  if (threadIdx.x == 0) s_ticket = atomicAdd(&st->ticket, 1u);
  __syncthreads();
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(s_ticket)));
}

__global__ __launch_bounds__(FSST_THREADS) __attribute__((amdgpu_waves_per_eu(6))) void k_fsst(
  const FsstChunk* __restrict__ chunks, uint32_t n_chunks, const FsstChunkInfo* __restrict__ info,
  const FsstSymTab* __restrict__ tabs, FsstState* __restrict__ st, int32_t* __restrict__ offsets,
  uint8_t* __restrict__ chars, uint64_t chars_cap, uint32_t total_rows, uint32_t spin_limit, uint32_t first,
  uint32_t ordered)
{
  __shared__ FsstSmem sm;
  const uint32_t c = chunk_number(st, first, ordered);
  if (c >= n_chunks) return;  // never taken: the grids are the chunk count
  const FsstChunk ch = chunks[c];
  fsst_chunk(ch, info[c], tabs + (ch.seg == FSST_GAP ? 0u : ch.seg), c, n_chunks, st, offsets, chars, chars_cap,
             total_rows, spin_limit, sm);
}

// A column without FSST segments, in chunks of up to RPT * 512 rows.  A kernel
// of its own: within k_fsst the decode was a call, which saved and restored
// registers through scratch memory, the larger part of its time (8 Mi labels
// 119 us, 2 M rows of 27 chars 57 us; here 57 us, with the labels in LDS 36 us, and
// 35 us, of which 8 us and 9 us are the tickets it no longer draws).  Six wavefronts to a
// SIMD are three workgroups to a CU; for four, rows' state spills (73 us, 70 us).
template <uint32_t RPT>
__global__ __launch_bounds__(FSST_THREADS) __attribute__((amdgpu_waves_per_eu(6))) void k_plain(
  const FsstChunk* __restrict__ chunks, uint32_t n_chunks, const FsstChunkInfo* __restrict__ info,
  FsstState* __restrict__ st, int32_t* __restrict__ offsets, uint8_t* __restrict__ chars, uint64_t chars_cap,
  uint32_t total_rows, uint32_t spin_limit, uint32_t first, uint32_t ordered)
{
  __shared__ PlainSmem sm;
  const uint32_t c = chunk_number(st, first, ordered);
  if (c >= n_chunks) return;  // never taken: the grids are the chunk count
  const FsstChunk ch     = sload(chunks + c);
  const FsstChunkInfo ci = sload(info + c);
  if (ch.seg != FSST_GAP && (ci.flags & FI_OK)) {
    const PlainArgs args{ci.bytes,   ci.bytes_size, ci.dict_end, ci.flags, ci.c_lo, ci.c_hi,   ch.row_begin, ch.rows,
                         ch.col_row, c,             n_chunks,    st,       offsets, chars,     chars_cap,    total_rows,
                         spin_limit};
    if ((ci.flags & FI_DICT) && ci.c_hi <= LABEL_ENTRIES && label_chunk<RPT>(args, sm)) return;
    plain_chunk<RPT>(args, sm);
    return;
  }
  // rows of no segment, or of one with a bad header, are empty
  const uint64_t base = fsst_lookback(c, n_chunks, 0u, st, spin_limit, sm);
  for (uint32_t r = threadIdx.x; r < ch.rows; r += FSST_THREADS)
    gbl(offsets)[ch.col_row + r] = static_cast<int32_t>(static_cast<uint32_t>(base));
  if (c == n_chunks - 1u && threadIdx.x == 0)
    gbl(offsets)[total_rows] = static_cast<int32_t>(static_cast<uint32_t>(base));
}

// Segment pre-pass: one workgroup per segment (grid-stride), which also clears
// the look-back status of its chunks (a launch of its own for that, and a copy
// of the ranges to the device before it, were 10 us of a 76 us call).
//
// Up to RANGES_INLINE ranges travel in the kernel arguments; more are read
// where they are, a device array or pinned memory.
//
// Few ranges have the chip to themselves: twice the waves share a segment's
// chunks (seven segments 10.6 -> 8.7 us).  956 segments fill it with 256-thread
// workgroups, and larger ones only start later (18.9 -> 22 us).
constexpr uint32_t RANGES_INLINE = 100;
struct DevRanges {
  static constexpr uint32_t THREADS = 256;
  const FsstSeg* p;
  __device__ __forceinline__ FsstSeg at(uint32_t i) const { return sload(p + i); }
};
struct RangesInline {
  static constexpr uint32_t THREADS = 512;
  FsstSeg seg[RANGES_INLINE];
  __device__ __forceinline__ FsstSeg at(uint32_t i) const { return uniform(seg[i]); }
};

template <uint32_t NT, class Src>
__device__ __forceinline__ void fsst_prep_block(const Src& src, uint32_t n_segs, uint32_t block, uint32_t blocks,
                                                FsstChunk* __restrict__ chunks, FsstChunkInfo* __restrict__ info,
                                                FsstSymTab* __restrict__ tabs, FsstState* __restrict__ st,
                                                FsstResult* __restrict__ result, FsstSeg* __restrict__ copy,
                                                FsstPrepSmem<NT>& sm)
{
  if (block == 0 && threadIdx.x == 0) {
    st->ticket = 0;
    st->error  = 0;
    st->total  = 0;
    st->result = result;
    st->failed = nullptr;
  }
  for (uint32_t i = block; i < n_segs; i += blocks) {
    const FsstSeg sg = src.at(i);
    for (uint32_t k = threadIdx.x; uint64_t{k} * sg.chunk_rows < sg.row_count; k += NT)
      gbl(st->status)[sg.first_chunk + k] = 0;
    if (copy && threadIdx.x == 0) copy[i] = sg;
    fsst_prep_segment(sg, i, chunks, info, tabs + i, sm);
  }
}

// Its first `prep` workgroups; the others build the column's null mask, a piece
// each (in a launch of its own after the decode that took 4 us of a call of 58).
template <class Src>
__global__ __launch_bounds__(Src::THREADS) void k_fsst_prep(Src src, uint32_t n_segs, uint32_t prep,
                                                            FsstChunk* __restrict__ chunks,
                                                            FsstChunkInfo* __restrict__ info,
                                                            FsstSymTab* __restrict__ tabs, FsstState* __restrict__ st,
                                                            FsstResult* __restrict__ result,
                                                            const MaskUnit* __restrict__ units,
                                                            uint32_t* __restrict__ counts)
{
  __shared__ union Smem {
    FsstPrepSmem<Src::THREADS> prep;
    MaskSmem<Src::THREADS> mask;
    __device__ Smem() {}
  } sm;
  if (blockIdx.x < prep) {
    fsst_prep_block(src, n_segs, blockIdx.x, prep, chunks, info, tabs, st, result, nullptr, sm.prep);
  } else {
    const uint32_t u = blockIdx.x - prep;
    mask_block(sload(units + u), u, counts, nullptr, sm.mask);
  }
}

// ---- DICT_FSST passes ----

constexpr uint32_t DFSST_PREP_THREADS = 1024;

__global__ void k_dfsst_headers(const FsstSeg* __restrict__ segs, uint32_t n, uint32_t* __restrict__ hdr)
{
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const FsstSeg sg = gload(segs + i);
    const bool has   = sg.codec == SDR_CODEC_DICT_FSST && sg.bytes && sg.bytes_size >= 16u;
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w) hdr[4u * i + w] = has ? ld_u32_any(sg.bytes + 4u * w) : 0u;
  }
}

// The descriptors come in pinned memory and go to d_desc as well, which the passes
// after this one read.
__global__ __launch_bounds__(DFSST_PREP_THREADS) void k_dfsst_prep(const DictFsstSeg* __restrict__ dseg, uint32_t n,
                                                                   DfsstWork wk, FsstSymTab* __restrict__ tabs,
                                                                   uint32_t* __restrict__ out)
{
  __shared__ DfsstPrepSmem<DFSST_PREP_THREADS> sm;
  for (uint32_t j = blockIdx.x; j < n; j += gridDim.x) {
    const DictFsstSeg d = sload(dseg + j);
    if (threadIdx.x == 0) wk.desc[j] = d;
    dfsst_prep_segment(d, wk.e_byte, wk.e_dec, tabs + d.range, out + 2u * j, wk.pre_size + j, sm);
    __syncthreads();  // sm is reused by the next segment
  }
}

// Eight workgroups share a segment's entries, predecoded to `pre` behind those of
// the segments before it; beside them the column's segment pre-pass, which needs
// nothing of theirs.
constexpr uint32_t PREDECODE_THREADS = 256;  // one code of the table per thread
constexpr uint32_t PREDECODE_SHARE   = 8;
struct PredecodeSmem {
  uint64_t sym[256];
  uint8_t len[256];
};
__device__ __forceinline__ void dfsst_predecode_block(const DfsstWork& wk, uint32_t j, uint32_t part,
                                                      const FsstSymTab* __restrict__ tabs, PredecodeSmem& sm)
{
  DictFsstSeg d = uniform(gload(wk.desc + j));
  if (!d.valid || d.mode == 0u || d.dict_count <= 1u) return;  // uniform per block
  uint64_t at = 0;
  for (uint32_t i = lane_id(); i < j; i += WAVE) at += gbl(wk.pre_size)[i];
  at         = readlane_u64(wave_incl_sum_u64(at), WAVE - 1);
  d.src      = wk.pre + at;
  d.src_size = gbl(wk.pre_size)[j];
  if (part == 0 && threadIdx.x == 0) {
    wk.desc[j].src      = d.src;
    wk.desc[j].src_size = d.src_size;
  }
  sm.sym[threadIdx.x] = gbl(tabs[d.range].sym)[threadIdx.x];
  sm.len[threadIdx.x] = gbl(tabs[d.range].len)[threadIdx.x];
  __syncthreads();
  dfsst_predecode(d, wk.e_byte, sm.sym, sm.len, part * PREDECODE_THREADS + threadIdx.x,
                  PREDECODE_SHARE * PREDECODE_THREADS);
}

template <class Src>
__global__ __launch_bounds__(PREDECODE_THREADS) void k_dfsst_front(Src src, uint32_t n_segs, uint32_t prep, DfsstWork wk,
                                                                   FsstChunk* __restrict__ chunks,
                                                                   FsstChunkInfo* __restrict__ info,
                                                                   FsstSymTab* __restrict__ tabs,
                                                                   FsstState* __restrict__ st,
                                                                   FsstResult* __restrict__ result,
                                                                   FsstSeg* __restrict__ copy)
{
  __shared__ union Smem {
    FsstPrepSmem<PREDECODE_THREADS> prep;
    PredecodeSmem pre;
    __device__ Smem() {}
  } sm;
  if (blockIdx.x < prep) {
    fsst_prep_block(src, n_segs, blockIdx.x, prep, chunks, info, tabs, st, result, copy, sm.prep);
  } else {
    const uint32_t b = blockIdx.x - prep;
    dfsst_predecode_block(wk, b / PREDECODE_SHARE, b % PREDECODE_SHARE, tabs, sm.pre);
  }
}

// DICT_FSST's inline NULLs: a thread per byte of the null mask, a tile of 256
// bytes at a time, whose ranges the workgroup finds once (a search by every row,
// and each row's index in turn, took 15 us for 2 M rows; now 7 us).  The rows
// cleared are counted per workgroup, into pinned memory.  `fresh`: the mask is all
// valid and not written yet.
__global__ __launch_bounds__(256) void k_dfsst_nulls(const FsstSeg* __restrict__ segs, uint32_t n_ranges,
                                                     uint8_t* __restrict__ mask, uint32_t total_rows, uint32_t fresh,
                                                     uint32_t* __restrict__ counts)
{
  __shared__ uint32_t s_sum[4];
  uint32_t cleared = 0;
  for (uint64_t t0 = uint64_t{blockIdx.x} * 2048u; t0 < total_rows; t0 += uint64_t{gridDim.x} * 2048u) {
    const uint32_t row0 = static_cast<uint32_t>(t0) + 8u * threadIdx.x;
    uint32_t lo = 0, hi = n_ranges;  // the range holding the tile's first row: the last with col_row <= t0
    while (hi - lo > 1u) {
      const uint32_t mid = (lo + hi) / 2u;
      if (segs[mid].col_row <= t0) lo = mid;
      else hi = mid;
    }
    const bool mine   = row0 < total_rows;
    const uint32_t m0 = !mine ? 0u : fresh ? 0xFFu : mask[row0 / 8u];
    uint32_t m        = total_rows - row0 < 8u && mine ? m0 & ((1u << (total_rows - row0)) - 1u) : m0;
    const uint32_t in = m;
    for (uint32_t k = lo; k < n_ranges; ++k) {
      const FsstSeg sg = uniform(gload(segs + k));
      if (sg.col_row >= t0 + 2048u) break;
      if (sg.codec != SDR_CODEC_DICT_FSST || !sg.bytes) continue;
      const DictFsstSeg d = uniform(gload(reinterpret_cast<const DictFsstSeg*>(sg.bytes)));
      if (m && uint64_t{sg.col_row} + sg.row_count > row0 && sg.col_row < uint64_t{row0} + 8u)
        m = dfsst_null_byte(m, row0, sg, d);
    }
    if (m != in || (fresh && mine)) {
      mask[row0 / 8u] = static_cast<uint8_t>(m0 & ~(in & ~m));
      cleared += static_cast<uint32_t>(__builtin_popcount(in & ~m));
    }
  }
  const uint32_t sum = wave_incl_sum_u32(cleared);
  if (lane_id() == WAVE - 1u) s_sum[threadIdx.x / WAVE] = sum;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
}

hipError_t launch_dfsst_headers(const FsstSeg* d_segs, uint32_t n_ranges, uint32_t* d_hdr, hipStream_t s)
{
  if (n_ranges == 0) return hipSuccess;
  const uint32_t blocks = (n_ranges + 255u) / 256u;
  hipLaunchKernelGGL(k_dfsst_headers, dim3(blocks), dim3(256), 0, s, d_segs, n_ranges, d_hdr);
  return hipGetLastError();
}

hipError_t launch_dfsst_prep(const DictFsstSeg* dseg, uint32_t n_dseg, const DfsstWork& wk, FsstSymTab* d_tabs,
                             uint32_t* out, hipStream_t s)
{
  if (n_dseg == 0) return hipSuccess;
  hipLaunchKernelGGL(k_dfsst_prep, dim3(n_dseg < 4096u ? n_dseg : 4096u), dim3(DFSST_PREP_THREADS), 0, s, dseg, n_dseg,
                     wk, d_tabs, out);
  return hipGetLastError();
}

hipError_t launch_dfsst_nulls(const FsstSeg* d_segs, uint32_t n_ranges, uint8_t* d_mask, uint32_t total_rows,
                              bool fresh, uint32_t* counts, hipStream_t s)
{
  if (total_rows == 0 || n_ranges == 0) return hipSuccess;
  hipLaunchKernelGGL(k_dfsst_nulls, dim3(dfsst_null_counts(total_rows)), dim3(256), 0, s, d_segs, n_ranges, d_mask,
                     total_rows, fresh ? 1u : 0u, counts);
  return hipGetLastError();
}

hipError_t launch_fsst_prep(const FsstSeg* segs, uint32_t n_segs, FsstChunk* d_chunks, FsstChunkInfo* d_info,
                            FsstSymTab* d_tabs, FsstState* d_state, FsstResult* result, hipStream_t s, bool host,
                            const DfsstWork* wk, uint32_t n_dseg, FsstSeg* copy, const MaskUnit* units,
                            uint32_t n_units, uint32_t* counts)
{
  if (n_segs == 0) return hipSuccess;
  const uint32_t blocks = n_segs < 4096u ? n_segs : 4096u;
  auto go = [&](auto src) {
    using S = decltype(src);
    if (wk) {
      const uint32_t pre = wk->pre ? n_dseg * PREDECODE_SHARE : 0u;
      hipLaunchKernelGGL((k_dfsst_front<S>), dim3(blocks + pre), dim3(PREDECODE_THREADS), 0, s, src, n_segs, blocks, *wk,
                         d_chunks, d_info, d_tabs, d_state, result, copy);
    } else {
      hipLaunchKernelGGL((k_fsst_prep<S>), dim3(blocks + n_units), dim3(S::THREADS), 0, s, src, n_segs, blocks, d_chunks,
                         d_info, d_tabs, d_state, result, units, counts);
    }
  };
  if (host && n_segs <= RANGES_INLINE) {
    RangesInline ri{};
    std::memcpy(ri.seg, segs, size_t{n_segs} * sizeof(FsstSeg));
    go(ri);
  } else {
    go(DevRanges{segs});
  }
  return hipGetLastError();
}

hipError_t launch_fsst(bool ordered, uint32_t chunk_rows, const FsstChunk* d_chunks, uint32_t first, uint32_t n,
                       uint32_t n_chunks_total, const FsstChunkInfo* d_info, const FsstSymTab* d_tabs,
                       FsstState* d_state, int32_t* d_offsets, uint8_t* d_chars, uint64_t chars_cap,
                       uint32_t total_rows, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  // Tickets are global chunk numbers: a launch covering [first, first + n)
  // runs after every launch of lower chunks on the same stream.
  const uint32_t bound = tune(SDR_TUNE_FSST_SPIN_LIMIT), spin = ordered ? bound : fsst_unordered_spins(bound);
  if (chunk_rows) {
    static_assert(FSST_CHUNK_ROWS == 2u * FSST_THREADS && WIDE_CHUNK_ROWS == 8u * FSST_THREADS, "one kernel a size");
    auto* const k = chunk_rows <= FSST_CHUNK_ROWS ? k_plain<2> : chunk_rows < WIDE_CHUNK_ROWS ? k_plain<4> : k_plain<8>;
    hipLaunchKernelGGL(k, dim3(n), dim3(FSST_THREADS), 0, s, d_chunks, n_chunks_total, d_info, d_state, d_offsets,
                       d_chars, chars_cap, total_rows, spin, first, ordered ? 1u : 0u);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_fsst, dim3(n), dim3(FSST_THREADS), 0, s, d_chunks, n_chunks_total, d_info, d_tabs, d_state,
                     d_offsets, d_chars, chars_cap, total_rows, spin, first, ordered ? 1u : 0u);
  return hipGetLastError();
}

}  // namespace sdr
