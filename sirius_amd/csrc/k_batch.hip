// k_batch.hip — persistent decode kernels of a mixed-codec batch.
//
// One launch decodes a whole device-resident work queue (sdr_batch.hpp):
// BITPACKING groups, RLE row slices, ALP/ALPRD vectors, UNCOMPRESSED and
// CONSTANT byte ranges and FSST chunks, from any number of columns and
// segments.  The queue is partitioned by codec and value width into groups
// (BatchGroup); each group is drained by its own persistent kernel,
// specialised for that one decoder, so it keeps the register and LDS
// footprint of the per-codec kernels instead of the union of all of them.
// A fixed-width group kernel's grid is its resident capacity.  Fixed-width
// entries are independent, so block b takes entries b, b + grid, ... with no
// claim at all; its four wavefronts decode an entry's units (an RLE slice is
// decoded by the whole block).  The FSST kernel runs one block per chunk, which
// waits for the offsets of the chunks before it in its column.  By
// default fixed-width segments are not queued: the front kernel decodes them
// beside the FSST pre-pass.
#include "dec_fsst.hpp"
#include "dec_groups.hpp"
#include "sdr_batch.hpp"

#include <algorithm>

namespace sdr {

// Per-wave staging of the fixed-width codecs, as in the per-codec kernels:
// 4 KiB of bitpacking or ALP codes, or the ALP-RD left stream plus 4 KiB of
// its right stream.
constexpr uint32_t BATCH_BP_STAGE = 4096;
static_assert(BATCH_WAVES == WAVES_PER_BLOCK, "fixed-width group block");

template <typename T>
__global__ __launch_bounds__(BLOCK_THREADS) void k_bgroup_bp(const BatchItem* __restrict__ items,
                                                             BatchQueue* __restrict__ q, uint32_t g)
{
  __shared__ uint32_t lds[WAVES_PER_BLOCK][(BATCH_BP_STAGE + 48) / 4];
  const uint32_t w     = wave_in_block();
  const uint32_t chunk = q->bp_chunk_rows[sizeof(T) == 1 ? 0 : sizeof(T) == 2 ? 1 : sizeof(T) == 4 ? 2 : 3];
  const uint32_t first = q->first[g], n = q->count[g];
  for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
    const BatchItem it = items[first + e];
    const uint32_t end = it.unit0 + it.n_units;
    for (uint32_t u = it.unit0 + w; u < end; u += WAVES_PER_BLOCK) {
      const uint32_t grc = it.row_count - u * BP_GROUP < BP_GROUP ? it.row_count - u * BP_GROUP : BP_GROUP;
      bp_group<T, BATCH_BP_STAGE>(it.seg, it.bytes_size, u, grc, reinterpret_cast<T*>(it.out) + size_t{u} * BP_GROUP,
                                  lds[w], chunk);
    }
  }
}

template <typename F, bool RD>
__global__ __launch_bounds__(BLOCK_THREADS) void k_bgroup_alp(const BatchItem* __restrict__ items,
                                                              BatchQueue* __restrict__ q, uint32_t g)
{
  __shared__ uint32_t lds[WAVES_PER_BLOCK][RD ? ALPRD_LEFT_WORDS + ALP_CHUNK_WORDS : ALP_CHUNK_WORDS];
  const uint32_t w     = wave_in_block();
  const uint32_t first = q->first[g], n = q->count[g];
  for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
    const BatchItem it = items[first + e];
    const uint32_t end = it.unit0 + it.n_units;
    for (uint32_t u = it.unit0 + w; u < end; u += WAVES_PER_BLOCK) {
      const uint32_t fill = it.row_count - u * ALP_VEC < ALP_VEC ? it.row_count - u * ALP_VEC : ALP_VEC;
      F* out = reinterpret_cast<F*>(it.out) + size_t{u} * ALP_VEC;
      if constexpr (RD) alprd_vector<F>(it.seg, it.bytes_size, u, fill, out, lds[w]);
      else alp_vector<F>(it.seg, it.bytes_size, u, fill, out, lds[w]);
    }
  }
}

template <uint32_t TS>
__global__ __launch_bounds__(RLE_THREADS) void k_bgroup_rle(const BatchItem* __restrict__ items,
                                                            BatchQueue* __restrict__ q, uint32_t g)
{
  __shared__ RleSmem sm;
  const uint32_t first = q->first[g], n = q->count[g];
  for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
    const BatchItem it = items[first + e];
    const uint32_t sr  = uint32_t{it.reserved} * 64u;
    for (uint32_t u = it.unit0; u < it.unit0 + it.n_units; ++u) {
      const uint32_t ra = u * sr;
      const uint32_t rb = it.row_count - ra < sr ? it.row_count : ra + sr;
      rle_slice_t<TS>(it.seg, it.bytes_size, it.row_count, ra, rb, it.out, sm);
    }
    __syncthreads();  // LDS reuse by the next entry
  }
}

__global__ __launch_bounds__(BLOCK_THREADS) void k_bgroup_copy(const BatchItem* __restrict__ items,
                                                               BatchQueue* __restrict__ q, uint32_t g)
{
  const uint32_t w     = wave_in_block();
  const uint32_t first = q->first[g], n = q->count[g];
  for (uint32_t e = blockIdx.x; e < n; e += gridDim.x) {
    const BatchItem it   = items[first + e];
    const uint64_t total = uint64_t{it.row_count} * it.ts;
    for (uint32_t u = it.unit0 + w; u < it.unit0 + it.n_units; u += WAVES_PER_BLOCK) {
      const uint64_t b0 = uint64_t{u} * COPY_UNIT_BYTES;
      const uint64_t b1 = total - b0 < COPY_UNIT_BYTES ? total : b0 + COPY_UNIT_BYTES;
      if (it.kind == BK_COPY) copy_span<WAVE>(it.seg, it.out, b0, b1, lane_id());
      else const_span<WAVE>(it.seg, it.ts, it.out, b0, b1, lane_id());
    }
  }
}

// Entry `idx` of the FSST group with the calling workgroup: on the columns' first
// states, or on those of the second attempt.
__device__ __forceinline__ void fsst_entry(const BatchQueue* __restrict__ q, uint32_t idx, bool again, FsstSmem& sm)
{
  // the entries list every column's chunks column by column, as the batch's
  // chunk and chunk-info arrays do: entry idx describes chunk idx of those
  // arrays, so the chunk loads need not wait for the column's; every lane
  // reads the same descriptors, kept in SGPRs
  const FsstEntry e      = uniform(gload(q->fsst_entries + idx));
  const FsstChunk ch     = uniform(gload(q->fsst_chunks + idx));
  const FsstChunkInfo ci = uniform(gload(q->fsst_info + idx));
  // the column comes through the scalar cache (read-only for the whole
  // launch), so its wait falls behind the loads of the symbol table and
  // the compressed bytes
  const FsstColumn col = sload(q->fsst_cols + e.col);
  fsst_chunk(ch, ci, q->fsst_tabs + (ch.seg == FSST_GAP ? 0u : ch.seg), e.chunk, col.n_chunks,
             again ? col.again : col.state, col.offsets, col.chars, col.chars_cap, col.total_rows,
             again ? q->spin_limit : fsst_unordered_spins(q->spin_limit), sm);
}

// One block per FSST entry (the grid is the group's entry count), that of its own
// number.  One chunk per block, with no loop around it, keeps the kernel at 80
// VGPRs: three workgroups of eight waves per CU.
__global__ __launch_bounds__(FSST_THREADS) __attribute__((amdgpu_waves_per_eu(6))) void k_bgroup_fsst(
  const BatchItem* __restrict__ items, BatchQueue* __restrict__ q, uint32_t g)
{
  __shared__ FsstSmem sm;
  (void)items;  // the FSST group's entries are q->fsst_entries
  if (blockIdx.x >= q->count[g]) return;  // the grid is the entry count: never taken
  fsst_entry(q, q->first[g] + blockIdx.x, false, sm);
}

// The columns that k_bgroup_fsst reported incomplete, from the start: their chunks
// in the order of tickets, so that a chunk's predecessors are done or held by
// workgroups that run, in whatever order those are started.  Right behind it on the
// stream: what follows a launch finds its columns complete.  Nearly always there are
// none (a served batch of 128 requests 334 us without this kernel, 333 us with it, 355 us
// with a ticket for each chunk at once).  Its occupancy is that of k_bgroup_fsst, with
// which it shares a called function.
__global__ __launch_bounds__(FSST_THREADS) __attribute__((amdgpu_waves_per_eu(6))) void k_batch_again(
  BatchQueue* __restrict__ q, uint32_t n)
{
  __shared__ FsstSmem sm;
  __shared__ uint32_t s_next;
  if (q->failed == 0u) return;
  for (;;) {
    if (threadIdx.x == 0) s_next = atomicAdd(&q->ticket, 1u);
    __syncthreads();
    const uint32_t i = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(s_next)));
    if (i >= n) return;
    const uint32_t idx = q->first[BG_FSST] + i;
    if (*gbl(&gload(q->fsst_cols + gload(q->fsst_entries + idx).col).state->error) != 0u) fsst_entry(q, idx, true, sm);
    __syncthreads();  // the next entry's use of sm and s_next
  }
}

// The FSST segment pre-pass over the queue's segments with `blocks` workgroups, of
// which this is the `block`-th; the first tells each column where its result goes.
template <uint32_t NT>
__device__ __forceinline__ void batch_prep(BatchQueue* __restrict__ q, uint32_t block, uint32_t blocks,
                                           FsstPrepSmem<NT>& sm)
{
  if (block == 0)
    for (uint32_t i = threadIdx.x; i < q->n_cols; i += NT) {
      const FsstColumn col      = gload(q->fsst_cols + i);
      gbl(col.state)->result = q->results + i;
      gbl(col.state)->failed = &q->failed;
      gbl(col.again)->result = q->results + q->n_cols + i;
    }
  const uint32_t n = q->n_fsst_segs;
  for (uint32_t i = block; i < n; i += blocks)
    fsst_prep_segment(gload(q->fsst_segs + i), i, q->fsst_chunks, q->fsst_info, q->fsst_tabs + i, sm);
}

__global__ __launch_bounds__(BATCH_PREP_THREADS) void k_batch_fsst_prep(BatchQueue* __restrict__ q)
{
  __shared__ FsstPrepSmem<BATCH_PREP_THREADS> sm;
  batch_prep(q, blockIdx.x, gridDim.x, sm);
}

// A launch's first kernel: the arena's upload, read where the host laid it out,
// the look-back states and the columns' results cleared.  (A copy to the device,
// and a reset after it, took 12 us and a gap of 20 us between them.)
__global__ __launch_bounds__(256) void k_batch_setup(u32x4* __restrict__ dst, const u32x4* __restrict__ src, uint32_t n,
                                                     uint64_t* __restrict__ words, uint32_t n_words,
                                                     uint64_t* __restrict__ results, uint32_t n_results)
{
  const uint32_t t = blockIdx.x * 256u + threadIdx.x, stride = gridDim.x * 256u;
  for (uint32_t i = t; i < n; i += stride) gbl(dst)[i] = gbl(src)[i];
  for (uint32_t i = t; i < n_words; i += stride) gbl(words)[i] = 0;
  for (uint32_t i = t; i < n_results; i += stride) gbl(results)[i] = 0;
}

// The FSST pre-pass (its first `prep` workgroups), the fixed-width segments and
// the null masks: the pre-pass waits on memory for most of its time and fills
// half the chip, so the others run beside it.
__global__ __launch_bounds__(BLOCK_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void k_batch_front(
  BatchQueue* __restrict__ q, uint32_t prep, DevSegs src, GroupTable t)
{
  __shared__ union Smem {
    FsstPrepSmem<BLOCK_THREADS> prep;
    GroupSmem groups;
    __device__ Smem() {}
  } sm;
  if (blockIdx.x < prep) batch_prep(q, blockIdx.x, prep, sm.prep);
  else groups_block(src, t, blockIdx.x - prep, sm.groups);
}

namespace {

// The kernel of group g (a BatchGroup).
const void* group_kernel(uint32_t g)
{
  switch (g) {
    case BG_BP1: return reinterpret_cast<const void*>(k_bgroup_bp<uint8_t>);
    case BG_BP2: return reinterpret_cast<const void*>(k_bgroup_bp<uint16_t>);
    case BG_BP4: return reinterpret_cast<const void*>(k_bgroup_bp<uint32_t>);
    case BG_BP8: return reinterpret_cast<const void*>(k_bgroup_bp<uint64_t>);
    case BG_RLE1: return reinterpret_cast<const void*>(k_bgroup_rle<1>);
    case BG_RLE2: return reinterpret_cast<const void*>(k_bgroup_rle<2>);
    case BG_RLE4: return reinterpret_cast<const void*>(k_bgroup_rle<4>);
    case BG_RLE8: return reinterpret_cast<const void*>(k_bgroup_rle<8>);
    case BG_ALP4: return reinterpret_cast<const void*>(k_bgroup_alp<float, false>);
    case BG_ALP8: return reinterpret_cast<const void*>(k_bgroup_alp<double, false>);
    case BG_ALPRD4: return reinterpret_cast<const void*>(k_bgroup_alp<float, true>);
    case BG_ALPRD8: return reinterpret_cast<const void*>(k_bgroup_alp<double, true>);
    case BG_COPY: return reinterpret_cast<const void*>(k_bgroup_copy);
    default: return reinterpret_cast<const void*>(k_bgroup_fsst);
  }
}

}  // namespace

hipError_t batch_group_launch_params(uint32_t g, const void** func, uint32_t* block, uint32_t* blocks_per_cu)
{
  *func  = group_kernel(g);
  *block = g == BG_FSST ? FSST_THREADS : (g >= BG_RLE1 && g <= BG_RLE8) ? RLE_THREADS : BLOCK_THREADS;
  int per = 0;
  const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, *func, static_cast<int>(*block), 0);
  *blocks_per_cu = per > 0 ? static_cast<uint32_t>(per) : 1u;
  return e;
}

hipError_t launch_batch_setup(void* dst, const void* src, size_t bytes, uint64_t* words, uint32_t n_words,
                              FsstResult* results, uint32_t n_results, hipStream_t s)
{
  static_assert(sizeof(FsstResult) % sizeof(uint64_t) == 0, "cleared by words");
  const uint32_t n = static_cast<uint32_t>(bytes / 16u), nr = n_results * static_cast<uint32_t>(sizeof(FsstResult) / 8u);
  const uint32_t most = std::max(n, std::max(n_words, nr));
  hipLaunchKernelGGL(k_batch_setup, dim3(std::min(512u, most / 256u + 1u)), dim3(256), 0, s, static_cast<u32x4*>(dst),
                     static_cast<const u32x4*>(src), n, words, n_words, reinterpret_cast<uint64_t*>(results), nr);
  return hipGetLastError();
}

hipError_t launch_batch_front(BatchQueue* q, uint32_t n_fsst_segs, const FixedGroup* groups, uint32_t n_groups,
                              const FixedSeg* segs, const MaskUnit* units, uint32_t* counts, hipStream_t s, bool* done)
{
  GroupTable t{};
  uint32_t blocks = 0;
  *done           = n_groups == 0 || device_groups(groups, n_groups, units, counts, &t, &blocks);
  // a multiple of 8 blocks ahead of the groups': a block's XCD stays its own
  const uint32_t prep = (std::min(n_fsst_segs, BATCH_PREP_GRID) + BATCH_XCDS - 1u) / BATCH_XCDS * BATCH_XCDS;
  *done               = *done && blocks <= MAX_BLOCKS - prep;
  if (!*done) return hipSuccess;
  if (prep + blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(k_batch_front, dim3(prep + blocks), dim3(BLOCK_THREADS), 0, s, q, prep, DevSegs{segs, 0}, t);
  return hipGetLastError();
}

hipError_t launch_batch_fsst_prep(BatchQueue* q, hipStream_t s)
{
  hipLaunchKernelGGL(k_batch_fsst_prep, dim3(BATCH_PREP_GRID), dim3(BATCH_PREP_THREADS), 0, s, q);
  return hipGetLastError();
}

const void* batch_fsst_prep_kernel() { return reinterpret_cast<const void*>(k_batch_fsst_prep); }

hipError_t launch_batch_again(BatchQueue* q, uint32_t n_entries, hipStream_t s)
{
  hipLaunchKernelGGL(k_batch_again, dim3(std::min(n_entries, 256u)), dim3(FSST_THREADS), 0, s, q, n_entries);
  return hipGetLastError();
}

hipError_t launch_batch_group(const BatchItem* items, BatchQueue* q, uint32_t g, uint32_t grid, hipStream_t s)
{
  const void* f = nullptr;
  uint32_t block = 0, per = 0;
  hipError_t e = batch_group_launch_params(g, &f, &block, &per);
  if (e != hipSuccess) return e;
  void* args[] = {&items, &q, &g};
  return hipLaunchKernel(f, dim3(grid), dim3(block), args, 0, s);
}

}  // namespace sdr
