// k_fixed.hip — gfx950 kernels for the fixed-width codecs: BITPACKING, RLE,
// ALP, ALPRD, UNCOMPRESSED, CONSTANT and the validity mask helpers.  One
// launch covers a batch of segments: blockIdx.y selects the segment,
// blockIdx.x * 4 + wave the work unit (decoders in dec_fixed.hpp).
#include "dec_groups.hpp"
#include "sdr_tune.hpp"

#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

namespace sdr {

template <typename T, class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_bitpacking(Src src, uint32_t gpw, uint32_t chunk_rows)
{
  __shared__ BpSmem sm;
  bp_block<T>(src.at(blockIdx.y), blockIdx.x, gpw, chunk_rows, sm);
}

// The segment (y) and the block of it (x) that a workgroup of a grid of gx blocks
// by segments takes: of `blocks` in all as GROUP_XCD_RUN says, or (0, and in the
// small calls whose descriptors are arguments) its own.
struct GridAt {
  uint32_t x, y;
};
template <class Src>
__device__ __forceinline__ GridAt grid_at(uint32_t gx, uint32_t blocks)
{
  if (std::is_same_v<Src, SegsInline> || !blocks) return {blockIdx.x, blockIdx.y};
  const uint32_t b = xcd_order(blockIdx.y * gx + blockIdx.x, blocks, GROUP_XCD_RUN);
  return {b % gx, b / gx};
}

template <typename T, bool RD, class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_alp(Src src, uint32_t vpw, uint32_t gx, uint32_t blocks)
{
  __shared__ AlpSmem<RD> sm;
  const GridAt at = grid_at<Src>(gx, blocks);
  alp_block<T, RD>(src.at(at.y), at.x, vpw, sm);
}

template <uint32_t TS, class Src>
__global__ __launch_bounds__(RLE_THREADS) void k_rle(Src src, uint32_t n_segs, uint32_t slices, uint32_t slice_rows)
{
  __shared__ RleSmem sm;
  rle_block<TS>(src, 0, n_segs, blockIdx.x, gridDim.x, slices, slice_rows, sm);
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_copy(Src src, uint32_t type_size, uint32_t gx, uint32_t blocks)
{
  const GridAt at = grid_at<Src>(gx, blocks);
  copy_block<false>(src.at(at.y), at.x, type_size);
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_constant(Src src, uint32_t type_size)
{
  copy_block<true>(src.at(blockIdx.y), blockIdx.x, type_size);
}

__global__ void k_fill_u8(uint8_t* p, uint8_t v, uint64_t n)
{
  for (uint64_t i = uint64_t{blockIdx.x} * blockDim.x + threadIdx.x; i < n; i += uint64_t{gridDim.x} * blockDim.x)
    p[i] = v;
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_null_mask(Src src, uint32_t* __restrict__ counts,
                                                             unsigned long long* __restrict__ total)
{
  __shared__ MaskSmem<> sm;
  mask_block(src.at(blockIdx.x), blockIdx.x, counts, total, sm);
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void k_groups(Src src, GroupTable t)
{
  __shared__ GroupSmem sm;
  groups_block(src, t, blockIdx.x, sm);
}

// ===========================================================================
// launch wrappers
// ===========================================================================
namespace {
constexpr uint32_t MAX_GRID_Y = 65535;

// Call f(src, m) for every launch over the n descriptors at
// segs[seg_base..]: device descriptors in pieces of at most max_m, or host
// descriptors copied into the kernel arguments SEGS_INLINE at a time.
template <typename F>
hipError_t for_segs(const FixedSeg* segs, uint32_t seg_base, uint32_t n, bool host, uint32_t max_m, F f)
{
  const uint32_t lim = host ? std::min(max_m, SEGS_INLINE) : max_m;
  for (uint32_t b = 0; b < n; b += lim) {
    const uint32_t m = n - b < lim ? n - b : lim;
    if (host) {
      SegsInline si{};
      std::memcpy(si.seg, segs + seg_base + b, size_t{m} * sizeof(FixedSeg));
      f(si, m);
    } else {
      f(DevSegs{segs, seg_base + b}, m);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
// What grid_at takes for a grid of gx by m blocks: 32 Mi rows of ALP take 81.9 us in
// plain order and 79.2 so (16 Mi of ALP-RD 71.6, 68.5; 32 Mi copied 120.9, 118.6),
// but a row group of ALP-RD 9.5 and 9.8 (the division), and ten 12.0 and 12.3.
// BITPACKING stays as it is (one byte 19.2, 19.7; four 29.9, 29.7).
uint32_t ordered_blocks(uint64_t gx, uint32_t m)
{
  const uint64_t n = gx * m;
  return n >= 4u * N_XCD * GROUP_XCD_RUN && n <= 0x7FFFFFFFull ? static_cast<uint32_t>(n) : 0u;
}
}  // namespace

hipError_t launch_bitpacking(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t ts,
                             hipStream_t s, bool host)
{
  if (n == 0 || max_rows == 0) return hipSuccess;
  const uint32_t gpw   = tune(SDR_TUNE_BP_GROUPS_PER_WAVE, ts);
  const uint32_t chunk = tune(SDR_TUNE_BP_CHUNK_ROWS, ts);
  const uint32_t units = (max_rows + BP_GROUP - 1) / BP_GROUP;
  const uint32_t gx    = (units + WAVES_PER_BLOCK * gpw - 1) / (WAVES_PER_BLOCK * gpw);
  return for_segs(segs, seg_base, n, host, MAX_GRID_Y, [&](auto src, uint32_t m) {
    using S = decltype(src);
    const dim3 g(gx, m);
    switch (ts) {
      case 1: hipLaunchKernelGGL((k_bitpacking<uint8_t, S>), g, dim3(BLOCK_THREADS), 0, s, src, gpw, chunk); break;
      case 2: hipLaunchKernelGGL((k_bitpacking<uint16_t, S>), g, dim3(BLOCK_THREADS), 0, s, src, gpw, chunk); break;
      case 4: hipLaunchKernelGGL((k_bitpacking<uint32_t, S>), g, dim3(BLOCK_THREADS), 0, s, src, gpw, chunk); break;
      default: hipLaunchKernelGGL((k_bitpacking<uint64_t, S>), g, dim3(BLOCK_THREADS), 0, s, src, gpw, chunk); break;
    }
  });
}

// Rows of a slice: what the knob says if it was set, else 8192, or fewer while
// the launch has less than two blocks for each CU.  Every block walks all of its
// segment's counts, so small slices walk more (64 Mi rows in runs of 16: 4096
// rows 154 us, 8192 111 us, 16384 119 us; 10 M in runs of 200: 16, 12, 13 us), but
// ten segments in slices of 8192 or 2048 rows are 150 or 600 blocks: 8.4 us, 6.5 us.
static uint32_t rle_slice_rows(uint32_t n_segs, uint32_t max_rows, uint32_t ts)
{
  if (!tune_rle_by_size(ts)) return tune(SDR_TUNE_RLE_SLICE_ROWS, ts);
  uint32_t sr = 8192;
  while (sr > 2048u && uint64_t{n_segs} * ((max_rows + sr - 1u) / sr) < 512u) sr /= 2u;
  return sr;
}

hipError_t launch_rle(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t ts,
                      hipStream_t s, bool host)
{
  if (n == 0 || max_rows == 0) return hipSuccess;
  const uint32_t sr     = rle_slice_rows(n, max_rows, ts);
  const uint32_t slices = (max_rows + sr - 1) / sr;
  // segments per launch so that the 1-D grid is one
  const uint32_t per = std::min(MAX_GRID_Y, MAX_BLOCKS / slices);
  return for_segs(segs, seg_base, n, host, per, [&](auto src, uint32_t m) {
    using S = decltype(src);
    const dim3 grid(m * slices), block(RLE_THREADS);
    switch (ts) {
      case 1: hipLaunchKernelGGL((k_rle<1, S>), grid, block, 0, s, src, m, slices, sr); break;
      case 2: hipLaunchKernelGGL((k_rle<2, S>), grid, block, 0, s, src, m, slices, sr); break;
      case 4: hipLaunchKernelGGL((k_rle<4, S>), grid, block, 0, s, src, m, slices, sr); break;
      default: hipLaunchKernelGGL((k_rle<8, S>), grid, block, 0, s, src, m, slices, sr); break;
    }
  });
}

hipError_t launch_alp(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t ts, bool rd,
                      hipStream_t s, bool host)
{
  if (n == 0 || max_rows == 0) return hipSuccess;
  const uint32_t vpw   = tune(SDR_TUNE_ALP_VECTORS_PER_WAVE, ts);
  const uint32_t units = (max_rows + ALP_VEC - 1) / ALP_VEC;
  const uint32_t gx    = (units + WAVES_PER_BLOCK * vpw - 1) / (WAVES_PER_BLOCK * vpw);
  return for_segs(segs, seg_base, n, host, MAX_GRID_Y, [&](auto src, uint32_t m) {
    using S = decltype(src);
    const dim3 g(gx, m);
    const uint32_t nb = ordered_blocks(gx, m);
    if (ts == 8) {
      if (rd) hipLaunchKernelGGL((k_alp<double, true, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw, gx, nb);
      else hipLaunchKernelGGL((k_alp<double, false, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw, gx, nb);
    } else {
      if (rd) hipLaunchKernelGGL((k_alp<float, true, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw, gx, nb);
      else hipLaunchKernelGGL((k_alp<float, false, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw, gx, nb);
    }
  });
}

hipError_t launch_uncompressed(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t ts,
                               hipStream_t s, bool host)
{
  if (n == 0 || max_rows == 0) return hipSuccess;
  const uint64_t gx = (uint64_t{max_rows} * ts + COPY_UNIT - 1) / COPY_UNIT;
  return for_segs(segs, seg_base, n, host, MAX_GRID_Y, [&](auto src, uint32_t m) {
    hipLaunchKernelGGL((k_copy<decltype(src)>), dim3(static_cast<uint32_t>(gx), m), dim3(BLOCK_THREADS), 0, s, src,
                       ts, static_cast<uint32_t>(gx), ordered_blocks(gx, m));
  });
}

hipError_t launch_constant(const FixedSeg* segs, uint32_t seg_base, uint32_t n, uint32_t max_rows, uint32_t ts,
                           hipStream_t s, bool host)
{
  if (n == 0 || max_rows == 0) return hipSuccess;
  const uint64_t gx = (uint64_t{max_rows} * ts + COPY_UNIT - 1) / COPY_UNIT;
  return for_segs(segs, seg_base, n, host, MAX_GRID_Y, [&](auto src, uint32_t m) {
    hipLaunchKernelGGL((k_constant<decltype(src)>), dim3(static_cast<uint32_t>(gx), m), dim3(BLOCK_THREADS), 0, s,
                       src, ts);
  });
}

// One y-block row per range (the reference's cudf::sequence per row group,
// duckdb_native_decoder.cpp:924-949, without the concatenation).
__global__ __launch_bounds__(BLOCK_THREADS) void k_rowids(const RowRange* __restrict__ ranges, int64_t* __restrict__ out)
{
  const RowRange r = gload(ranges + blockIdx.y);
  const gptr<int64_t> o = gbl(out + r.out_offset);
  for (uint32_t i = blockIdx.x * BLOCK_THREADS + threadIdx.x; i < r.count; i += gridDim.x * BLOCK_THREADS)
    o[i] = r.first_row + static_cast<int64_t>(i);
}

hipError_t launch_rowids(const RowRange* d_ranges, uint32_t n, uint32_t max_count, int64_t* out, hipStream_t s)
{
  if (n == 0 || max_count == 0) return hipSuccess;
  uint32_t gx = (max_count + BLOCK_THREADS - 1) / BLOCK_THREADS;
  if (gx > 1024) gx = 1024;
  for (uint32_t b = 0; b < n; b += 65535) {  // grid y limit
    const uint32_t m = n - b < 65535 ? n - b : 65535;
    hipLaunchKernelGGL(k_rowids, dim3(gx, m), dim3(BLOCK_THREADS), 0, s, d_ranges + b, out);
  }
  return hipGetLastError();
}

hipError_t launch_fill_u8(uint8_t* p, uint8_t v, uint64_t n, hipStream_t s)
{
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill_u8, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}

hipError_t launch_null_mask(const MaskUnit* units, uint32_t n, uint32_t* counts, unsigned long long* total,
                            hipStream_t s, bool host)
{
  if (!host) {
    if (n)
      hipLaunchKernelGGL((k_null_mask<DevMasks>), dim3(n), dim3(BLOCK_THREADS), 0, s, DevMasks{units}, counts, total);
    return hipGetLastError();
  }
  for (uint32_t b = 0; b < n; b += MASKS_INLINE) {
    const uint32_t m = n - b < MASKS_INLINE ? n - b : MASKS_INLINE;
    MasksInline mi{};
    std::memcpy(mi.unit, units + b, size_t{m} * sizeof(MaskUnit));
    hipLaunchKernelGGL((k_null_mask<MasksInline>), dim3(m), dim3(BLOCK_THREADS), 0, s, mi,
                       counts ? counts + b : nullptr, total);
  }
  return hipGetLastError();
}

// A group of n descriptors as the fused launch takes it, its first block to be set.
static Group group_of(const FixedGroup& f, uint32_t n)
{
  Group g{};
  const uint32_t lg = f.ts == 1 ? 0u : f.ts == 2 ? 1u : f.ts == 4 ? 2u : 3u;
  g.n_segs          = n;
  uint64_t blocks   = 0;
  switch (f.codec) {
    case SDR_CODEC_BITPACKING: {
      g.kind            = GK_BITPACKING + lg;
      g.a               = tune(SDR_TUNE_BP_GROUPS_PER_WAVE, f.ts);
      g.b               = tune(SDR_TUNE_BP_CHUNK_ROWS, f.ts);
      const uint32_t un = (f.max_rows + BP_GROUP - 1) / BP_GROUP;
      g.per_seg         = (un + WAVES_PER_BLOCK * g.a - 1) / (WAVES_PER_BLOCK * g.a);
      break;
    }
    case SDR_CODEC_RLE:
      g.kind    = GK_RLE + lg;
      g.a       = rle_slice_rows(n, f.max_rows, f.ts);
      g.per_seg = (f.max_rows + g.a - 1) / g.a;
      break;
    case SDR_CODEC_ALP:
    case SDR_CODEC_ALPRD: {
      g.kind            = (f.codec == SDR_CODEC_ALP ? GK_ALP : GK_ALPRD) + lg;
      g.a               = tune(SDR_TUNE_ALP_VECTORS_PER_WAVE, f.ts);
      const uint32_t un = (f.max_rows + ALP_VEC - 1) / ALP_VEC;
      g.per_seg         = (un + WAVES_PER_BLOCK * g.a - 1) / (WAVES_PER_BLOCK * g.a);
      break;
    }
    case MASK_GROUP:
      g.kind    = GK_MASK;
      g.per_seg = 1;
      break;
    default:
      g.kind    = f.codec == SDR_CODEC_UNCOMPRESSED ? GK_COPY : GK_CONSTANT;
      g.a       = f.ts;
      g.per_seg = static_cast<uint32_t>((uint64_t{f.max_rows} * f.ts + COPY_UNIT - 1) / COPY_UNIT);
  }
  blocks = uint64_t{n} * g.per_seg;
  g.blocks = blocks <= MAX_BLOCKS ? static_cast<uint32_t>(blocks) : 0u;  // 0: too many for a launch
  return g;
}

// The groups in the order their blocks are started: what reads most for a byte it
// writes first, what reads nothing last.  Of the orders tried this one is the
// best or equal throughout (10 M rows of six widths in the order of the columns 88
// us, so 78 us, with the constants first 82 us; 64 Mi rows RLE before bit-packing
// 246 us, after it 238 us; ALP before ALP-RD 112 us, after it 109 us).
static std::vector<FixedGroup> start_order(const FixedGroup* groups, uint32_t n_groups)
{
  auto rank = [](const FixedGroup& g) {
    switch (g.codec) {
      case MASK_GROUP: return 0;
      case SDR_CODEC_UNCOMPRESSED: return 1;
      case SDR_CODEC_ALPRD: return 2;
      case SDR_CODEC_ALP: return 3;
      case SDR_CODEC_BITPACKING: return 4;
      case SDR_CODEC_RLE: return 5;
      default: return 6;
    }
  };
  std::vector<FixedGroup> v(groups, groups + n_groups);
  std::stable_sort(v.begin(), v.end(), [&](const FixedGroup& a, const FixedGroup& b) { return rank(a) < rank(b); });
  return v;
}

bool device_groups(const FixedGroup* in_groups, uint32_t n_groups, const MaskUnit* units, uint32_t* counts, GroupTable* t,
                   uint32_t* blocks)
{
  const std::vector<FixedGroup> groups = start_order(in_groups, n_groups);
  *t              = GroupTable{};
  t->units        = units;
  t->counts       = counts;
  uint64_t first  = 0;
  for (uint32_t i = 0; i < n_groups; ++i) {
    if (!groups[i].count) continue;
    if (t->n == GROUPS_MAX) return false;
    Group g = group_of(groups[i], groups[i].count);
    if (g.blocks == 0 || first + g.blocks > MAX_BLOCKS) return false;
    g.first = static_cast<uint32_t>(first);
    g.seg   = groups[i].codec == MASK_GROUP ? 0u : groups[i].first;
    if (groups[i].codec == MASK_GROUP) g.a = 0;
    t->g[t->n++] = g;
    *blocks      = g.first + g.blocks;
    first        = (uint64_t{*blocks} + N_XCD - 1) / N_XCD * N_XCD;
  }
  return t->n != 0;
}

hipError_t launch_groups(const FixedGroup* in_groups, uint32_t n_groups, const FixedSeg* segs, const MaskUnit* units,
                         const MaskUnit* host_units, uint32_t* counts, hipStream_t s, bool host, bool* done)
{
  *done = false;
  if (n_groups < 2u || n_groups > GROUPS_MAX) return hipSuccess;
  const std::vector<FixedGroup> groups = start_order(in_groups, n_groups);
  if (!host) {
    GroupTable t;
    uint32_t blocks = 0;
    if (!device_groups(in_groups, n_groups, units, counts, &t, &blocks)) return hipSuccess;
    *done = true;
    hipLaunchKernelGGL((k_groups<DevSegs>), dim3(blocks), dim3(BLOCK_THREADS), 0, s, DevSegs{segs, 0}, t);
    return hipGetLastError();
  }
  // mask pieces travel with the descriptors if one launch holds all
  uint64_t total = 0;
  for (uint32_t i = 0; i < n_groups; ++i) total += groups[i].count;
  const bool carry = host_units && total <= SEGS_INLINE;
  // launches of at most SEGS_INLINE descriptors, groups cut where one is full
  GroupTable t{};
  SegsInline si{};
  uint64_t blocks = 0;
  uint32_t held   = 0;
  std::vector<GroupTable> tables;
  std::vector<SegsInline> inl;
  auto flush = [&]() {
    if (t.n == 0) return;
    t.units  = carry ? nullptr : units;
    t.counts = counts;
    tables.push_back(t);
    inl.push_back(si);
    t      = GroupTable{};
    blocks = 0;
    held   = 0;
  };
  for (uint32_t i = 0; i < n_groups; ++i) {
    const FixedGroup& f = groups[i];
    for (uint32_t b = 0; b < f.count;) {
      const bool here = f.codec != MASK_GROUP || carry;
      if (here && held == SEGS_INLINE) flush();
      const uint32_t n = here ? std::min(f.count - b, SEGS_INLINE - held) : f.count;
      Group g          = group_of(f, n);
      if (g.blocks == 0 || blocks + g.blocks > MAX_BLOCKS) return hipSuccess;
      g.first = static_cast<uint32_t>(blocks);
      if (f.codec == MASK_GROUP) g.a = b;
      if (here) {
        g.seg = held;
        if (f.codec == MASK_GROUP) std::memcpy(si.seg + held, host_units + b, size_t{n} * sizeof(MaskUnit));
        else std::memcpy(si.seg + held, segs + f.first + b, size_t{n} * sizeof(FixedSeg));
      }
      t.g[t.n++] = g;
      blocks     = (blocks + g.blocks + N_XCD - 1) / N_XCD * N_XCD;
      if (here) held += n;
      b += n;
    }
  }
  flush();
  *done = true;
  for (size_t i = 0; i < tables.size(); ++i) {
    const GroupTable& gt = tables[i];
    const Group& last    = gt.g[gt.n - 1u];
    const dim3 grid(last.first + last.blocks);
    hipLaunchKernelGGL((k_groups<SegsInline>), grid, dim3(BLOCK_THREADS), 0, s, inl[i], gt);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace sdr
