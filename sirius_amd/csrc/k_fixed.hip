// k_fixed.hip — gfx950 kernels for the fixed-width codecs: BITPACKING, RLE,
// ALP, ALPRD, UNCOMPRESSED, CONSTANT and the validity mask helpers.  One
// launch covers a batch of segments: blockIdx.y selects the segment,
// blockIdx.x * 4 + wave the work unit (decoders in dec_fixed.hpp).
#include "dec_fixed.hpp"
#include "dec_rle.hpp"
#include "sdr_tune.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

namespace sdr {

// Where a launch finds its segment descriptors: a device array, or the
// kernel arguments themselves (at most SEGS_INLINE descriptors, 3 KiB of the
// 4 KiB kernel-argument segment), which spares a small call the descriptor
// upload.  blockIdx-indexed, so the load is uniform per workgroup.
// A descriptor read at a workgroup-uniform index, its fields made uniform
// (scalar registers), so the decoders' address arithmetic on them stays
// scalar as with a restrict kernel-argument pointer.
__device__ __forceinline__ FixedSeg uniform_seg(const FixedSeg& v)
{
  const uint64_t b = reinterpret_cast<uint64_t>(v.bytes), o = reinterpret_cast<uint64_t>(v.out);
  FixedSeg r;
  r.bytes = reinterpret_cast<const uint8_t*>(
    (uint64_t{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(b >> 32)))} << 32) |
    static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(b))));
  r.out = reinterpret_cast<uint8_t*>(
    (uint64_t{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(o >> 32)))} << 32) |
    static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(o))));
  r.bytes_size = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v.bytes_size)));
  r.row_count  = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v.row_count)));
  return r;
}

struct DevSegs {
  const FixedSeg* p;
  uint32_t base;
  __device__ __forceinline__ FixedSeg at(uint32_t i) const { return uniform_seg(gload(p + base + i)); }
};
struct SegsInline {
  FixedSeg seg[SEGS_INLINE];
  __device__ __forceinline__ FixedSeg at(uint32_t i) const { return uniform_seg(seg[i]); }
};

// Wave w of a segment's block x decodes groups [(4x + w) * gpw, (4x + w + 1) * gpw).
constexpr uint32_t BP_STAGE = 4096;  // bytes of packed bits per wave; keeps 8 waves per SIMD resident
struct BpSmem {
  uint32_t lds[WAVES_PER_BLOCK][(BP_STAGE + 48) / 4];
};
template <typename T>
__device__ __forceinline__ void bp_block(const FixedSeg& sd, uint32_t x, uint32_t gpw, uint32_t chunk_rows, BpSmem& sm)
{
  const uint32_t w   = wave_in_block();
  const uint32_t ngr = (sd.row_count + BP_GROUP - 1) / BP_GROUP;
  const uint32_t k0  = (x * WAVES_PER_BLOCK + w) * gpw;
  for (uint32_t k = k0; k < k0 + gpw && k < ngr; ++k) {
    const uint32_t grc = sd.row_count - k * BP_GROUP < BP_GROUP ? sd.row_count - k * BP_GROUP : BP_GROUP;
    bp_group<T, BP_STAGE>(sd.bytes, sd.bytes_size, k, grc, reinterpret_cast<T*>(sd.out) + size_t{k} * BP_GROUP,
                          sm.lds[w], chunk_rows);
  }
}
template <typename T, class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_bitpacking(Src src, uint32_t gpw, uint32_t chunk_rows)
{
  __shared__ BpSmem sm;
  bp_block<T>(src.at(blockIdx.y), blockIdx.x, gpw, chunk_rows, sm);
}

template <bool RD>
struct AlpSmem {
  uint32_t lds[WAVES_PER_BLOCK][RD ? ALPRD_LEFT_WORDS + ALP_CHUNK_WORDS : ALP_CHUNK_WORDS];
};
template <typename T, bool RD>
__device__ __forceinline__ void alp_block(const FixedSeg& sd, uint32_t x, uint32_t vpw, AlpSmem<RD>& sm)
{
  const uint32_t w  = wave_in_block();
  const uint32_t nv = (sd.row_count + ALP_VEC - 1) / ALP_VEC;
  const uint32_t v0 = (x * WAVES_PER_BLOCK + w) * vpw;
  for (uint32_t v = v0; v < v0 + vpw && v < nv; ++v) {
    const uint32_t fill = sd.row_count - v * ALP_VEC < ALP_VEC ? sd.row_count - v * ALP_VEC : ALP_VEC;
    T* out = reinterpret_cast<T*>(sd.out) + size_t{v} * ALP_VEC;
    if constexpr (RD) alprd_vector<T>(sd.bytes, sd.bytes_size, v, fill, out, sm.lds[w]);
    else alp_vector<T>(sd.bytes, sd.bytes_size, v, fill, out, sm.lds[w]);
  }
}
template <typename T, bool RD, class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_alp(Src src, uint32_t vpw)
{
  __shared__ AlpSmem<RD> sm;
  alp_block<T, RD>(src.at(blockIdx.y), blockIdx.x, vpw, sm);
}

// One block per (segment, slice of `slice_rows` rows) over a 1-D grid of
// n_blocks (a multiple of 8).  Workgroups are dispatched to the 8 XCDs
// round-robin, so block b runs on XCD b % 8; the remap below hands each XCD
// a contiguous range of (segment, slice) pairs, so the slices of a segment
// share one L2 and its counts are fetched from HBM about once.
constexpr uint32_t N_XCD = 8;

// Block `block` of `blocks` (a multiple of 8, the first of them on an XCD 0).
template <uint32_t TS, class Src>
__device__ __forceinline__ void rle_block(const Src& src, uint32_t seg0, uint32_t n_segs, uint32_t block,
                                          uint32_t blocks, uint32_t slices, uint32_t slice_rows, RleSmem& sm)
{
  const uint32_t per_xcd = blocks / N_XCD;
  const uint32_t logical = (block % N_XCD) * per_xcd + block / N_XCD;
  const uint32_t sgi     = logical / slices;
  if (sgi >= n_segs) return;
  const FixedSeg sd = src.at(seg0 + sgi);
  const uint32_t ra = (logical % slices) * slice_rows;
  if (ra >= sd.row_count) return;
  const uint32_t rb = sd.row_count - ra < slice_rows ? sd.row_count : ra + slice_rows;
  rle_slice_t<TS>(sd.bytes, sd.bytes_size, sd.row_count, ra, rb, sd.out, sm);
}
template <uint32_t TS, class Src>
__global__ __launch_bounds__(RLE_THREADS) void k_rle(Src src, uint32_t n_segs, uint32_t slices, uint32_t slice_rows)
{
  __shared__ RleSmem sm;
  rle_block<TS>(src, 0, n_segs, blockIdx.x, gridDim.x, slices, slice_rows, sm);
}

// ===========================================================================
// UNCOMPRESSED copy and CONSTANT broadcast (thin paths; the reference's
// gpu_native_decode.cu:108-115 and :186-216).  A unit is 64 KiB of output:
// on a 256 MiB copy, 16 KiB units took 225 us, 64 KiB 186 us, 128 KiB 183 us
// and 256 KiB 311 us (too few blocks to fill the chip).
// ===========================================================================
constexpr uint32_t COPY_UNIT = 65536;

template <bool CONST>
__device__ __forceinline__ void copy_block(const FixedSeg& sd, uint32_t x, uint32_t type_size)
{
  const uint64_t total = uint64_t{sd.row_count} * type_size;
  const uint64_t b0    = uint64_t{x} * COPY_UNIT;
  if (b0 >= total) return;
  const uint64_t b1 = total - b0 < COPY_UNIT ? total : b0 + COPY_UNIT;
  if constexpr (CONST) const_span<BLOCK_THREADS>(sd.bytes, type_size, sd.out, b0, b1, threadIdx.x);
  else copy_span<BLOCK_THREADS>(sd.bytes, sd.out, b0, b1, threadIdx.x);
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_copy(Src src, uint32_t type_size)
{
  copy_block<false>(src.at(blockIdx.y), blockIdx.x, type_size);
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

// Null masks: a block copies one piece of a validity segment and counts its
// zero bits on the way.  A mask is a few bytes for thousands of rows, so the
// cost is launches and latency: one launch builds every mask of a call.  (A
// device copy per segment, then a count with one atomic per wave on one
// address, took 700 us beside a 57 us decode of 32 Mi nullable rows in 274
// segments, and 300 us beside 43 us for ten row groups of five columns.)
struct DevMasks {
  const MaskUnit* p;
  __device__ __forceinline__ MaskUnit at(uint32_t i) const { return uniform(gload(p + i)); }
};
struct MasksInline {
  MaskUnit unit[MASKS_INLINE];
  __device__ __forceinline__ MaskUnit at(uint32_t i) const { return uniform(unit[i]); }
};

struct MaskSmem {
  uint32_t wave_nulls[WAVES_PER_BLOCK];
};
__device__ __forceinline__ void mask_block(const MaskUnit& u, uint32_t index, uint32_t* __restrict__ counts,
                                           unsigned long long* __restrict__ total, MaskSmem& sm)
{
  const uint32_t t = threadIdx.x;
  const gptr<uint8_t> dst = gbl(u.dst);
  uint32_t nulls          = 0;
  if (!u.src) {
    // 16-byte blocks of all-valid rows between single bytes at the ends
    const uint32_t head = static_cast<uint32_t>(-reinterpret_cast<uintptr_t>(u.dst)) & 15u;
    const uint32_t h    = head < u.bytes ? head : u.bytes;
    const uint32_t nb   = (u.bytes - h) / 16u;
    if (t < h) dst[t] = 0xFFu;
    const gptr<u32x4> v = reinterpret_cast<gptr<u32x4>>(dst + h);
    for (uint32_t i = t; i < nb; i += BLOCK_THREADS) v[i] = u32x4{~0u, ~0u, ~0u, ~0u};
    const uint32_t e = h + nb * 16u + t;
    if (e < u.bytes && t < 16u) dst[e] = 0xFFu;
  } else {
    // four-byte words of the destination, the source's bytes whatever their
    // alignment (words holding requested bytes only); single bytes at the ends
    const uint32_t head = static_cast<uint32_t>(-reinterpret_cast<uintptr_t>(u.dst)) & 3u;
    const uint32_t h    = head < u.bytes ? head : u.bytes;
    const uint32_t nw   = (u.bytes - h) / 4u;
    const gptr<uint32_t> v = reinterpret_cast<gptr<uint32_t>>(dst + h);
    auto one               = [&](uint32_t i) {
      const uint32_t b = ld_u8(u.src + i);
      dst[i]           = static_cast<uint8_t>(b);
      nulls += 8u - static_cast<uint32_t>(__builtin_popcount(b));
    };
    if (t < h) one(t);
    constexpr uint32_t K = MASK_UNIT_BYTES / 4u / BLOCK_THREADS;  // a thread's words, loaded together
    uint32_t w[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t i = k * BLOCK_THREADS + t;
      w[k]             = i < nw ? ld_u32_any(u.src + h + 4u * i) : ~0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t i = k * BLOCK_THREADS + t;
      if (i < nw) v[i] = w[k];
      nulls += 32u - static_cast<uint32_t>(__builtin_popcount(w[k]));
    }
    const uint32_t e = h + nw * 4u + t;
    if (e < u.bytes && t < 4u) one(e);
    // bits past the column's rows are not rows
    if (t == 0 && u.past) nulls -= static_cast<uint32_t>(__builtin_popcount(~ld_u8(u.src + u.bytes - 1u) & u.past));
  }
  const uint32_t sum = wave_incl_sum_u32(nulls);
  if (lane_id() == WAVE - 1u) sm.wave_nulls[wave_in_block()] = sum;
  __syncthreads();
  if (t == 0) {
    uint32_t all = 0;
#pragma unroll
    for (uint32_t k = 0; k < WAVES_PER_BLOCK; ++k) all += sm.wave_nulls[k];
    if (counts) gbl(counts)[index] = all;
    else if (all) atomicAdd(total, static_cast<unsigned long long>(all));
  }
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) void k_null_mask(Src src, uint32_t* __restrict__ counts,
                                                             unsigned long long* __restrict__ total)
{
  __shared__ MaskSmem sm;
  mask_block(src.at(blockIdx.x), blockIdx.x, counts, total, sm);
}

// Every codec group of a call, and its null masks, in one launch.  The groups'
// kernels, one after another, each end in a tail of few blocks and begin with
// the latency of their first loads; a small call is nothing else: ten row groups
// of five nullable columns took 48 us for the call, now 30 us (one launch in place
// of five of 4 to 11 us); 10 M rows of six other widths 111 and 90 us; 16 Mi rows
// of ALP and ALP-RD 123 and 116 us; 32 Mi nullable rows 118 and 97 us.  Eight
// wavefronts a SIMD, as most of the codecs' own kernels.
//
// A group's blocks are consecutive and begin at a multiple of 8, so that a block
// runs on the XCD its number within the group says.
enum GroupKind : uint32_t {  // + log2 of the value width
  GK_BITPACKING = 0,
  GK_RLE        = 4,
  GK_ALP        = 8,
  GK_ALPRD      = 12,
  GK_COPY       = 16,
  GK_CONSTANT   = 17,
  GK_MASK       = 18,
};
struct Group {
  uint32_t first, blocks;  // its blocks of the launch
  uint32_t kind;
  uint32_t seg, n_segs;    // its descriptors (GK_MASK: the first of its counts)
  uint32_t per_seg;        // blocks of a segment
  uint32_t a, b;           // as the codec's own kernel takes them
};
constexpr uint32_t GROUPS_MAX = 19;
struct GroupTable {
  uint32_t n;
  const MaskUnit* units;  // mask pieces, or null: among the descriptors in the arguments
  uint32_t* counts;
  Group g[GROUPS_MAX];
};
__device__ __forceinline__ MaskUnit mask_unit(const SegsInline& src, const GroupTable& t, uint32_t i)
{
  if (t.units) return uniform(gload(t.units + i));
  const FixedSeg f = src.at(i);
  return MaskUnit{f.bytes, f.out, f.bytes_size, f.row_count};
}
__device__ __forceinline__ MaskUnit mask_unit(const DevSegs&, const GroupTable& t, uint32_t i)
{
  return uniform(gload(t.units + i));
}

template <class Src>
__global__ __launch_bounds__(BLOCK_THREADS) __attribute__((amdgpu_waves_per_eu(8))) void k_groups(Src src, GroupTable t)
{
  static_assert(BLOCK_THREADS == RLE_THREADS, "one workgroup size");
  __shared__ union Smem {
    BpSmem bp;
    AlpSmem<false> alp;
    AlpSmem<true> alprd;
    RleSmem rle;
    MaskSmem mask;
    __device__ Smem() {}
  } sm;
  uint32_t i = 0;
  while (i + 1u < t.n && blockIdx.x >= t.g[i + 1u].first) ++i;
  const Group g        = t.g[i];
  const uint32_t block = blockIdx.x - g.first;
  if (block >= g.blocks) return;  // between two groups
  if (g.kind - GK_RLE < 4u) {
    switch (g.kind - GK_RLE) {
      case 0: rle_block<1>(src, g.seg, g.n_segs, block, g.blocks, g.per_seg, g.a, sm.rle); break;
      case 1: rle_block<2>(src, g.seg, g.n_segs, block, g.blocks, g.per_seg, g.a, sm.rle); break;
      case 2: rle_block<4>(src, g.seg, g.n_segs, block, g.blocks, g.per_seg, g.a, sm.rle); break;
      default: rle_block<8>(src, g.seg, g.n_segs, block, g.blocks, g.per_seg, g.a, sm.rle); break;
    }
    return;
  }
  if (g.kind == GK_MASK) {
    mask_block(mask_unit(src, t, g.seg + block), g.a + block, t.counts, nullptr, sm.mask);
    return;
  }
  const uint32_t y  = block / g.per_seg, x = block - y * g.per_seg;
  const FixedSeg sd = src.at(g.seg + y);
  switch (g.kind) {
    case GK_BITPACKING + 0: bp_block<uint8_t>(sd, x, g.a, g.b, sm.bp); break;
    case GK_BITPACKING + 1: bp_block<uint16_t>(sd, x, g.a, g.b, sm.bp); break;
    case GK_BITPACKING + 2: bp_block<uint32_t>(sd, x, g.a, g.b, sm.bp); break;
    case GK_BITPACKING + 3: bp_block<uint64_t>(sd, x, g.a, g.b, sm.bp); break;
    case GK_ALP + 2: alp_block<float, false>(sd, x, g.a, sm.alp); break;
    case GK_ALP + 3: alp_block<double, false>(sd, x, g.a, sm.alp); break;
    case GK_ALPRD + 2: alp_block<float, true>(sd, x, g.a, sm.alprd); break;
    case GK_ALPRD + 3: alp_block<double, true>(sd, x, g.a, sm.alprd); break;
    case GK_COPY: copy_block<false>(sd, x, g.a); break;
    default: copy_block<true>(sd, x, g.a); break;
  }
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
  const uint32_t set = tune(SDR_TUNE_RLE_SLICE_ROWS, ts);
  if (set != RLE_SLICE_ROWS) return set;
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
  // segments per launch so that the 1-D grid stays below 2^31 blocks
  const uint32_t per = static_cast<uint32_t>(std::min<uint64_t>(MAX_GRID_Y, (0x7FFFFFF0ull / slices)));
  return for_segs(segs, seg_base, n, host, per, [&](auto src, uint32_t m) {
    using S = decltype(src);
    const uint64_t blocks = (uint64_t{m} * slices + N_XCD - 1) / N_XCD * N_XCD;
    const dim3 grid(static_cast<uint32_t>(blocks)), block(RLE_THREADS);
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
    if (ts == 8) {
      if (rd) hipLaunchKernelGGL((k_alp<double, true, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw);
      else hipLaunchKernelGGL((k_alp<double, false, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw);
    } else {
      if (rd) hipLaunchKernelGGL((k_alp<float, true, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw);
      else hipLaunchKernelGGL((k_alp<float, false, S>), g, dim3(BLOCK_THREADS), 0, s, src, vpw);
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
                       ts);
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
  if (f.codec == SDR_CODEC_RLE) blocks = (blocks + N_XCD - 1) / N_XCD * N_XCD;
  g.blocks = blocks < 0x7FFFFFF0u ? static_cast<uint32_t>(blocks) : 0u;  // 0: too many for a launch
  return g;
}

hipError_t launch_groups(const FixedGroup* groups, uint32_t n_groups, const FixedSeg* segs, const MaskUnit* units,
                         const MaskUnit* host_units, uint32_t* counts, hipStream_t s, bool host, bool* done)
{
  *done = false;
  if (n_groups < 2u || n_groups > GROUPS_MAX) return hipSuccess;
  // mask pieces travel with the descriptors if one launch holds all
  uint64_t total = 0;
  for (uint32_t i = 0; i < n_groups; ++i) total += groups[i].count;
  const bool carry = host && host_units && total <= SEGS_INLINE;
  // pieces of at most a launch's descriptors, all of them in device memory
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
    if (host) inl.push_back(si);
    t      = GroupTable{};
    blocks = 0;
    held   = 0;
  };
  for (uint32_t i = 0; i < n_groups; ++i) {
    const FixedGroup& f = groups[i];
    for (uint32_t b = 0; b < f.count;) {
      const bool here = host && (f.codec != MASK_GROUP || carry);
      if (here && held == SEGS_INLINE) flush();
      const uint32_t n = here ? std::min(f.count - b, SEGS_INLINE - held) : f.count;
      Group g          = group_of(f, n);
      if (g.blocks == 0 || (t.n && blocks + g.blocks + N_XCD > 0x7FFFFFF0ull)) return hipSuccess;
      g.first = static_cast<uint32_t>(blocks);
      if (f.codec == MASK_GROUP) g.a = b;
      if (here) {
        g.seg = held;
        if (f.codec == MASK_GROUP) std::memcpy(si.seg + held, host_units + b, size_t{n} * sizeof(MaskUnit));
        else std::memcpy(si.seg + held, segs + f.first + b, size_t{n} * sizeof(FixedSeg));
      } else {
        g.seg = f.codec == MASK_GROUP ? 0u : f.first;
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
    if (host) hipLaunchKernelGGL((k_groups<SegsInline>), grid, dim3(BLOCK_THREADS), 0, s, inl[i], gt);
    else hipLaunchKernelGGL((k_groups<DevSegs>), grid, dim3(BLOCK_THREADS), 0, s, DevSegs{segs, 0}, gt);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace sdr
