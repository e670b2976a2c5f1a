// dec_groups.hpp — a workgroup of each fixed-width codec and of the null masks,
// and of a launch that holds several of them.  Used by the codecs' own kernels
// and the fused one (k_fixed.hip) and by a mixed batch's first kernel
// (k_batch.hip).
#pragma once

#include "dec_fixed.hpp"
#include "dec_rle.hpp"
#include "sdr_kernels.hpp"

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
  __device__ __forceinline__ FixedSeg at(uint32_t i) const { return sload(p + base + i); }
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

// Workgroups are dispatched to the 8 XCDs round-robin, each with an L2 and address
// translations of its own.  The block of a grid of `blocks` that the `block`-th
// workgroup takes, so that an XCD takes `run` in a row and the next XCD the next
// `run`; what is left after whole turns of all XCDs is taken in plain order.
constexpr uint32_t N_XCD = 8;
__device__ __forceinline__ uint32_t xcd_order(uint32_t block, uint32_t blocks, uint32_t run)
{
  const uint32_t in_turn = block % (N_XCD * run), turn = block - in_turn;
  return turn + N_XCD * run <= blocks ? turn + in_turn % N_XCD * run + in_turn / N_XCD : block;
}

// One block per (segment, slice of `slice_rows` rows) over a 1-D grid.  Every
// slice reads all of its segment's counts, so an XCD takes eight in a row, half a
// row group, and the chip writes within 4 MiB at a time.  An eighth of the whole
// launch to each XCD, as it was, reads the counts once but writes eight places far
// apart, and memory takes that less well (32 Mi int64 rows in runs of 64: 56.0 us,
// so 54.0; runs of 16: 65.0, 62.6; runs of 2, whose counts are as much as a quarter
// of what is moved: 180.1, 181.0; int32 in runs of 300: 32.9, 31.6, of 2: 194.5,
// 197.0; 64 Mi integers and dates 230.9, 227.5).
constexpr uint32_t RLE_XCD_RUN = 8;

// Block `block` of `blocks`, the first of them on an XCD 0.
template <uint32_t TS, class Src>
__device__ __forceinline__ void rle_block(const Src& src, uint32_t seg0, uint32_t n_segs, uint32_t block,
                                          uint32_t blocks, uint32_t slices, uint32_t slice_rows, RleSmem& sm)
{
  const uint32_t logical = xcd_order(block, blocks, RLE_XCD_RUN);
  const uint32_t sgi     = logical / slices;
  if (sgi >= n_segs) return;
  const FixedSeg sd = src.at(seg0 + sgi);
  const uint32_t ra = (logical % slices) * slice_rows;
  if (ra >= sd.row_count) return;
  const uint32_t rb = sd.row_count - ra < slice_rows ? sd.row_count : ra + slice_rows;
  rle_slice_t<TS>(sd.bytes, sd.bytes_size, sd.row_count, ra, rb, sd.out, sm);
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

// Null masks: a block copies one piece of a validity segment and counts its
// zero bits on the way.  A mask is a few bytes for thousands of rows, so the
// cost is launches and latency: one launch builds every mask of a call.  (A
// device copy per segment, then a count with one atomic per wave on one
// address, took 700 us beside a 57 us decode of 32 Mi nullable rows in 274
// segments, and 300 us beside 43 us for ten row groups of five columns.)
struct DevMasks {
  const MaskUnit* p;
  __device__ __forceinline__ MaskUnit at(uint32_t i) const { return sload(p + i); }
};
struct MasksInline {
  MaskUnit unit[MASKS_INLINE];
  __device__ __forceinline__ MaskUnit at(uint32_t i) const { return uniform(unit[i]); }
};

template <uint32_t NT = BLOCK_THREADS>
struct MaskSmem {
  uint32_t wave_nulls[NT / WAVE];
};
template <uint32_t NT>
__device__ __forceinline__ void mask_block(const MaskUnit& u, uint32_t index, uint32_t* __restrict__ counts,
                                           unsigned long long* __restrict__ total, MaskSmem<NT>& sm)
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
    for (uint32_t i = t; i < nb; i += NT) v[i] = u32x4{~0u, ~0u, ~0u, ~0u};
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
    constexpr uint32_t K = MASK_UNIT_BYTES / 4u / NT;  // a thread's words, loaded together
    uint32_t w[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t i = k * NT + t;
      w[k]             = i < nw ? ld_u32_any(u.src + h + 4u * i) : ~0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t i = k * NT + t;
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
    for (uint32_t k = 0; k < NT / WAVE; ++k) all += sm.wave_nulls[k];
    if (counts) gbl(counts)[index] = all;
    else if (all) atomicAdd(total, static_cast<unsigned long long>(all));
  }
}


// Every codec group of a call, and its null masks, in one launch.  The groups'
// kernels, one after another, each end in a tail of few blocks and begin with
// the latency of their first loads; a small call is nothing else: ten row groups
// of five nullable columns took 48 us for the call, now 30 us (one launch in place
// of five of 4 to 11 us); 10 M rows of six other widths 111 and 78 us; 16 Mi rows
// of ALP and ALP-RD 123 and 112 us; 32 Mi nullable rows 118 and 97 us.  Eight
// wavefronts a SIMD, as most of the codecs' own kernels.
//
// A group's blocks are consecutive and begin at a multiple of 8, so that a block
// runs on the XCD its number within the group says.  An XCD takes 32 of them in a
// row, so that it translates the addresses of an eighth of the pages that are in
// use (in plain order, and 32 in a row: 16 Mi rows of ALP and ALP-RD 107.4 and
// 104.6 us, 64 Mi integers and dates 227.8 and 226.0, 10 M rows of six widths 76.2
// and 75.0; 8 in a row 105.6, 228.4, 75.5; 128 in a row 104.5, 230.0, 76.9).
constexpr uint32_t GROUP_XCD_RUN = 32;
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
// Workgroups along a dimension of a grid: a launch of 2^32 threads or more along one
// reports no error and starts what is left of that modulo 2^32.
constexpr uint32_t MAX_BLOCKS = 0xFFFFFFFFu / BLOCK_THREADS;
constexpr uint32_t GROUPS_MAX = 24;  // 22 pairs of codec and width, and the masks
struct GroupTable {
  uint32_t n;
  const MaskUnit* units;  // mask pieces, or null: among the descriptors in the arguments
  uint32_t* counts;
  Group g[GROUPS_MAX];
};
__device__ __forceinline__ MaskUnit mask_unit(const SegsInline& src, const GroupTable& t, uint32_t i)
{
  if (t.units) return sload(t.units + i);
  const FixedSeg f = src.at(i);
  return MaskUnit{f.bytes, f.out, f.bytes_size, f.row_count};
}
__device__ __forceinline__ MaskUnit mask_unit(const DevSegs&, const GroupTable& t, uint32_t i)
{
  return sload(t.units + i);
}

union GroupSmem {
  BpSmem bp;
  AlpSmem<false> alp;
  AlpSmem<true> alprd;
  RleSmem rle;
  MaskSmem<> mask;
  __device__ GroupSmem() {}
};

template <class Src>
__device__ __forceinline__ void groups_block(const Src& src, const GroupTable& t, uint32_t at, GroupSmem& sm)
{
  static_assert(BLOCK_THREADS == RLE_THREADS, "one workgroup size");
  uint32_t i = 0;
  while (i + 1u < t.n && at >= t.g[i + 1u].first) ++i;
  const Group g        = t.g[i];
  const uint32_t block = at - g.first;
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
  const uint32_t b  = xcd_order(block, g.blocks, GROUP_XCD_RUN);
  const uint32_t y  = b / g.per_seg, x = b - y * g.per_seg;
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

// The table of a launch over descriptors and mask pieces in device memory, and
// its blocks; false if it would take too many groups or blocks.
bool device_groups(const FixedGroup* groups, uint32_t n_groups, const MaskUnit* units, uint32_t* counts, GroupTable* t,
                   uint32_t* blocks);

}  // namespace sdr
