// dec_fsst.hpp — gfx950 FSST chunk decoder: VARCHAR segments to int32
// offsets + chars.  Used by the per-column kernel (k_fsst.hip) and the
// persistent mixed-codec kernel (k_batch.hip).
//
// Segment layout, header checks and symbol-table format: the reference's
// src/cuda/scan/strings/fsst.cu:17-44, :69-87 and
// src/include/cuda/scan/detail/fsst.cuh:50-96 (a device port of DuckDB's
// duckdb_fsst_import).  Decoded lengths and bytes follow DuckDB's serial
// decompressor: a code emits its symbol, an escape (255) emits the next byte
// literally, a trailing escape is dropped (fsst.cu:273-281).
//
// One 512-thread workgroup decodes one chunk of up to FSST_CHUNK_ROWS rows.
// Chunks are numbered in column row order and taken in that order (by workgroup
// number or by ticket, see FSST_UNORDERED_SHARE): each chunk publishes its
// decoded byte count, looks back over its predecessors for the column-wide
// exclusive prefix (a decoupled look-back), writes its rows' int32 offsets
// and then its chars.
//
// A chunk's compressed bytes are one contiguous range (rows are stored back
// to front), cut on a 16-byte grid into groups that are spread over the
// threads whatever rows they cut, and held in registers between two walks.
// The first walk looks up the decoded length of every byte and leaves, per
// group, their prefix sums (packed bytes) and, per row, the prefix at the
// row's first byte; the second ORs every symbol into a zeroed LDS copy of the
// chunk's output, which leaves in 16-byte stores.  Neither walk follows rows
// byte by byte: a bitmap holds the row starts, and a byte's row is the
// population count of the bits up to it.  Chunks whose compressed bytes do
// not fit the registers and malformed ones take a row-per-thread path that
// reads global memory.
#pragma once

#include "sdr_device.hpp"
#include "sdr_fsst.hpp"

#include <cstddef>

namespace sdr {

constexpr uint32_t FSST_THREADS   = 512;  // a chunk's workgroup
constexpr uint32_t FSST_WAVES     = FSST_THREADS / WAVE;
constexpr uint32_t ROWS_PER_THR   = FSST_CHUNK_ROWS / FSST_THREADS;
constexpr uint32_t FSST_PIECE     = 8192;  // LDS output piece of the row-wise path
constexpr uint32_t FSST_ESC       = 255;
constexpr uint32_t FSST_NSYM      = 255;
constexpr uint64_t FSST_VERSION   = 20190218ull;
constexpr uint64_t FSST_CORRUPT   = 32774747032022883ull;  // "corrupt\0"
constexpr uint32_t SYMTAB_MAX     = 8192;
constexpr uint64_t ST_AGG         = 1ull << 62;  // aggregate published
constexpr uint64_t ST_INC         = 2ull << 62;  // inclusive prefix published
constexpr uint64_t ST_RUN         = 3ull << 62;  // a long chunk, begun: nothing published yet
constexpr uint64_t ST_VAL         = (1ull << 62) - 1;

// Bytes of a segment read in order through aligned words; bytes at or past
// `end` read as zero.
__device__ __forceinline__ uint32_t byte_at(const uint8_t* p, const uint8_t* end)
{
  if (p >= end) return 0;
  return *gbl(p);
}

// w-bit value at bit `bitpos` of the stream starting at `base`; bytes at or
// past `end` read as zero (only malformed segments reach them).
__device__ __forceinline__ uint32_t stream_bits32(const uint8_t* base, const uint8_t* end, uint64_t bitpos,
                                                  uint32_t w)
{
  if (w == 0) return 0;
  const uint8_t* p   = base + (bitpos >> 3);
  const uint32_t off = static_cast<uint32_t>(bitpos & 7u);
  const uint32_t nb  = (off + w + 7u) >> 3;  // bytes spanned, <= 5
  uint64_t v = 0;
  if (p + nb <= end) {
    uintptr_t a = reinterpret_cast<uintptr_t>(p);
    const uint32_t sh = static_cast<uint32_t>(a & 3u);
    const gptr<const uint32_t> wp = gbl(reinterpret_cast<const uint32_t*>(a - sh));
    const uint32_t need = (sh + nb + 3u) >> 2;  // words spanned, <= 3
    uint32_t w0 = wp[0], w1 = need > 1 ? wp[1] : 0u, w2 = need > 2 ? wp[2] : 0u;
    const uint64_t lo = static_cast<uint64_t>(w0) | (static_cast<uint64_t>(w1) << 32);
    v = (lo >> (8u * sh)) | (sh ? (static_cast<uint64_t>(w2) << (64u - 8u * sh)) : 0ull);
  } else {
    for (uint32_t b = 0; b < nb; ++b) v |= static_cast<uint64_t>(byte_at(p + b, end)) << (8u * b);
  }
  v >>= off;
  return static_cast<uint32_t>(w >= 32u ? v : (v & ((1ull << w) - 1ull)));
}

// Sequential reader of w-bit fields (w <= 32) from an LSB-first stream,
// loading each aligned word only when its bits are needed.
struct BitCursor {
  gptr<const uint32_t> w;
  uint64_t acc;
  uint32_t nbits;
  __device__ __forceinline__ BitCursor(const uint8_t* base, uint64_t bitpos)
  {
    uintptr_t a = reinterpret_cast<uintptr_t>(base + (bitpos >> 3));
    const uint32_t skip = static_cast<uint32_t>((a & 3u) * 8u + (bitpos & 7u));
    w     = gbl(reinterpret_cast<const uint32_t*>(a & ~uintptr_t{3}));
    acc   = static_cast<uint64_t>(*w++) >> skip;
    nbits = 32u - skip;
  }
  __device__ __forceinline__ uint32_t next(uint32_t wd)
  {
    if (nbits < wd) {
      acc |= static_cast<uint64_t>(*w++) << nbits;
      nbits += 32u;
    }
    const uint32_t v = static_cast<uint32_t>(wd >= 32u ? acc : (acc & ((1ull << wd) - 1ull)));
    acc >>= wd;
    nbits -= wd;
    return v;
  }
};

// Sequential byte reader over global bytes [p, p + n) using aligned 4-byte loads.
struct ByteReader {
  gptr<const uint32_t> w;
  uint32_t cur;
  uint32_t boff;
  __device__ __forceinline__ explicit ByteReader(const uint8_t* p)
  {
    boff = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3u);
    w    = gbl(reinterpret_cast<const uint32_t*>(p - boff));
    cur  = *w;
  }
  __device__ __forceinline__ uint32_t next()
  {
    if (boff == 4u) {
      cur  = *++w;
      boff = 0;
    }
    return (cur >> (8u * boff++)) & 0xFFu;
  }
};

// A workgroup barrier for LDS alone: each wave's LDS operations complete
// first, global loads stay in flight.  (__syncthreads() also waits for every
// pending load while the compiler tracks LDS-direct loads, which it cannot
// tell apart from register loads.)
__device__ __forceinline__ void lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Block-wide exclusive scan of one value per thread (NW wavefronts); returns
// the exclusive prefix and writes the block total to *total.
template <uint32_t NW = FSST_WAVES>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_wave, uint32_t* total)
{
  const uint32_t incl = wave_incl_sum_u32(v);
  const uint32_t w    = threadIdx.x >> 6;
  if (lane_id() == 63) s_wave[w] = incl;
  __syncthreads();
  uint32_t before = 0, tot = 0;
#pragma unroll
  for (uint32_t k = 0; k < NW; ++k) {
    const uint32_t x = s_wave[k];
    before += k < w ? x : 0u;
    tot += x;
  }
  __syncthreads();
  *total = tot;
  return before + incl - v;
}

// Exclusive scan of one value per thread with one barrier, for LDS alone
// (global loads stay in flight); s_wave must not be written again before the
// caller's next barrier.
__device__ __forceinline__ uint32_t block_excl_scan_lds(uint32_t v, uint32_t* s_wave, uint32_t* total)
{
  static_assert(FSST_WAVES <= 16, "one DPP row of wave sums");
  const uint32_t incl = wave_incl_sum_u32(v);
  const uint32_t w    = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
  if (lane_id() == WAVE - 1u) s_wave[w] = incl;
  lds_barrier();
  const uint32_t ws = s_wave[lane_id() & (FSST_WAVES - 1u)];  // every wave scans the wave sums
  const uint32_t wi = row_incl_sum_u32(ws);
  *total            = __builtin_amdgcn_readlane(wi, FSST_WAVES - 1u);
  return __builtin_amdgcn_readlane(wi, w) - __builtin_amdgcn_readlane(ws, w) + incl - v;
}

// Exclusive scans of two values per thread with one barrier, for LDS alone
// (global loads stay in flight); s_wave[2 * FSST_WAVES] must not be written
// again before the caller's next barrier.
__device__ __forceinline__ void block_excl_scan2(uint32_t a, uint32_t b, uint32_t* s_wave, uint32_t& pre_a,
                                                 uint32_t& pre_b, uint32_t& tot_a, uint32_t& tot_b)
{
  static_assert(FSST_WAVES == 8, "both values' wave sums fill one 16-lane DPP row");
  const uint32_t ia = wave_incl_sum_u32(a), ib = wave_incl_sum_u32(b);
  const uint32_t w  = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)));
  if (lane_id() == WAVE - 1u) {
    s_wave[w]              = ia;
    s_wave[FSST_WAVES + w] = ib;
  }
  lds_barrier();
  // every wave scans the wave sums, the second value's on top of the first's
  const uint32_t ws = s_wave[lane_id() & (2u * FSST_WAVES - 1u)];
  const uint32_t wi = row_incl_sum_u32(ws);
  tot_a             = __builtin_amdgcn_readlane(wi, FSST_WAVES - 1u);
  tot_b             = __builtin_amdgcn_readlane(wi, 2u * FSST_WAVES - 1u) - tot_a;
  pre_a = __builtin_amdgcn_readlane(wi, w) - __builtin_amdgcn_readlane(ws, w) + ia - a;
  pre_b = __builtin_amdgcn_readlane(wi, FSST_WAVES + w) - __builtin_amdgcn_readlane(ws, FSST_WAVES + w) - tot_a + ib - b;
}

// Shape of a chunk decode, and why.  The decode is bound by the instructions
// that every compressed byte costs (VALU, at one wave instruction per cycle and
// CU, and LDS: 4-7 cycles for each lookup or OR of 64 lanes at random
// addresses), not by HBM.  The form before this one walked rows byte by byte
// in 256-thread workgroups with an 11 KiB window: 70 VALU and 52 LDS cycles
// per 64 bytes, 560 us for 16 Mi rows of 27 chars (12.9 compressed).  Row
// starts as a bitmap, packed prefix sums and two lookups and two to three ORs
// per byte take it to 32 VALU and 31 LDS cycles, both busy 60% of the time, and
// 272 us (293 us when chunks were taken by ticket, see FSST_UNORDERED_SHARE).
// 512 threads with two groups each keep a 16 KiB run in registers, so nothing is
// read twice; three such workgroups share a CU (51 KB of LDS, 80 VGPRs), whose
// 38 KiB window builds most chunks in one piece.  Rows of 70 and 200 chars,
// whose chunks take several runs, went from 945 to 221 and from 2956 to 324 us
// (137 and 197 MB of chars); the row-wise path is left to malformed chunks and to
// rows that no run holds.
constexpr uint32_t FSST_SYMSTAGE = 17u + 8u * FSST_NSYM;  // the largest symbol table (2057 bytes)
// Compressed bytes that the staged path takes at a time, the head of up to
// 15 bytes before them included: GROUPS_PER_THR 16-byte groups per thread.
constexpr uint32_t FSST_CSTAGE    = 16384;
constexpr uint32_t GROUPS_PER_THR = FSST_CSTAGE / (16u * FSST_THREADS);
static_assert(GROUPS_PER_THR == 2, "the staged path's registers and its packed scans");
// Output window: at most this many chars are built in LDS at a time.
constexpr uint32_t FSST_WINDOW = 38u << 10;
// What a chunk without compressed bytes loads as its groups (never used).
static __device__ __attribute__((aligned(16))) const uint32_t fsst_zero_group[4] = {0u, 0u, 0u, 0u};

constexpr uint32_t ROW_HUGE = 1u << 20;  // a staged row is shorter than this
// Packed prefixes: decoded bytes (at most 8 * FSST_CSTAGE, bits 0-17) or a
// run's compressed bytes, with a count of at most 1024 rows above.
constexpr uint32_t PK_LEN = 18;
// len[] of the escape code in a staged chunk's table, so that the lengths a
// group looks up tell whether it holds an escape.
constexpr uint32_t LEN_ESC = 0x80;

struct FsstSmem {
  // the segment's FsstSymTab, staged whole
  __attribute__((aligned(16))) uint64_t sym[256];  // symbol bytes, zero above its length
  uint8_t len[256];
  // row-wise path: comp[] is the segment-relative inclusive compressed prefix,
  // dec[] the chunk-relative exclusive decoded offset.  Staged path: comp[g] is
  // the decoded prefix at group g's first byte; of the rows with compressed
  // bytes in storage order (rank), dec[k + 1] is what takes a decoded prefix
  // inside row k to its output position.
  uint32_t comp[FSST_CHUNK_ROWS + 1];
  uint32_t dec[FSST_CHUNK_ROWS + 4];
  uint32_t bits[FSST_CSTAGE / 32];  // bit y: a row's first byte is stage position y
  // output window (and the slack its last symbol's words reach); before that,
  // the compressed-length fields, then the groups' packed prefixes (byte y:
  // decoded bytes of stage position y's group before it)
  __attribute__((aligned(16))) uint8_t out[FSST_WINDOW + 48];
  uint32_t wave[2 * FSST_WAVES];
  uint32_t part[2 * FSST_WAVES];
  uint64_t base;
  __device__ __forceinline__ uint32_t* plain_part() { return comp; }
  __device__ __forceinline__ uint64_t* plain_sum() { return sym; }
};

// Walk the n compressed bytes of one row with DuckDB's serial semantics:
// emit(byte) for a literal after an escape, sym(code) for a symbol; a
// trailing escape emits nothing.  `fetch(i)` returns byte i of the row.
template <typename Fetch, typename Lit, typename Sym>
__device__ __forceinline__ void fsst_walk(uint32_t n, Fetch fetch, Lit lit, Sym sym)
{
  bool esc = false;
  for (uint32_t i = 0; i < n; ++i) {
    const uint32_t b = fetch(i);
    if (esc) {
      if (!lit(b)) return;
      esc = false;
    } else if (b == FSST_ESC) {
      esc = true;
    } else if (!sym(b)) {
      return;
    }
  }
}

// Decoded length of the n compressed bytes of one row at p (global memory),
// read a word at a time (only the aligned words holding the row).
template <class SM>
__device__ __forceinline__ uint32_t fsst_row_len(const uint8_t* p, uint32_t n, const SM& sm)
{
  const uint32_t boff = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3u);
  const gptr<const uint32_t> w = gbl(reinterpret_cast<const uint32_t*>(p - boff));
  const uint32_t end  = boff + n;
  bool esc            = false;
  uint32_t d          = 0;
  for (uint32_t q = 0; q * 4u < end; ++q) {
    const uint32_t word = w[q];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t idx = q * 4u + j;
      const uint32_t b   = (word >> (8u * j)) & 0xFFu;
      if (idx >= boff && idx < end) {
        d += esc ? 1u : sm.len[b];  // len[255] == 0: an escape emits nothing
        esc = !esc && b == FSST_ESC;
      }
    }
  }
  return d;
}

// ---- row-per-thread path (unstaged or malformed chunks) ----

// dec[] and the decoded total of a chunk, one row per thread at a time,
// reading the compressed bytes from global memory.  Rows whose compressed
// range leaves [0, dict_end) decode to nothing.
template <class SM>
__device__ __attribute__((noinline)) uint32_t fsst_lengths_rows(SM& sm, const uint8_t* seg,
                                                                uint32_t dict_end, uint32_t rows)
{
  uint32_t T = 0;
#pragma unroll 1
  for (uint32_t k = 0; k < ROWS_PER_THR; ++k) {
    const uint32_t r = k * FSST_THREADS + threadIdx.x;
    uint32_t d       = 0;
    if (r < rows) {
      const uint32_t cum = sm.comp[r + 1], prev = sm.comp[r];
      if (cum <= dict_end && prev <= cum && cum != prev) d = fsst_row_len(seg + dict_end - cum, cum - prev, sm);
    }
    uint32_t tot      = 0;
    const uint32_t ex = block_excl_scan(d, sm.wave, &tot);
    if (r < rows) sm.dec[r] = T + ex;
    T += tot;
  }
  if (threadIdx.x == 0) sm.dec[rows] = T;
  __syncthreads();
  return T;
}

// Chars of a chunk from dec[], one row per thread, in 8 KiB LDS pieces
// aligned to the absolute chars address: whole 16-byte blocks leave with
// vector stores, the partial first/last blocks byte-wise (they share 16
// bytes with the neighbours).
template <class SM>
__device__ __attribute__((noinline)) void fsst_emit_rows(SM& sm, const uint8_t* seg, uint32_t dict_end,
                                                        uint32_t rows, uint32_t T, uint64_t base, uint8_t* chars,
                                                        uint64_t chars_cap)
{
  const uint32_t tid = threadIdx.x;
  const uintptr_t cb = reinterpret_cast<uintptr_t>(chars);
  const uintptr_t g0 = cb + base;
  const uintptr_t g1 = cb + ((base + T < chars_cap) ? base + T : chars_cap);
  constexpr int32_t PIECE = static_cast<int32_t>(FSST_PIECE);
  for (uintptr_t pa = g0 & ~uintptr_t{15}; pa < g1; pa += FSST_PIECE) {
    const uintptr_t pb = pa + FSST_PIECE;
#pragma unroll 1
    for (uint32_t k = 0; k < ROWS_PER_THR; ++k) {
      const uint32_t r = k * FSST_THREADS + tid;
      if (r >= rows) continue;
      const uint32_t d0 = sm.dec[r], dl = sm.dec[r + 1] - d0;
      const uintptr_t o0 = g0 + d0;
      if (dl == 0 || o0 + dl <= pa || o0 >= pb) continue;
      const uint32_t cum = sm.comp[r + 1], prev = sm.comp[r];
      int32_t o = static_cast<int32_t>(static_cast<intptr_t>(o0 - pa));  // may start before the piece
      auto put = [&](uint64_t v, uint32_t l) {
        for (uint32_t j = 0; j < l; ++j, ++o)
          if (o >= 0 && o < PIECE) sm.out[o] = static_cast<uint8_t>(v >> (8u * j));
        return o < PIECE;
      };
      ByteReader br(seg + dict_end - cum);
      fsst_walk(cum - prev, [&](uint32_t) -> uint32_t { return br.next(); },
                [&](uint32_t b) { return put(b, 1u); }, [&](uint32_t b) { return put(sm.sym[b], sm.len[b]); });
    }
    __syncthreads();
    const uintptr_t lo = pa > g0 ? pa : g0;
    const uintptr_t hi = pb < g1 ? pb : g1;
    for (uintptr_t blk = pa + uintptr_t{tid} * 16u; blk < hi; blk += uintptr_t{FSST_THREADS} * 16u) {
      if (blk >= lo && blk + 16u <= hi) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(&sm.out[blk - pa]);
        __builtin_nontemporal_store(v, gbl(reinterpret_cast<u32x4*>(blk)));
      } else {
        for (uintptr_t x = blk; x < blk + 16u; ++x)
          if (x >= lo && x < hi) *gbl(reinterpret_cast<uint8_t*>(x)) = sm.out[x - pa];
      }
    }
    __syncthreads();
  }
}

// ---- staged path ----
//
// A chunk's rows are taken whole, as many at a time as their compressed bytes
// fit FSST_CSTAGE (a run of rows; nearly always the whole chunk).  Stage
// coordinates: the run's bytes are stage positions [c_h, y_hi), position 0
// being the 16-byte-aligned address at or below the first of them.  Rows are
// stored back to front, so row indices fall as the position rises; the rows
// that have bytes are ranked in that order.

// One thread's 16-byte group between the two walks.
struct FsstGroup {
  uint32_t q[4];  // the bytes
  uint32_t p[4];      // decoded bytes of the group before each byte, packed like q
  uint32_t m;     // bit j: a row starts at byte j
  uint32_t lit;   // bit j: byte j is a literal (it follows an escape)
  uint32_t d;     // decoded bytes of the run before the group
  uint32_t r;     // rows that start before the group
};

// Byte j (0..15) of a 16-byte group.
__device__ __forceinline__ uint32_t group_byte(const uint32_t (&q)[4], uint32_t j)
{
  return (q[j >> 2] >> (8u * (j & 3u))) & 0xFFu;
}

// 0x01 in byte i for each bit i (0..3) of x.
__device__ __forceinline__ uint32_t spread4(uint32_t x) { return ((x & 15u) * 0x00204081u) & 0x01010101u; }

// The literals of a group: a byte follows an escape of its own row.  e: the
// bytes equal to 255, m: the row starts, esc: an escape ends just before the
// group.
__device__ __forceinline__ uint32_t literal_mask(uint32_t e, uint32_t m, bool esc)
{
  uint32_t lit = 0;
#pragma unroll 1
  for (uint32_t j = 0; j < 16; ++j) {
    const uint32_t b = 1u << j;
    esc              = esc && !(m & b);
    lit |= esc ? b : 0u;
    esc = !esc && (e & b);
  }
  return lit;
}

// The groups of a run whose last byte is stage position y_hi - 1, and the
// word before each wave's first one: 2 * GROUPS_PER_THR loads per thread, with
// no branch around them (a group past the run's bytes rereads the last one).
__device__ __forceinline__ void fsst_load_groups(FsstGroup (&gr)[GROUPS_PER_THR], uint32_t (&prev)[GROUPS_PER_THR],
                                                 const uint8_t* stage, uint32_t y_hi)
{
  const gptr<const u32x4> cg    = gbl(reinterpret_cast<const u32x4*>(stage));
  const gptr<const uint32_t> cw = gbl(reinterpret_cast<const uint32_t*>(stage));
  const uint32_t last           = y_hi ? (y_hi - 1u) >> 4 : 0u;
#pragma unroll
  for (uint32_t k = 0; k < GROUPS_PER_THR; ++k) {
    const uint32_t g  = k * FSST_THREADS + threadIdx.x;
    const uint32_t wg = k * FSST_THREADS + (threadIdx.x & ~(WAVE - 1u));
    const u32x4 q     = cg[g < last ? g : last];
#pragma unroll
    for (uint32_t d = 0; d < 4; ++d) gr[k].q[d] = q[d];
    prev[k] = cw[wg && wg <= last ? 4u * wg - 1u : 0u];
  }
}

// First walk of group g: every byte's decoded length, summed.  `prev` is the
// word before the group.  Bytes that are not the run's become escapes, whose
// symbol is empty.  Returns the group's decoded bytes; *lits is wave-uniform:
// some group of the wave holds a literal.
__device__ __forceinline__ uint32_t fsst_group_lengths(FsstGroup& gr, const FsstSmem& sm, uint32_t g, uint32_t prev,
                                                       uint32_t c_h, uint32_t y_hi, const uint8_t* stage, bool* lits)
{
  const bool live = 16u * g < y_hi;
  uint32_t L[4];
#pragma unroll
  for (uint32_t d = 0; d < 4; ++d) {
    const uint32_t w = gr.q[d];
    L[d] = sm.len[w & 0xFFu] | static_cast<uint32_t>(sm.len[(w >> 8) & 0xFFu]) << 8 |
           static_cast<uint32_t>(sm.len[(w >> 16) & 0xFFu]) << 16 | static_cast<uint32_t>(sm.len[w >> 24]) << 24;
  }
  gr.m               = live ? (sm.bits[g >> 1] >> (16u * (g & 1u))) & 0xFFFFu : 0u;
  gr.lit             = 0;
  const uint32_t y   = 16u * g;
  const bool has_esc = live && ((L[0] | L[1] | L[2] | L[3]) & 0x80808080u) != 0;
  const bool after   = live && (prev >> 24) == FSST_ESC && y > c_h;
  *lits              = false;
  uint32_t valid     = 0xFFFFu;  // the bytes that are the run's
  if (ballot(live && (y < c_h || y + 16u > y_hi)) != 0) {
    const uint32_t lo = c_h > y ? c_h - y : 0u;  // c_h < 16
    const uint32_t hi = live ? (y_hi - y < 16u ? y_hi - y : 16u) : lo;
    valid             = ((1u << hi) - 1u) & ~((1u << lo) - 1u);
#pragma unroll
    for (uint32_t d = 0; d < 4; ++d) {
      const uint32_t in = spread4(valid >> (4u * d)) * 0xFFu;
      L[d] &= in;
      gr.q[d] |= ~in;
    }
  }
  if (ballot(has_esc || after) != 0) {
    uint32_t e = 0;
#pragma unroll
    for (uint32_t j = 0; j < 16; ++j) e |= group_byte(gr.q, j) == FSST_ESC ? 1u << j : 0u;
    e &= valid;
    bool esc = false;  // an odd run of 255s of the row ends just before the group
    if (after && !(gr.m & 1u)) {
      for (uint32_t x = y; x > c_h; --x) {
        if (ld_u8(stage + x - 1u) != FSST_ESC) break;
        esc = !esc;
        if ((sm.bits[(x - 1u) >> 5] >> ((x - 1u) & 31u)) & 1u) break;  // the row's first byte
      }
    }
    gr.lit = live ? literal_mask(e, gr.m, esc) & valid : 0u;
#pragma unroll
    for (uint32_t d = 0; d < 4; ++d) {
      const uint32_t one = spread4(gr.lit >> (4u * d));
      L[d]               = (L[d] & 0x7F7F7F7Fu & ~(one * 0xFFu)) | one;
    }
    *lits = ballot(gr.lit != 0) != 0;
  }
  // exclusive prefixes of the 16 lengths, four to a word (at most 128 in all)
  uint32_t t = 0;  // the running total in every byte
#pragma unroll
  for (uint32_t d = 0; d < 4; ++d) {
    const uint32_t s2 = (L[d] << 8) + L[d], s = (s2 << 16) + s2;  // inclusive within the word
    gr.p[d]           = (s << 8) + t;
    t                 = __builtin_amdgcn_perm(0u, s + t, 0x03030303u);
  }
  return live ? t & 0xFFu : 0u;
}

// Both groups' first walk and the run's decoded total T.  Leaves every group's
// decoded prefix in sm.comp[] and its packed prefixes in sm.out, so that after
// the caller's next barrier run_prefix() tells the decoded prefix at any stage
// position.  (Each lane collecting it for the rows that start in its groups,
// one loop iteration per row, cost a tenth of the kernel's instructions.)
__device__ __forceinline__ uint32_t fsst_walk_lengths(FsstGroup (&gr)[GROUPS_PER_THR], FsstSmem& sm,
                                                      const uint32_t (&prev)[GROUPS_PER_THR], uint32_t c_h,
                                                      uint32_t y_hi, const uint8_t* stage,
                                                      bool (&lits)[GROUPS_PER_THR])
{
  const uint32_t tid  = threadIdx.x;
  const uint32_t lane = lane_id();
  const uint32_t w    = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(tid >> 6)));
  uint32_t v[GROUPS_PER_THR] = {}, incl[GROUPS_PER_THR] = {};
#pragma unroll
  for (uint32_t k = 0; k < GROUPS_PER_THR; ++k) {
    lits[k] = false;
    gr[k].m = gr[k].lit = 0;
    if (16u * (k * FSST_THREADS + w * WAVE) < y_hi) {  // the wave has groups of the run
      // the word before the group: the lane below holds it, lane 0 loaded it
      const uint32_t pw = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
        static_cast<int>(prev[k]), static_cast<int>(gr[k].q[3]), 0x138, 0xF, 0xF, false));  // wave_shr:1
      v[k] = fsst_group_lengths(gr[k], sm, k * FSST_THREADS + tid, pw, c_h, y_hi, stage, &lits[k]);
      v[k] |= static_cast<uint32_t>(__builtin_popcount(gr[k].m)) << PK_LEN;
      incl[k] = wave_incl_sum_u32(v[k]);
    }
    if (lane == WAVE - 1) sm.part[k * FSST_WAVES + w] = incl[k];
  }
  lds_barrier();
  // every wave scans the 2 x FSST_WAVES wave sums in one 16-lane row
  static_assert(GROUPS_PER_THR * FSST_WAVES == 16, "one DPP row of wave sums");
  const uint32_t ws = sm.part[lane & 15u];
  const uint32_t wi = row_incl_sum_u32(ws);
  const uint32_t T  = static_cast<uint32_t>(__builtin_amdgcn_readlane(wi, 15)) & ((1u << PK_LEN) - 1u);
#pragma unroll
  for (uint32_t k = 0; k < GROUPS_PER_THR; ++k) {
    const uint32_t i  = k * FSST_WAVES + w;
    const uint32_t ex = __builtin_amdgcn_readlane(wi, i) - __builtin_amdgcn_readlane(ws, i) + incl[k] - v[k];
    gr[k].d           = ex & ((1u << PK_LEN) - 1u);
    gr[k].r           = ex >> PK_LEN;
    const uint32_t g  = k * FSST_THREADS + tid;
    if (16u * g < y_hi) {
      sm.comp[g]                               = gr[k].d;
      reinterpret_cast<u32x4*>(sm.out)[g] = u32x4{gr[k].p[0], gr[k].p[1], gr[k].p[2], gr[k].p[3]};
    }
  }
  if (tid == 0 && !(y_hi & 15u)) {  // the position after the last byte starts a group of its own
    sm.comp[y_hi >> 4] = T;
    sm.out[y_hi]       = 0;
  }
  return T;
}

// The decoded prefix of the run at stage position y.
__device__ __forceinline__ uint32_t run_prefix(const FsstSmem& sm, uint32_t y) { return sm.comp[y >> 4] + sm.out[y]; }

// OR symbol bytes v at window position o.
__device__ __forceinline__ void window_or(uint8_t* out, uint32_t o, uint64_t v)
{
  const uint32_t s  = (o << 3) & 24u;
  const uint64_t x  = v << s;
  const uint32_t x2 = (static_cast<uint32_t>(v >> 32) >> 1) >> (31u - s);
  uint32_t* d       = reinterpret_cast<uint32_t*>(out + (o & 0xFFFCu));
  __hip_atomic_fetch_or(d, static_cast<uint32_t>(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  __hip_atomic_fetch_or(d + 1, static_cast<uint32_t>(x >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (x2) __hip_atomic_fetch_or(d + 2, x2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Second walk of one group into the window over output bytes [w0, w0 +
// FSST_WINDOW) of the run.  MULTI: the run's output takes several windows;
// a wave skips a window that none of its groups reaches, and words outside
// the window go to a word past it.
template <bool MULTI>
__device__ __forceinline__ void fsst_group_emit(const FsstGroup& gr, FsstSmem& sm, uint32_t g, uint32_t y_hi, bool lits,
                                                uint32_t w0)
{
  bool live         = 16u * g < y_hi;
  const uint32_t pc = static_cast<uint32_t>(__builtin_popcount(gr.m));
  if constexpr (MULTI) {
    // rows that follow lie below in the output: the group's bytes are inside
    // [lo, hi), 128 of them at most in a row (lo may be negative: a row may
    // start inside the group)
    const int32_t lo = live ? static_cast<int32_t>(sm.dec[gr.r + pc] + gr.d - w0) : 0;
    const int32_t hi = live ? static_cast<int32_t>(sm.dec[gr.r] + gr.d + 128u - w0) : 0;
    live             = live && lo < static_cast<int32_t>(FSST_WINDOW) && hi > 0;
  } else if (!lits && !ballot(live && pc > 3u)) {
    if (!live) return;
    // at most four rows cross a group: what takes a prefix to its output
    // position, 16 bits for each, in two registers; a byte's row (0..3)
    // selects one with a byte permutation
    const uint32_t* b  = &sm.dec[gr.r];
    const uint32_t b01 = __builtin_amdgcn_perm(b[1] + gr.d, b[0] + gr.d, 0x05040100u);
    const uint32_t b23 = __builtin_amdgcn_perm(b[3] + gr.d, b[2] + gr.d, 0x05040100u);
#pragma unroll
    for (uint32_t h = 0; h < 16; h += 8) {
      uint64_t v[8];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) v[i] = sm.sym[group_byte(gr.q, h + i)];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) {
        const uint32_t j   = h + i;
        const uint32_t row = static_cast<uint32_t>(__builtin_popcount(gr.m & ((2u << j) - 1u)));
        const uint32_t bo  = __builtin_amdgcn_perm(b23, b01, 0x0C0C0100u + row * 0x0202u);
        window_or(sm.out, bo + group_byte(gr.p, j), v[i]);
      }
    }
    return;
  }
  if (!live) return;
  // any number of rows and partial windows: four bytes at a time, the row's
  // entry read for each
  uint32_t q[4], p[4];
#pragma unroll
  for (uint32_t d = 0; d < 4; ++d) {
    q[d] = gr.q[d];
    p[d] = gr.p[d];
  }
  uint32_t m = gr.m, lit = gr.lit, row = gr.r;
#pragma unroll 1
  for (uint32_t d = 0; d < 4; ++d) {
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t c = (q[0] >> (8u * j)) & 0xFFu;
      row += (m >> j) & 1u;
      const uint64_t v = (lit >> j) & 1u ? uint64_t{c} : sm.sym[c];
      const uint32_t o = sm.dec[row] + gr.d + ((p[0] >> (8u * j)) & 0xFFu) - w0;
      if constexpr (!MULTI) {
        window_or(sm.out, o, v);
      } else {
        const uint32_t s  = (o << 3) & 24u;
        const uint64_t x  = v << s;
        const uint32_t x2 = (static_cast<uint32_t>(v >> 32) >> 1) >> (31u - s);
        const int32_t w   = static_cast<int32_t>(o) >> 2;
        auto put          = [&](int32_t i, uint32_t b) {
          const uint32_t at = static_cast<uint32_t>(i) < FSST_WINDOW / 4u ? static_cast<uint32_t>(i) : FSST_WINDOW / 4u + 4u;
          __hip_atomic_fetch_or(reinterpret_cast<uint32_t*>(sm.out) + at, b, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        put(w, static_cast<uint32_t>(x));
        put(w + 1, static_cast<uint32_t>(x >> 32));
        put(w + 2, x2);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < 3; ++i) {
      q[i] = q[i + 1];
      p[i] = p[i + 1];
    }
    m >>= 4;
    lit >>= 4;
  }
}

// Clear the window's bytes [0, n) and the words a last symbol may reach, with
// 4-byte stores: in an earlier form of this kernel, clearing with 16-byte stores
// (ds_write_b128) and then ORing from other waves after a barrier lost about 0.2% of
// the ORed bytes once five or more workgroups shared a CU, and 4-byte stores never
// did.  No cause was found in the code or its assembly.
template <class SM>
__device__ __forceinline__ void window_clear(SM& sm, uint32_t n)
{
  for (uint32_t i = threadIdx.x * 4u; i < n + 12u; i += FSST_THREADS * 4u)
    *reinterpret_cast<uint32_t*>(&sm.out[i]) = 0u;
}

// 16 bytes at byte 16 - D (D = 1..16) of the pair of blocks a, b.
template <uint32_t WORD>
__device__ __forceinline__ u32x4 funnel16(const u32x4& a, const u32x4& b, uint32_t byte)
{
  const uint32_t c[9] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3], 0u};
  return u32x4{__builtin_amdgcn_alignbyte(c[WORD + 1], c[WORD], byte),
               __builtin_amdgcn_alignbyte(c[WORD + 2], c[WORD + 1], byte),
               __builtin_amdgcn_alignbyte(c[WORD + 3], c[WORD + 2], byte),
               __builtin_amdgcn_alignbyte(c[WORD + 4], c[WORD + 3], byte)};
}

// Whole 16-byte blocks of the window's store: block i of the destination
// (16-byte aligned) starts at window byte 16 i - skew, so its bytes come from
// the aligned window blocks i - 1 and i at an offset that is the same for the
// whole chunk.
template <uint32_t WORD, class SM>
__device__ __forceinline__ void window_store_blocks(const SM& sm, uintptr_t dst, uint32_t i0, uint32_t i1,
                                                    uint32_t byte)
{
  const u32x4* w = reinterpret_cast<const u32x4*>(sm.out);
  for (uint32_t i = i0 + threadIdx.x; i < i1; i += FSST_THREADS) {
    u32x4 v;
    if constexpr (WORD == 4) v = w[i];
    else v = funnel16<WORD>(w[i - 1u], w[i], byte);
    __builtin_nontemporal_store(v, gbl(reinterpret_cast<u32x4*>(dst + 16u * uintptr_t{i})));
  }
}

// The window's n bytes to global address g: 16-byte stores, single bytes
// where the first and last 16-byte blocks are shared with other chunks.
template <class SM>
__device__ __forceinline__ void window_store(const SM& sm, uintptr_t g, uint32_t n)
{
  const uint32_t skew = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(g & 15u)));
  const uintptr_t dst = g - skew;
  const uint32_t i0   = skew ? 1u : 0u;       // first whole block
  const uint32_t i1   = (skew + n) / 16u;     // past the last whole block
  const uint32_t at   = 16u - skew;           // the first byte's place in a pair of window blocks
  if (i1 > i0) {
    switch (at >> 2) {
      case 0: window_store_blocks<0>(sm, dst, i0, i1, at & 3u); break;
      case 1: window_store_blocks<1>(sm, dst, i0, i1, at & 3u); break;
      case 2: window_store_blocks<2>(sm, dst, i0, i1, at & 3u); break;
      case 3: window_store_blocks<3>(sm, dst, i0, i1, at & 3u); break;
      default: window_store_blocks<4>(sm, dst, i0, i1, 0u); break;
    }
  }
  // bytes before the first whole block and after the last one
  const uint32_t head = skew ? (16u - skew < n ? 16u - skew : n) : 0u;
  const uint32_t tail = i1 >= i0 && i1 * 16u > skew ? i1 * 16u - skew : head;
  if (threadIdx.x < 16u) {
    if (threadIdx.x < head) *gbl(reinterpret_cast<uint8_t*>(g + threadIdx.x)) = sm.out[threadIdx.x];
  } else if (threadIdx.x < 32u) {
    const uint32_t x = (tail > head ? tail : head) + threadIdx.x - 16u;
    if (x < n) *gbl(reinterpret_cast<uint8_t*>(g + x)) = sm.out[x];
  }
}

// Decoupled look-back for the column-wide chars offset of chunk c, by wave
// 0: publish this chunk's aggregate T (fsst_lookback_publish), then sum
// predecessors 64 at a time back to the nearest published inclusive prefix
// (fsst_lookback_wait).  Between the two the workgroup may do other work.  A
// chunk waits at most `spin_limit` sleeps for predecessors that show nothing;
// past that (or at once when spin_limit is 0, which only tests set) it sets
// the column's error flag and ends, so that the decode is repeated or its failure
// reported and no wave hangs.  Where the only ones missing have said that they
// have begun (fsst_lookback_begin), which chunks do whose lengths take long, it
// waits for them FSST_SPIN_LIMIT sleeps, whatever `spin_limit`.  A status word carries its flag and value together and is the
// only datum exchanged between chunks, so device-scope relaxed atomics
// (coherent across the XCDs' L2s) suffice; release/acquire orderings would
// add an L2 write-back / invalidate per access.
__device__ __forceinline__ void fsst_lookback_publish(uint32_t c, uint64_t T, FsstState* st, uint32_t spin_limit)
{
  if (threadIdx.x == 0) {
    const gptr<uint64_t> status = gbl(st->status);
    if (c == 0) __hip_atomic_store(&status[0], ST_INC | T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else if (spin_limit != 0) __hip_atomic_store(&status[c], ST_AGG | T, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Chunk c has begun and will publish: for chunks that take long to (the
// compressed bytes of several runs, or of rows that no run holds, are walked
// first: a row of 120 KB takes milliseconds).
__device__ __forceinline__ void fsst_lookback_begin(uint32_t c, FsstState* st, uint32_t spin_limit)
{
  if (threadIdx.x == 0 && spin_limit != 0)
    __hip_atomic_store(&gbl(st->status)[c], ST_RUN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void fsst_lookback_failed(FsstState* st)
{
  __hip_atomic_fetch_or(gbl(&st->error), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (FsstResult* const r = *gbl(&st->result)) *gbl(&r->error) = 1u;
  if (uint32_t* const f = *gbl(&st->failed)) *gbl(f) = 1u;
}

// The wait half: synchronises the workgroup and returns the exclusive prefix
// to every thread.
template <class SM>
__device__ __forceinline__ uint64_t fsst_lookback_wait(uint32_t c, uint32_t n_chunks, uint64_t T, FsstState* st,
                                                       uint32_t spin_limit, SM& sm)
{
  if (threadIdx.x < WAVE) {
    const uint32_t lane = threadIdx.x;
    const gptr<uint64_t> status = gbl(st->status);
    uint64_t excl64     = 0;
    if (c == 0) {
      // published inclusive already
    } else if (spin_limit == 0) {  // no waiting allowed: report the look-back as failed
      if (lane == 0) fsst_lookback_failed(st);
    } else {
      uint32_t p = c - 1, spins = 0, begun = 0;
      for (;;) {
        const bool valid = lane <= p;
        const uint64_t s =
          valid ? __hip_atomic_load(&status[p - lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        const uint64_t flag = s & ~ST_VAL;
        const uint64_t incm = ballot(valid && flag == ST_INC);
        const uint32_t stop = incm ? static_cast<uint32_t>(__builtin_ctzll(incm)) : (p < WAVE - 1 ? p : WAVE - 1);
        const uint64_t need = stop == WAVE - 1 ? ~0ull : ((2ull << stop) - 1ull);
        const uint64_t none = ballot(valid && flag == 0) & need;
        if (none | (ballot(valid && flag == ST_RUN) & need)) {  // a predecessor has not published yet
          if (none ? ++spins > spin_limit : ++begun > FSST_SPIN_LIMIT) {  // give up rather than hang
            if (lane == 0) fsst_lookback_failed(st);
            break;
          }
          __builtin_amdgcn_s_sleep(1);
          continue;
        }
        excl64 += readlane_u64(wave_incl_sum_u64(lane <= stop ? (s & ST_VAL) : 0ull), WAVE - 1);
        if (incm || p < WAVE) break;  // chunk 0 always publishes an inclusive prefix
        p -= WAVE;
      }
      if (lane == 0)
        __hip_atomic_store(&status[c], ST_INC | ((excl64 + T) & ST_VAL), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (lane == 0) {
      sm.base = excl64;
      if (c == n_chunks - 1) {
        *gbl(&st->total) = excl64 + T;
        if (FsstResult* const r = *gbl(&st->result)) *gbl(&r->total) = excl64 + T;
      }
    }
  }
  __syncthreads();
  return sm.base;
}

// Both halves with nothing between them.
template <class SM>
__device__ __forceinline__ uint64_t fsst_lookback(uint32_t c, uint32_t n_chunks, uint64_t T, FsstState* st,
                                                  uint32_t spin_limit, SM& sm)
{
  fsst_lookback_publish(c, T, st, spin_limit);
  return fsst_lookback_wait(c, n_chunks, T, st, spin_limit, sm);
}

// Column offsets of the chunk's rows (and the column's closing offset).
template <class SM>
__device__ __forceinline__ void fsst_offsets(const FsstChunk& ch, uint32_t c, uint32_t n_chunks, uint32_t rows,
                                             uint32_t T, uint64_t base, int32_t* offsets, uint32_t total_rows,
                                             const SM& sm)
{
  const gptr<int32_t> off = gbl(offsets);
  for (uint32_t i = threadIdx.x; i < rows; i += FSST_THREADS)
    off[ch.col_row + i] = static_cast<int32_t>(static_cast<uint32_t>(base + sm.dec[i]));
  if (c == n_chunks - 1 && threadIdx.x == 0) off[total_rows] = static_cast<int32_t>(static_cast<uint32_t>(base + T));
}

// ---- segment pre-pass ----

constexpr uint32_t PREP_STAGE = 16384;  // segment bytes of the length stream staged at a time

// A pre-pass workgroup of NT threads, 256 or more (a symbol table is imported
// one code per thread).
template <uint32_t NT>
struct FsstPrepSmem {
  __attribute__((aligned(16))) uint8_t st[FSST_SYMSTAGE + 48];
  __attribute__((aligned(16))) uint32_t fields[(PREP_STAGE + 128) / 4];
  uint8_t len[256];  // code lengths of a DICT_FSST dictionary's table
  uint32_t sum[NT];
  uint8_t huge[NT];
  uint32_t wave[NT / WAVE];
};

// Sum of the w-bit fields [f0, f1) of the length stream at `base`, and
// whether one of them reaches ROW_HUGE.  Fields past `end` read as zero.
__device__ __forceinline__ uint32_t fields_sum(const uint8_t* base, const uint8_t* end, uint32_t f0, uint32_t f1,
                                               uint32_t w, bool* huge)
{
  uint32_t s = 0, mx = 0;
  if (f0 < f1 && w) {
    if (base + ((uint64_t{f1} * w + 7u) >> 3) <= end) {
      BitCursor bc(base, uint64_t{f0} * w);
      for (uint32_t f = f0; f < f1; ++f) {
        const uint32_t v = bc.next(w);
        s += v;
        mx = v > mx ? v : mx;
      }
    } else {
      for (uint32_t f = f0; f < f1; ++f) {
        const uint32_t v = stream_bits32(base, end, uint64_t{f} * w, w);
        s += v;
        mx = v > mx ? v : mx;
      }
    }
  }
  *huge = mx >= ROW_HUGE;
  return s;
}

// Sum of the first n (at most 16) w-bit fields (1 <= w <= 32) from bit `bit` of
// a stream staged in LDS, and the largest of them into *mx.  All 16 are read,
// so that no branch or earlier read holds one back (a word cursor, or a branch
// around each field, took 250 cycles a field): up to 68 bytes past the first
// field must be readable.
__device__ __forceinline__ uint32_t lds_fields_sum(const uint32_t* lds, uint32_t bit, uint32_t n, uint32_t w,
                                                   uint32_t* mx)
{
  uint32_t v[16], s = 0, m = 0;
#pragma unroll
  for (uint32_t f = 0; f < 16; ++f) v[f] = lds_bits32(lds, bit + f * w, w);
#pragma unroll
  for (uint32_t f = 0; f < 16; ++f) {
    const uint32_t x = f < n ? v[f] : 0u;
    s += x;
    m = x > m ? x : m;
  }
  *mx = m;
  return s;
}

// ---- DICTIONARY and UNCOMPRESSED strings ----
//
// DICTIONARY (strings/dictionary.cu:17-33): a 20-byte header {dict_size,
// dict_end, index_buffer_offset, index_buffer_count, bitpacking_width}, the
// bit-packed selection values from byte 20 (0 is NULL), u32 cumulative
// entry ends at index_buffer_offset and entry bytes stored back to front
// ending at dict_end: entry s is [dict_end - idx[s], dict_end - idx[s-1]).
// The header is valid if the index buffer and dict_end lie inside the
// segment and the width is <= 32 (:57-64).
//
// UNCOMPRESSED (strings/uncompressed.cu:17-33): {dict_size, dict_end} then
// one int32 cumulative end per row from byte 8, read as |v| (the sign is
// DuckDB's in-memory marker); row i is [dict_end - |off[i]|, dict_end -
// |off[i-1]|).  The segment is valid if its offsets fit (:66); dict_end
// must also lie inside the segment here (the reference does not check it).
//
// Malformed input only: a row whose end passes dict_end or falls below its
// start decodes empty, where the reference would copy from outside the
// segment; a DICTIONARY selection >= index_buffer_count is empty in both of
// the reference's passes' intent (its length pass gives 0).

// Per-chunk info of a plain segment, one thread per chunk.
template <uint32_t NT>
__device__ __forceinline__ void plain_prep_segment(const FsstSeg& sg, FsstChunkInfo* __restrict__ info)
{
  const uint8_t* seg = sg.bytes;
  const bool dict    = sg.codec == SDR_CODEC_DICTIONARY;
  uint32_t dict_end = 0, ibo = 0, ibc = 0, width = 0;
  bool ok = false;
  if (dict) {
    if (sg.bytes_size >= 20u) {
      dict_end = su32(seg + 4);
      ibo      = su32(seg + 8);
      ibc      = su32(seg + 12);
      width    = su32(seg + 16);
      ok = uint64_t{ibo} + 4ull * ibc <= sg.bytes_size && dict_end <= sg.bytes_size && width <= 32u;
    }
  } else if (uint64_t{sg.bytes_size} >= 8ull + 4ull * sg.row_count) {
    dict_end = su32(seg + 4);
    ok       = dict_end <= sg.bytes_size;
  }
  const uint32_t flags = (dict ? FI_DICT | (width & FI_WIDTH) : FI_UNC) | (ok ? FI_OK : 0u);
  for (uint32_t k = threadIdx.x; uint64_t{k} * sg.chunk_rows < sg.row_count; k += NT) {
    FsstChunkInfo ci;
    ci.bytes      = seg;
    ci.c_lo       = ibo;
    ci.c_hi       = ibc;
    ci.dict_end   = dict_end;
    ci.flags      = flags;
    ci.bytes_size = sg.bytes_size;
    ci.pad        = 0;
    const gptr<u32x4> dst = gbl(reinterpret_cast<u32x4*>(info + sg.first_chunk + k));
    const u32x8 cv        = __builtin_bit_cast(u32x8, ci);
    dst[0]                = cv.lo;
    dst[1]                = cv.hi;
  }
}

// ---- DICT_FSST strings ----
//
// strings/dict_fsst.cu:17-38: a 16-byte header, the dictionary entries front
// to back from byte 16 (entry 0 is the NULL slot), in the FSST modes (1, 2)
// a symbol table, the bit-packed entry lengths and, except in mode 2, the
// bit-packed row indices; mode 0 keeps entries raw, mode 1 FSST-compresses
// them, mode 2 has one entry per row (row i is entry i + 1).  The host reads
// the headers and fills DictFsstSeg (region offsets, :516-525); a pre-pass
// per segment builds the entry offsets (:160-235), a predecode pass writes
// the FSST entries once (:268-320), and the rows copy their entry like
// DICTIONARY rows (:246-265, :324-360).  Bytes past the segment read as
// zero; the byte a trailing escape counts is written as 0.

// Calls f(byte) for n bytes in order, the first of them byte `skew` (0..3) of word
// 0 of those that w(k) reads, four words in flight (a byte at a time, each load
// waited for, was most of the DICT_FSST passes).
template <typename W, typename F>
__device__ __forceinline__ void each_byte(W w, uint32_t skew, uint32_t n, F f)
{
  if (n == 0) return;
  const uint64_t stop = uint64_t{skew} + n;
  const uint32_t last = static_cast<uint32_t>((stop - 1u) >> 2);
  for (uint32_t k = 0; k <= last; k += 4) {
    uint32_t v[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) v[j] = w(k + j < last ? k + j : last);
#pragma unroll
    for (uint32_t b = 0; b < 16; ++b) {
      const uint64_t y = 4ull * k + b;
      if (y >= skew && y < stop) f(v[b / 4u] >> (8u * (b % 4u)) & 0xFFu);
    }
  }
}

// The words at p rounded down, in memory.
struct GlobalWords {
  gptr<const uint32_t> w;
  uint32_t skew;
  __device__ __forceinline__ explicit GlobalWords(const uint8_t* p)
    : skew(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3u))
  {
    w = gbl(reinterpret_cast<const uint32_t*>(p - skew));
  }
  __device__ __forceinline__ uint32_t operator()(uint32_t k) const { return w[k]; }
};

// Decoded length of one compressed entry of n bytes, of which those past the first
// `in` read as zero, i.e. as code 0: a code adds its symbol's length, an escape
// adds one (len[255]) and skips the next byte, even past the entry's end.
template <typename W>
__device__ __forceinline__ uint32_t dfsst_entry_len(W w, uint32_t skew, uint32_t n, uint64_t in, const uint8_t* len)
{
  const uint32_t n_in = n < in ? n : static_cast<uint32_t>(in);
  uint32_t dl = 0;
  bool esc    = false;
  each_byte(w, skew, n_in, [&](uint32_t code) {
    dl += esc ? 0u : len[code];
    esc = !esc && code == FSST_ESC;
  });
  const uint32_t zeros = n - n_in;  // past the segment
  if (zeros) dl += (zeros - (esc ? 1u : 0u)) * len[0];
  return dl;
}

// The offsets of thread t's rows 2t and 2t + 1, and the column's closing one.
__device__ __forceinline__ void fsst_row_offsets(uint32_t c, uint32_t n_chunks, uint32_t col_row, uint32_t rows,
                                                 uint64_t T, uint64_t base, uint32_t o0, uint32_t o1, int32_t* offsets,
                                                 uint32_t total_rows)
{
  const uint32_t r        = 2u * threadIdx.x;
  const gptr<int32_t> off = gbl(offsets) + col_row;
  if (r < rows) off[r] = static_cast<int32_t>(static_cast<uint32_t>(base) + o0);
  if (r + 1u < rows) off[r + 1u] = static_cast<int32_t>(static_cast<uint32_t>(base) + o1);
  if (c == n_chunks - 1u && threadIdx.x == 0)
    gbl(offsets)[total_rows] = static_cast<int32_t>(static_cast<uint32_t>(base + T));
}

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

// The w-bit field (1 <= w <= 32) at bit `bit` from the word p, of a stream that
// holds all of it.
__device__ __forceinline__ uint32_t bits32_inside(gptr<const uint32_t> p, uint32_t bit, uint32_t w)
{
  const uint32_t k = bit >> 5, off = bit & 31u;
  const uint32_t lo = p[k], hi = p[k + (off + w > 32u ? 1u : 0u)];
  return __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(hi, lo, off), 0u, w);
}

// A row's bytes into the window over chunk output bytes [w0, w0 + FSST_WINDOW)
// (cleared): bytes [src, src + len) of `seg` are output bytes [d, d + len);
// those at or past `size` (not 0) are zeros.  Sixteen bytes a load, funnelled
// into words of the window and ORed in, since a row's first and last word are
// shared with its neighbours.
template <class SM>
__device__ __forceinline__ void plain_copy_row(SM& sm, const uint8_t* seg, uint32_t size, uint32_t src, uint32_t len,
                                               uint32_t d, uint32_t w0)
{
  const uint32_t skew          = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(seg) & 3u);
  const gptr<const uint32_t> w = gbl(reinterpret_cast<const uint32_t*>(seg - skew));
  const uint32_t w_last        = static_cast<uint32_t>((uint64_t{skew} + size - 1u) >> 2);  // the last that may be read
  const uint32_t left          = src < size ? size - src : 0u;
  const uint32_t have          = len < left ? len : left;
  const uint32_t j0            = d < w0 ? w0 - d : 0u;
  const uint32_t lim           = w0 + FSST_WINDOW > d ? w0 + FSST_WINDOW - d : 0u;
  const uint32_t j1            = have < lim ? have : lim;
  if (j0 >= j1) return;
  // Source words k0, k0 + 1, ...: k0 holds the first byte.  Words k0 + k - 1 and
  // k0 + k make window word o + k, from byte ph on; f: the first pair makes none
  // of the row's.
  const uint32_t p  = d + j0 - w0;  // first window byte
  const uint32_t x  = src + j0;
  const uint32_t x3 = (x & 3u) + skew;
  const uint32_t sh = p & 3u;
  const uint32_t nb = sh + (j1 - j0);  // bytes from the first window word's start
  const uint32_t ph = x3 - sh;         // the funnel takes it modulo 4
  const uint32_t f  = (x3 & 3u) >= sh ? 1u : 0u;
  const uint32_t o  = (p >> 2) - f;
  const uint32_t k0 = (x >> 2) + (x3 >> 2);
  const uint32_t nw = ((nb + 3u) >> 2) + f;
  uint32_t carry    = 0;
#pragma unroll 1
  for (uint32_t k = 0; k < nw; k += 4) {
    u32x4 n;
    if (ballot(k0 + k + 3u > w_last) == 0) {
      n = *(gptr<const u32x4_a4>)(w + k0 + k);
    } else {
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) n[j] = w[k0 + k + j < w_last ? k0 + k + j : w_last];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t at = 4u * (k + j - f);  // wraps where f drops the first
      uint32_t v        = __builtin_amdgcn_alignbyte(n[j], carry, ph);
      carry             = n[j];
      if (at < nb) {
        if (at == 0) v &= ~0u << (8u * sh);
        if (nb - at < 4u) v &= (1u << (8u * (nb - at))) - 1u;
        __hip_atomic_fetch_or(reinterpret_cast<uint32_t*>(sm.out) + (o + k + j), v, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
  }
}

// plain_copy_row for B rows of which each lies whole in the window, which begins
// with the chunk's output, and in the segment: row i's bytes [src[i], src[i] +
// len[i]) are window bytes [d[i], d[i] + len[i]).  The copy costs instructions
// as much as loads, so what is not needed then is left out, and the first
// word's mask is applied to the source, the last word's made once.  Where a
// lane needs no further words it loads its row's first again (a row without
// bytes, the segment's): no branch holds a load back.
template <uint32_t B, class SM>
__device__ __forceinline__ void plain_copy_whole(SM& sm, const uint8_t* seg, uint32_t size, const uint32_t* src,
                                                 const uint32_t* len, const uint32_t* d)
{
  const uint32_t skew          = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(seg) & 3u);
  const gptr<const uint8_t> w  = gbl(seg - skew);
  const uint32_t w_last        = (skew + size - 1u) >> 2;  // the last word that may be read
  // Source words k0 + k: k0 holds the row's first byte.  Words k0 + k - 1 and
  // k0 + k make, from byte ph on, window word o + k; the first pair makes none of
  // the row's if `skip`, the one with 4 k = `last` its last, of which `tail` are
  // its bytes.
  uint32_t k0[B], ph[B], o[B], last[B], tail[B], carry[B] = {}, most = 0;
  bool skip[B];
#pragma unroll
  for (uint32_t i = 0; i < B; ++i) {
    const uint32_t sh = d[i] & 3u;
    const uint32_t x  = src[i] + skew;
    skip[i]           = (x & 3u) >= sh;
    const uint32_t f4 = skip[i] ? 4u : 0u;
    const uint32_t e  = sh + len[i] + f4;  // where the row ends, from word o on
    ph[i]             = x - sh;            // the funnel takes it modulo 4
    o[i]              = (d[i] >> 2) - (f4 >> 2);
    k0[i]             = len[i] ? x >> 2 : 0u;
    last[i]           = (e - 1u) & ~3u;
    tail[i]           = ~0u >> (8u * ((0u - e) & 3u));
    if (len[i] == 0u) {  // no word of the window
      skip[i] = true;
      last[i] = 0u;
    }
    most = last[i] > most ? last[i] : most;
  }
#pragma unroll 1
  for (uint32_t k = 0;; k += 4) {
    u32x4 n[B];
    uint32_t at[B];
    bool past = false;
#pragma unroll
    for (uint32_t i = 0; i < B; ++i) {
      at[i] = k0[i] + (4u * k <= last[i] ? k : 0u);
      past  = past || at[i] + 3u > w_last;
    }
    if (ballot(past) == 0) {
#pragma unroll
      for (uint32_t i = 0; i < B; ++i) n[i] = *(gptr<const u32x4_a4>)(w + 4u * at[i]);
    } else {
#pragma unroll
      for (uint32_t i = 0; i < B; ++i)
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
          n[i][j] = *(gptr<const uint32_t>)(w + 4u * (at[i] + j < w_last ? at[i] + j : w_last));
    }
#pragma unroll
    for (uint32_t i = 0; i < B; ++i) {
      if (k == 0) n[i][0] &= ~0u << (8u * ((src[i] + skew) & 3u));  // uniform
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t t = 4u * (k + j);
        const uint32_t v = __builtin_amdgcn_alignbyte(n[i][j], carry[i], ph[i]) & (t == last[i] ? tail[i] : ~0u);
        carry[i]         = n[i][j];
        if (t <= last[i] && !(j == 0 && k == 0 && skip[i]))
          __hip_atomic_fetch_or(reinterpret_cast<uint32_t*>(sm.out) + (o[i] + k + j), v, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    }
    if (4u * (k + 4u) > most) break;
  }
}

// A DICTIONARY segment's entries in LDS: as many and as long ones as there is room for.
constexpr uint32_t LABEL_ENTRIES = 256;
constexpr uint32_t LABEL_BYTES   = 32;

// LDS of a workgroup that decodes no FSST chunk.
struct PlainSmem {
  __attribute__((aligned(16))) uint32_t lead[4];  // a row's first word may be ORed, with zeros, one before the window
  __attribute__((aligned(16))) uint8_t out[FSST_WINDOW + 48];
  __attribute__((aligned(16))) uint32_t label[LABEL_ENTRIES][LABEL_BYTES / 4];  // zero past an entry's end
  uint32_t label_src[LABEL_ENTRIES];  // where it lies in the segment
  uint8_t label_len[LABEL_ENTRIES];
  uint32_t part[WAVE];
  uint32_t flag[FSST_WAVES];
  uint64_t sum[FSST_WAVES];
  uint64_t base;
  __device__ __forceinline__ uint32_t* plain_part() { return part; }
  __device__ __forceinline__ uint64_t* plain_sum() { return sum; }
};

struct PlainArgs {
  const uint8_t* seg;
  uint32_t bytes_size, dict_end, flags, ibo, ibc, row_begin, rows, col_row, c, n_chunks;
  FsstState* st;
  int32_t* offsets;
  uint8_t* chars;
  uint64_t chars_cap;
  uint32_t total_rows, spin_limit;
};

// Decode chunk c of a valid DICTIONARY, UNCOMPRESSED or DICT_FSST segment: per-
// row lengths (dictionary.cu:84-108, uncompressed.cu:56-81), the chunk's
// look-back for its chars offset, offsets, and the bytes (dictionary.cu:
// 117-140, uncompressed.cu:88-120).  Every thread must call it.
//
// Bound by latency and instructions alike: a chunk takes its descriptors, the
// rows' indices, their entries and bytes, and the look-back,
// each a round trip to memory that the next waits for.  So a thread owns RPT
// rows, 512 apart (offsets are then stored whole lines at a time, and a chunk's
// output leaves in row order however few rows a window holds), and its loads of
// one kind are in flight together.  8 Mi label rows 119 -> 57 us, 2 M rows of 27
// chars 57 -> 35 us (with a kernel of its own and without tickets, see k_plain).
template <uint32_t RPT, class SM>
__device__ __forceinline__ void plain_chunk(const PlainArgs& args, SM& sm)
{
  const PlainArgs a   = uniform(args);
  const uint32_t bytes_size = a.bytes_size, dict_end = a.dict_end, flags = a.flags, ibo = a.ibo, ibc = a.ibc;
  const uint32_t row_begin = a.row_begin, rows = a.rows, col_row = a.col_row, c = a.c, n_chunks = a.n_chunks;
  FsstState* const st = a.st;
  const uint64_t chars_cap  = a.chars_cap;
  const uint32_t spin_limit = a.spin_limit;
  const uint8_t* seg        = a.seg;
  const uint32_t tid  = threadIdx.x;
  const bool dict     = flags & FI_DICT;
  const bool dfsst    = flags & FI_DFSST;
  uint32_t w          = flags & FI_WIDTH;
  const uint8_t* bits = seg + 20;  // selection values or indices
  const uint8_t* end  = seg + bytes_size;
  const uint8_t* ent  = seg + (dict ? uint64_t{ibo} : 4ull);  // entry k is between words k - 1 and k
  uint32_t n_ent      = dict ? ibc : 1u << 30;  // past every row of an UNCOMPRESSED segment
  uint32_t size       = bytes_size;  // of the bytes the rows copy from
  bool implied        = !dict;       // row r is entry r + 1
  if (dfsst) {  // seg is the segment's descriptor; rows copy from its entries
    const DictFsstSeg dd = uniform(gload(reinterpret_cast<const DictFsstSeg*>(seg)));
    w       = dd.diw;
    bits    = dd.bytes + dd.off_didx;
    end     = dd.bytes + dd.bytes_size;
    seg     = dd.src;
    size    = dd.src_size < ~0u ? static_cast<uint32_t>(dd.src_size) : ~0u;
    ent     = reinterpret_cast<const uint8_t*>(dd.e + 1);  // entry k is between e[k] and e[k + 1]
    n_ent   = dd.dict_count;
    implied = dd.mode == 2u;
  }
  uint32_t idx[RPT];
  if (implied) {
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) idx[i] = row_begin + FSST_THREADS * i + tid + 1u;
  } else if (w && bits + ((uint64_t{row_begin + rows} * w + 7u) >> 3) <= end) {
    const uint64_t bit0          = uint64_t{row_begin} * w;
    const uintptr_t at           = reinterpret_cast<uintptr_t>(bits) + (bit0 >> 3);
    const uint32_t skew          = 8u * static_cast<uint32_t>(at & 3u) + static_cast<uint32_t>(bit0 & 7u);
    const gptr<const uint32_t> p = gbl(reinterpret_cast<const uint32_t*>(at & ~uintptr_t{3}));
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) {
      const uint32_t r = FSST_THREADS * i + tid;
      idx[i]           = bits32_inside(p, skew + (r < rows ? r : 0u) * w, w);
    }
  } else {
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) {
      const uint32_t r = FSST_THREADS * i + tid;
      idx[i]           = r < rows ? stream_bits32(bits, end, uint64_t{row_begin + r} * w, w) : 0u;
    }
  }
  uint32_t e0[RPT] = {}, e1[RPT] = {};
  if (n_ent > 1u) {
    uint32_t k[RPT];
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i)
      k[i] = FSST_THREADS * i + tid < rows && idx[i] < n_ent && idx[i] ? idx[i] - 1u : 0u;
    if ((reinterpret_cast<uintptr_t>(ent) & 3u) == 0 && n_ent <= 1u << 30) {  // uniform; offsets of 32 bits
#pragma unroll
      for (uint32_t i = 0; i < RPT; ++i) {
        const u32x2_a4 e = *(gptr<const u32x2_a4>)(gbl(ent) + 4u * k[i]);
        e0[i]            = e[0];
        e1[i]            = e[1];
      }
    } else {
#pragma unroll
      for (uint32_t i = 0; i < RPT; ++i) {
        e0[i] = ld_u32_any(ent + 4ull * k[i]);
        e1[i] = ld_u32_any(ent + 4ull * k[i] + 4u);
      }
    }
  }
  uint32_t len[RPT], src[RPT], out[RPT];
  uint32_t big = 0;
  bool clip    = size > ~0u - 8u;  // the rows' bytes may end past the source's, or wrap
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) {
    const uint32_t r = FSST_THREADS * i + tid;
    if (flags & FI_UNC) {  // |v|: the sign is a marker; word -1 is not an offset
      const int32_t v0 = row_begin + r ? static_cast<int32_t>(e0[i]) : 0, v1 = static_cast<int32_t>(e1[i]);
      e0[i] = v0 < 0 ? 0u - static_cast<uint32_t>(v0) : static_cast<uint32_t>(v0);
      e1[i] = v1 < 0 ? 0u - static_cast<uint32_t>(v1) : static_cast<uint32_t>(v1);
    }
    // a DICT_FSST segment's entries are front to back, the others' back to
    // front; a row whose end passes dict_end or falls below its start is empty
    const bool sound = r < rows && idx[i] && idx[i] < n_ent && e1[i] >= e0[i] && (dfsst || e1[i] <= dict_end);
    len[i]           = sound ? e1[i] - e0[i] : 0u;
    src[i]           = !sound ? 0u : dfsst ? e0[i] : dict_end - e1[i];
    big |= len[i] >> 18;
    clip = clip || uint64_t{src[i]} + len[i] > size;
  }
  // Output positions modulo 2^32: each wave's rows of step i, behind the waves
  // and steps before them.  2^12 rows of less than 2^18 bytes can not overflow;
  // a chunk with a longer one adds its total up in 64 bits as well.
  uint32_t* const part = sm.plain_part();  // [i][wave]
  uint64_t* const sum  = sm.plain_sum();   // [wave]
  const uint32_t wv    = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(tid / WAVE)));
  uint64_t wave_sum    = 0;
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) {
    out[i] = wave_incl_sum_u32(len[i]);
    if (lane_id() == WAVE - 1u) part[FSST_WAVES * i + wv] = out[i];
    wave_sum += static_cast<uint32_t>(__builtin_amdgcn_readlane(out[i], WAVE - 1));
    out[i] -= len[i];
  }
  if (ballot(big != 0u)) {
    wave_sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) wave_sum += len[i];
    wave_sum = readlane_u64(wave_incl_sum_u64(wave_sum), WAVE - 1) | 1ull << 63;
  }
  if (ballot(clip)) wave_sum |= 1ull << 62;
  if (lane_id() == 0u) sum[wv] = wave_sum;
  __syncthreads();
  static_assert(FSST_WAVES * RPT <= WAVE, "a lane per step and wave");
  const uint32_t mine = lane_id() < FSST_WAVES * RPT ? part[lane_id()] : 0u;
  const uint32_t incl = wave_incl_sum_u32(mine);
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) out[i] += __builtin_amdgcn_readlane(incl - mine, FSST_WAVES * i + wv);
  uint64_t T64 = static_cast<uint32_t>(__builtin_amdgcn_readlane(incl, WAVE - 1));
  const uint32_t marks = static_cast<uint32_t>(sum[lane_id() % FSST_WAVES] >> 62);
  if (ballot(marks & 2u)) {  // the same in every wave
    T64 = 0;
    for (uint32_t v = 0; v < FSST_WAVES; ++v) T64 += sum[v] & ~(3ull << 62);
  }
  // publish a saturated total past 2^31, so the column reports overflow
  const uint64_t Tp = T64 > 0x7FFFFFFFull ? 0x80000000ull : T64;
  const uint32_t T  = static_cast<uint32_t>(Tp);
  fsst_lookback_publish(c, Tp, st, spin_limit);
  auto store_offsets = [&](uint64_t base) {
    const gptr<int32_t> off = gbl(a.offsets) + col_row;
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) {
      const uint32_t r = FSST_THREADS * i + tid;
      if (r < rows) off[r] = static_cast<int32_t>(static_cast<uint32_t>(base) + out[i]);
    }
    if (c == n_chunks - 1u && tid == 0)
      gbl(a.offsets)[a.total_rows] = static_cast<int32_t>(static_cast<uint32_t>(base + Tp));
  };
  if (Tp != T64) {  // nothing but the offsets can be written
    store_offsets(fsst_lookback_wait(c, n_chunks, Tp, st, spin_limit, sm));
    return;
  }
  // Rows are copied B at a time, the arrays turned by B after each: one copy of
  // the code, and only B rows' state in registers.
  constexpr uint32_t B = 2;
  auto turn = [&](uint32_t by) {
    if (RPT == by) return;
#pragma unroll
    for (uint32_t j = 0; j < by; ++j) {
      const uint32_t s0 = src[0], l0 = len[0], o0 = out[0];
#pragma unroll
      for (uint32_t i = 0; i + 1u < RPT; ++i) {
        src[i] = src[i + 1u];
        len[i] = len[i + 1u];
        out[i] = out[i + 1u];
      }
      src[RPT - 1u] = s0;
      len[RPT - 1u] = l0;
      out[RPT - 1u] = o0;
    }
  };
  if (T <= FSST_WINDOW && size && ballot(marks & 1u) == 0) {
    window_clear(sm, T);
    __syncthreads();
#pragma unroll 1
    for (uint32_t i = 0; i < RPT; i += B) {
      plain_copy_whole<B>(sm, seg, size, src, len, out);
      turn(B);
    }
    const uint64_t at = fsst_lookback_wait(c, n_chunks, Tp, st, spin_limit, sm);  // synchronises the workgroup
    store_offsets(at);
    if (at < chars_cap)
      window_store(sm, reinterpret_cast<uintptr_t>(a.chars) + at,
                   at + T <= chars_cap ? T : static_cast<uint32_t>(chars_cap - at));
    return;
  }
  // A window or more for each step of 512 rows, output bytes [w0, hi)
  const uint64_t base = fsst_lookback_wait(c, n_chunks, Tp, st, spin_limit, sm);
  store_offsets(base);
  uint32_t w0 = 0;
#pragma unroll 1
  for (uint32_t i = 0; i < RPT; ++i) {
    const uint32_t hi =
      i + 1u < RPT ? static_cast<uint32_t>(__builtin_amdgcn_readlane(incl - mine, FSST_WAVES * (i + 1u))) : T;
    while (w0 < hi) {
      const uint32_t nw = hi - w0 < FSST_WINDOW ? hi - w0 : FSST_WINDOW;
      window_clear(sm, nw);
      __syncthreads();
      __asm__ volatile("" : "+v"(src[0]), "+v"(len[0]), "+v"(out[0]));  // keep no more of the row between windows
      if (size) plain_copy_row(sm, seg, size, src[0], len[0], out[0], w0);
      __syncthreads();
      const uint64_t at = base + w0;
      if (at >= chars_cap) return;
      window_store(sm, reinterpret_cast<uintptr_t>(a.chars) + at,
                   at + nw <= chars_cap ? nw : static_cast<uint32_t>(chars_cap - at));
      w0 += nw;
      __syncthreads();  // the stores have read the window
    }
    turn(1);
  }
}

// ORs the bytes of label e into the window (cleared) at byte p.
__device__ __forceinline__ void label_or(PlainSmem& sm, uint32_t e, uint32_t p)
{
  static_assert(offsetof(PlainSmem, out) == sizeof(PlainSmem::lead), "the lead is the word before the window");
  const uint32_t sh = p & 3u;
  const uint32_t f  = sh ? 0u : 1u;                       // then the first pair of words makes nothing
  const uint32_t nb = sm.label_len[e] + sh + 4u * f;      // bytes from the first word ORed
  const uint32_t ph = 0u - sh;                            // the funnel takes it modulo 4
  uint32_t* const o = sm.lead + (4u + (p >> 2) - f);
  uint32_t carry    = 0;
#pragma unroll
  for (uint32_t h = 0; h < LABEL_BYTES / 16u; ++h) {
    if (h && !ballot(nb > 16u * h)) return;
    const u32x4 n = *reinterpret_cast<const u32x4*>(&sm.label[e][4u * h]);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t v = __builtin_amdgcn_alignbyte(n[j], carry, ph);
      carry            = n[j];
      if (16u * h + 4u * j < nb)
        __hip_atomic_fetch_or(o + 4u * h + j, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  if (nb > LABEL_BYTES)
    __hip_atomic_fetch_or(o + LABEL_BYTES / 4u, __builtin_amdgcn_alignbyte(0u, carry, ph), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_WORKGROUP);
}

// plain_chunk for a DICTIONARY segment of at most LABEL_ENTRIES entries of at most
// LABEL_BYTES bytes, and whether it was one: the entries go to LDS, whole words
// and zero past their ends, so that a row costs an index, a length and an OR for
// each word of its entry (8 Mi label rows: 57 us through memory, 189 vector
// instructions for 64 rows; here 36 us).
template <uint32_t RPT>
__device__ __forceinline__ bool label_chunk(const PlainArgs& args, PlainSmem& sm)
{
  const PlainArgs a   = uniform(args);
  const uint32_t tid  = threadIdx.x;
  const uint32_t w    = a.flags & FI_WIDTH;
  const uint32_t rows = a.rows;
  const uint8_t* bits = a.seg + 20;
  if (!w || bits + ((uint64_t{a.row_begin + rows} * w + 7u) >> 3) > a.seg + a.bytes_size) return false;
  uint32_t idx[RPT];
  {
    const uint64_t bit0          = uint64_t{a.row_begin} * w;
    const uintptr_t at           = reinterpret_cast<uintptr_t>(bits) + (bit0 >> 3);
    const uint32_t skew          = 8u * static_cast<uint32_t>(at & 3u) + static_cast<uint32_t>(bit0 & 7u);
    const gptr<const uint32_t> p = gbl(reinterpret_cast<const uint32_t*>(at & ~uintptr_t{3}));
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) {
      const uint32_t r = FSST_THREADS * i + tid;
      idx[i]           = bits32_inside(p, skew + (r < rows ? r : 0u) * w, w);
    }
  }
  // entry k is [dict_end - end[k], dict_end - end[k - 1]); 0 is NULL; one whose end
  // passes dict_end or falls below its start is empty
  uint32_t elen = 0, esrc = 0;
  if (tid != 0u && tid < a.ibc) {
    const uint8_t* e  = a.seg + a.ibo + 4ull * tid;
    const uint32_t e1 = ld_u32_any(e), e0 = ld_u32_any(e - 4);
    if (e1 >= e0 && e1 <= a.dict_end) {
      elen = e1 - e0;
      esrc = a.dict_end - e1;
    }
  }
  if (tid < LABEL_ENTRIES) {
    sm.label_len[tid] = static_cast<uint8_t>(elen);
    sm.label_src[tid] = esrc;
  }
  const bool longer = ballot(elen > LABEL_BYTES) != 0;
  if (lane_id() == 0u) sm.flag[tid / WAVE] = longer;
  __syncthreads();
  if (ballot(sm.flag[lane_id() % FSST_WAVES] != 0u)) return false;  // the same in every wave
  {  // half an entry a thread
    static_assert(LABEL_ENTRIES * 2u == FSST_THREADS && LABEL_BYTES == 32u, "16 bytes a thread");
    const uint32_t e = tid / 2u, h = 16u * (tid & 1u), l = sm.label_len[e];
    const uint32_t n = l > h ? (l - h < 16u ? l - h : 16u) : 0u;
    u32x4 v          = {0u, 0u, 0u, 0u};
    if (n) {
      const uint8_t* p             = a.seg + sm.label_src[e] + h;
      const uint32_t skew          = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p) & 3u);
      const gptr<const uint32_t> g = gbl(reinterpret_cast<const uint32_t*>(p - skew));
      const uint32_t last          = (skew + n - 1u) >> 2;
      uint32_t x[5];
#pragma unroll
      for (uint32_t j = 0; j < 5; ++j) x[j] = g[j < last ? j : last];
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t y = __builtin_amdgcn_alignbyte(x[j + 1], x[j], skew);
        v[j] = n >= 4u * j + 4u ? y : n > 4u * j ? y & ((1u << (8u * (n - 4u * j))) - 1u) : 0u;
      }
    }
    *reinterpret_cast<u32x4*>(&sm.label[e][h / 4u]) = v;
  }
  // output positions, as in plain_chunk
  const uint32_t wv = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(tid / WAVE)));
  uint32_t out[RPT];
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) {
    idx[i]             = FSST_THREADS * i + tid < rows && idx[i] < a.ibc ? idx[i] : 0u;
    const uint32_t len = sm.label_len[idx[i]];
    out[i]             = wave_incl_sum_u32(len);
    if (lane_id() == WAVE - 1u) sm.part[FSST_WAVES * i + wv] = out[i];
    out[i] -= len;
  }
  __syncthreads();
  static_assert(FSST_WAVES * RPT <= WAVE, "a lane per step and wave");
  const uint32_t mine = lane_id() < FSST_WAVES * RPT ? sm.part[lane_id()] : 0u;
  const uint32_t incl = wave_incl_sum_u32(mine);
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) out[i] += __builtin_amdgcn_readlane(incl - mine, FSST_WAVES * i + wv);
  const uint32_t T = __builtin_amdgcn_readlane(incl, WAVE - 1);
  fsst_lookback_publish(a.c, T, a.st, a.spin_limit);
  // one window if the chunk fits it, else one for each step of 512 rows
  static_assert(FSST_THREADS * LABEL_BYTES <= FSST_WINDOW, "a step fits the window");
  const bool whole = T <= FSST_WINDOW;
  if (whole) {
    window_clear(sm, T);
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < RPT; ++i) label_or(sm, idx[i], out[i]);
  }
  const uint64_t base     = fsst_lookback_wait(a.c, a.n_chunks, T, a.st, a.spin_limit, sm);  // synchronises the workgroup
  const gptr<int32_t> off = gbl(a.offsets) + a.col_row;
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) {
    const uint32_t r = FSST_THREADS * i + tid;
    if (r < rows) off[r] = static_cast<int32_t>(static_cast<uint32_t>(base) + out[i]);
  }
  if (a.c == a.n_chunks - 1u && tid == 0)
    gbl(a.offsets)[a.total_rows] = static_cast<int32_t>(static_cast<uint32_t>(base + T));
  auto store = [&](uint32_t w0, uint32_t n) {
    const uint64_t at = base + w0;
    if (at < a.chars_cap)
      window_store(sm, reinterpret_cast<uintptr_t>(a.chars) + at,
                   at + n <= a.chars_cap ? n : static_cast<uint32_t>(a.chars_cap - at));
  };
  if (whole) {
    store(0u, T);
    return true;
  }
#pragma unroll
  for (uint32_t i = 0; i < RPT; ++i) {
    const uint32_t lo = __builtin_amdgcn_readlane(incl - mine, FSST_WAVES * i);
    const uint32_t hi = i + 1u < RPT ? __builtin_amdgcn_readlane(incl - mine, FSST_WAVES * (i + 1u) % WAVE) : T;
    window_clear(sm, hi - lo);
    __syncthreads();
    label_or(sm, idx[i], out[i] - lo);
    __syncthreads();
    store(lo, hi - lo);
    __syncthreads();  // the stores have read the window
  }
  return true;
}

// Import the symbol table serialised at seg + symoff (at most
// FSST_SYMSTAGE bytes inside the segment are read; the rest read as zero)
// into `tab`, one code per thread (detail/fsst.cuh:50-96); returns the
// length of the calling thread's code.  A table whose version word does not
// match decodes every code to nothing.  Every thread of the block must call
// it.
template <uint32_t NT>
__device__ __forceinline__ uint32_t import_symtab(const uint8_t* seg, uint32_t bytes_size, uint32_t symoff, bool ok,
                                                  FsstSymTab* __restrict__ tab, FsstPrepSmem<NT>& sm)
{
  const uint32_t tid = threadIdx.x;
  __syncthreads();  // the previous segment's use of sm is done
  uint32_t sym_n = 0, sym_h = 0;
  if (ok) {
    sym_n = bytes_size - symoff;
    if (sym_n > FSST_SYMSTAGE) sym_n = FSST_SYMSTAGE;
    sym_h = block_issue<NT>(reinterpret_cast<uint32_t*>(sm.st), seg + symoff, sym_n);
  }
  __builtin_amdgcn_s_waitcnt(WAITCNT_VMEM_DONE);  // and for what the caller issued
  __syncthreads();
  uint32_t len = 0;
  uint64_t sym = 0;
  if (tid >= 256u) return 0;  // one code per thread (uniform per wave)
  if (ok) {
    auto sb = [&](uint32_t i) -> uint32_t { return i < sym_n ? sm.st[sym_h + i] : 0u; };
    uint64_t version = 0;
    for (uint32_t i = 0; i < 8; ++i) version |= static_cast<uint64_t>(sb(i)) << (8u * i);
    const uint32_t code = tid;
    if ((version >> 32) == FSST_VERSION && code < FSST_NSYM) {
      const uint32_t zt = sb(8) & 1u;
      uint32_t next_code = zt, pos = 17, found = 0;
      len = 8;
      sym = FSST_CORRUPT;
      if (zt && code == 0) {
        len   = 1;
        sym   = 0;
        found = 1;
      }
      // groups in code order: lengths 2,3,...,8 then 1
      for (uint32_t l = 1; l <= 8 && !found; ++l) {
        const uint32_t h  = l & 7u;
        const uint32_t sl = h + 1u;
        uint32_t cnt      = sb(9 + h);
        if (h == 0 && zt) cnt = (cnt - 1u) & 0xFFu;
        if (code >= next_code && code < next_code + cnt) {
          const uint32_t at = pos + (code - next_code) * sl;
          sym               = 0;
          for (uint32_t j = 0; j < sl; ++j) sym |= static_cast<uint64_t>(sb(at + j)) << (8u * j);
          len   = sl;
          found = 1;
        }
        next_code += cnt;
        pos += cnt * sl;
      }
    }
  }
  gbl(tab->sym)[tid] = sym;
  gbl(tab->len)[tid] = static_cast<uint8_t>(len);
  return len;
}

// LDS of a dictionary pre-pass: what fits of the dictionary is staged.
constexpr uint32_t DICT_STAGE = 32768;
template <uint32_t NT>
struct DfsstPrepSmem {
  FsstPrepSmem<NT> tab;
  __attribute__((aligned(16))) uint32_t dict[(DICT_STAGE + 64) / 4];
};

// Dictionary pre-pass of one DICT_FSST segment with the calling block: the
// entry byte offsets e_byte[0..dict_count] (scanned bit-packed lengths), for
// the FSST modes with more than one entry the symbol table and the decoded
// entry offsets (entry 0 empty), otherwise the byte offsets again, into
// e_dec; out = {decoded total, inline-NULL flag} and *pre = the bytes its
// predecoded entries take.  32-bit sums, as the reference's scans.
//
// Bound by latency, there being few dictionaries: the entries go to LDS beside
// the symbol table, two to a thread (66 dictionaries of 2000 entries: 22 us with
// four to a thread, each walked in memory; now 17 us).
template <uint32_t NT>
__device__ __forceinline__ void dfsst_prep_segment(const DictFsstSeg& d, uint32_t* __restrict__ e_byte,
                                                   uint32_t* __restrict__ e_dec, FsstSymTab* __restrict__ tab,
                                                   uint32_t* __restrict__ out, uint32_t* __restrict__ pre,
                                                   DfsstPrepSmem<NT>& dsm)
{
  constexpr uint32_t EPT = 2;  // entries of a thread
  FsstPrepSmem<NT>& sm   = dsm.tab;
  const uint32_t tid     = threadIdx.x;
  if (!d.valid) {  // uniform per block
    if (tid == 0) out[0] = out[1] = *pre = 0;
    return;
  }
  const uint8_t* seg  = d.bytes;
  const uint8_t* end  = seg + d.bytes_size;
  const bool fsst     = d.mode != 0u && d.dict_count > 1u;
  const uint8_t* dict = seg + d.off_dict;
  const uint32_t left = d.bytes_size > d.off_dict ? d.bytes_size - d.off_dict : 0u;
  const uint32_t bn   = !fsst ? 0u : left < DICT_STAGE ? left : DICT_STAGE;
  const uint32_t head = block_issue<NT>(dsm.dict, dict, bn);
  const uint32_t mylen = import_symtab(seg, d.bytes_size, d.off_symtab, fsst && d.off_symtab < d.bytes_size, tab, sm);
  if (tid < 256u) sm.len[tid] = static_cast<uint8_t>(tid == FSST_ESC ? 1u : mylen);
  __syncthreads();
  const uint8_t* slens = seg + d.off_slens;
  const uint32_t w     = d.slw;
  const bool inside    = w && uint64_t{d.off_slens} + ((uint64_t{d.dict_count} * w + 7u) >> 3) <= d.bytes_size;
  uint32_t carry_b = 0, carry_d = 0, first_len = 0;
  for (uint32_t k0 = 0; k0 < d.dict_count; k0 += EPT * NT) {
    uint32_t v[EPT], dl[EPT], sb = 0, sd = 0;
    const uint64_t bit0          = uint64_t{k0} * w;
    const uintptr_t at           = reinterpret_cast<uintptr_t>(slens) + (bit0 >> 3);
    const uint32_t skew          = 8u * static_cast<uint32_t>(at & 3u) + static_cast<uint32_t>(bit0 & 7u);
    const gptr<const uint32_t> p = gbl(reinterpret_cast<const uint32_t*>(at & ~uintptr_t{3}));
#pragma unroll
    for (uint32_t i = 0; i < EPT; ++i) {
      const uint32_t k = k0 + EPT * tid + i;
      if (inside) v[i] = bits32_inside(p, skew + (k < d.dict_count ? k - k0 : 0u) * w, w);  // uniform
      else v[i] = k < d.dict_count ? stream_bits32(slens, end, uint64_t{k} * w, w) : 0u;
      v[i] = k < d.dict_count ? v[i] : 0u;
      sb += v[i];
    }
    uint32_t tb = 0;
    uint32_t run = carry_b + block_excl_scan<NT / WAVE>(sb, sm.wave, &tb);
    const bool staged = ballot(uint64_t{run} + sb > bn) == 0;  // the wave's entries
#pragma unroll
    for (uint32_t i = 0; i < EPT; ++i) {
      const uint32_t k = k0 + EPT * tid + i;
      if (k < d.dict_count) e_byte[d.e_byte + k] = run;
      if (!fsst) {
        dl[i] = v[i];
      } else if (staged) {
        const uint32_t* ew = dsm.dict + ((head + run) >> 2);
        dl[i] = dfsst_entry_len([&](uint32_t j) { return ew[j]; }, (head + run) & 3u, v[i], v[i], sm.len);
      } else {
        const uint8_t* ep = dict + run;
        const GlobalWords gw(ep);
        dl[i] = dfsst_entry_len(gw, gw.skew, v[i], ep < end ? static_cast<uint64_t>(end - ep) : 0u, sm.len);
      }
      if (fsst && k == 0u) dl[i] = 0u;
      if (k == 0u) first_len = v[i];
      run += v[i];
      sd += dl[i];
    }
    uint32_t td = 0;
    uint32_t rd = carry_d + block_excl_scan<NT / WAVE>(sd, sm.wave, &td);
#pragma unroll
    for (uint32_t i = 0; i < EPT; ++i) {
      const uint32_t k = k0 + EPT * tid + i;
      if (k < d.dict_count) e_dec[d.e_byte + k] = rd;
      rd += dl[i];
    }
    carry_b += tb;
    carry_d += td;
  }
  if (tid == 0) {
    e_byte[d.e_byte + d.dict_count] = carry_b;
    e_dec[d.e_byte + d.dict_count]  = carry_d;
    out[0] = carry_d;
    out[1] = d.mode != 2u && d.dict_count > 1u && first_len == 0u;
    *pre   = fsst ? carry_d : 0u;
  }
}

// Bytes [o, lim) of `out`, appended up to eight at a time: whole words where
// they are the writer's alone, single bytes at both ends.
struct WordWriter {
  uint8_t* at;   // word the next byte falls in
  uint8_t* lim;
  uint64_t acc = 0;     // bytes from `at` on
  uint32_t fill, skip;  // of these, how many there are and how many are others'
  __device__ __forceinline__ WordWriter(uint8_t* o, uint8_t* l) : lim(l)
  {
    skip = fill = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(o) & 3u);
    at          = o - fill;
  }
  __device__ __forceinline__ bool room() const { return at + fill < lim; }
  __device__ __forceinline__ void put_bytes(uint32_t n)
  {
    for (uint32_t b = skip; b < n; ++b)
      if (at + b < lim) *gbl(at + b) = static_cast<uint8_t>(acc >> (8u * b));
  }
  __device__ __forceinline__ void append4(uint32_t v, uint32_t n)  // v is zero above its n <= 4 bytes
  {
    acc |= static_cast<uint64_t>(v) << (8u * fill);
    fill += n;
    if (fill < 4u) return;
    if (skip == 0u && at + 4 <= lim) *gbl(reinterpret_cast<uint32_t*>(at)) = static_cast<uint32_t>(acc);
    else put_bytes(4u);
    skip = 0;
    acc >>= 32;
    fill -= 4u;
    at += 4;
  }
  __device__ __forceinline__ void append(uint64_t v, uint32_t n)
  {
    append4(static_cast<uint32_t>(v), n < 4u ? n : 4u);
    if (n > 4u) append4(static_cast<uint32_t>(v >> 32), n - 4u);
  }
  __device__ __forceinline__ void finish()
  {
    while (room()) append(0u, 8u);  // zeros up to the limit
    put_bytes(fill);
  }
};

// Predecode the FSST entries k >= 1 of one segment into d.src at d.e[k]
// (exactly d.e[k + 1] - d.e[k] bytes; the byte of a trailing escape and
// bytes past the decoded ones are 0), entries strided over `stride`
// threads starting at `t`.
__device__ __forceinline__ void dfsst_predecode(const DictFsstSeg& d, const uint32_t* __restrict__ e_byte,
                                                const uint64_t* sym, const uint8_t* len, uint32_t t, uint32_t stride)
{
  const uint8_t* end  = d.bytes + d.bytes_size;
  const uint8_t* dict = d.bytes + d.off_dict;
  uint8_t* out        = const_cast<uint8_t*>(d.src);
  for (uint32_t k = 1u + t; k < d.dict_count; k += stride) {
    const uint32_t c0 = gbl(e_byte)[d.e_byte + k], c1 = gbl(e_byte)[d.e_byte + k + 1u];
    const uint32_t n  = c1 >= c0 ? c1 - c0 : 0u;
    uint64_t o        = gbl(d.e)[k];
    uint64_t lim      = gbl(d.e)[k + 1u];
    if (lim > d.src_size) lim = d.src_size;
    if (lim <= o) continue;
    const uint8_t* p    = dict + c0;
    const uint64_t in   = p < end ? static_cast<uint64_t>(end - p) : 0u;
    const uint32_t n_in = n < in ? n : static_cast<uint32_t>(in);
    WordWriter w(out + o, out + lim);
    const GlobalWords gw(p);
    bool esc = false;
    each_byte(gw, gw.skew, n_in, [&](uint32_t code) {
      if (!esc && code == FSST_ESC) {
        esc = true;
        return;
      }
      if (w.room()) w.append(esc ? code : sym[code], esc ? 1u : len[code]);
      esc = false;
    });
    // zeros past the segment: one may be an escape's byte, the others are code 0
    for (uint32_t z = n_in; z < n && w.room(); ++z) {
      w.append(esc ? 0u : sym[0], esc ? 1u : len[0]);
      esc = false;
    }
    w.finish();
  }
}

// Clears the bits of null-mask byte `b` (value m0) of rows that are NULL in their
// DICT_FSST range sg, whose descriptor is d: every row when the range is
// invalid, outside mode 2 those that select entry 0 (dict_fsst.cu:426-446).
__device__ __forceinline__ uint32_t dfsst_null_byte(uint32_t m, uint32_t row0, const FsstSeg& sg, const DictFsstSeg& d)
{
  if (d.valid && d.mode == 2u) return m;
  // rows [j0, j1) of the byte's eight
  const uint32_t j0 = sg.col_row > row0 ? sg.col_row - row0 : 0u;
  const uint64_t e  = uint64_t{sg.col_row} + sg.row_count - row0;
  const uint32_t j1 = e < 8u ? static_cast<uint32_t>(e) : 8u;
  if (j0 >= j1) return m;
  const uint32_t rows = (0xFFu >> (8u - (j1 - j0))) << j0;
  if (!d.valid) return m & ~rows;
  const uint8_t* bits = d.bytes + d.off_didx;
  const uint8_t* end  = d.bytes + d.bytes_size;
  const uint32_t w    = d.diw;
  const uint32_t sr   = row0 + j0 - sg.col_row;
  uint32_t null       = 0;
  if (w && bits + ((uint64_t{sr + (j1 - j0)} * w + 7u) >> 3) <= end) {
    const uint64_t bit0          = uint64_t{sr} * w;
    const uintptr_t at           = reinterpret_cast<uintptr_t>(bits) + (bit0 >> 3);
    const uint32_t skew          = 8u * static_cast<uint32_t>(at & 3u) + static_cast<uint32_t>(bit0 & 7u);
    const gptr<const uint32_t> p = gbl(reinterpret_cast<const uint32_t*>(at & ~uintptr_t{3}));
#pragma unroll
    for (uint32_t j = 0; j < 8u; ++j)
      null |= (bits32_inside(p, skew + (j < j1 - j0 ? j : 0u) * w, w) == 0u ? 1u : 0u) << j;
    null <<= j0;
  } else {
    for (uint32_t j = j0; j < j1; ++j)
      null |= (stream_bits32(bits, end, uint64_t{sr + j - j0} * w, w) == 0u ? 1u : 0u) << j;
  }
  return m & ~(null & rows);
}

// Range `si` with the calling NT-thread workgroup: its chunk descriptors
// into chunks[first_chunk + k]; for a segment, header checks
// (fsst.cu:79-87), the symbol table import, one code per thread
// (detail/fsst.cuh:50-96), into `tab`, and for each chunk k its
// compressed-length prefix bounds (fsst.cu:132-188) and flags into
// info[first_chunk + k].  Bytes past the segment read as zero; no symbol
// table parse reads past byte 2057.
template <uint32_t NT>
__device__ __forceinline__ void fsst_prep_segment(const FsstSeg sg, uint32_t si, FsstChunk* __restrict__ chunks,
                                                  FsstChunkInfo* __restrict__ info, FsstSymTab* __restrict__ tab,
                                                  FsstPrepSmem<NT>& sm)
{
  const uint32_t tid = threadIdx.x;
  const uint8_t* seg = sg.bytes;
  const uint8_t* end = seg + sg.bytes_size;
  const bool gap     = seg == nullptr;
  for (uint32_t k = tid; uint64_t{k} * sg.chunk_rows < sg.row_count; k += NT) {
    const uint32_t r0 = k * sg.chunk_rows;
    const uint32_t n  = sg.row_count - r0 < sg.chunk_rows ? sg.row_count - r0 : sg.chunk_rows;
    const FsstChunk fc{gap ? FSST_GAP : si, gap ? 0u : r0, n, sg.col_row + r0};
    *gbl(reinterpret_cast<u32x4*>(chunks + sg.first_chunk + k)) = __builtin_bit_cast(u32x4, fc);
  }
  if (gap) return;  // uniform: nothing else of a gap is read
  if (sg.codec == SDR_CODEC_DICTIONARY || sg.codec == SDR_CODEC_UNCOMPRESSED) {
    plain_prep_segment<NT>(sg, info);
    return;  // uniform per segment
  }
  if (sg.codec == SDR_CODEC_DICT_FSST) {  // bytes: the range's DictFsstSeg; pad: 1 if valid
    for (uint32_t k = tid; uint64_t{k} * sg.chunk_rows < sg.row_count; k += NT) {
      FsstChunkInfo ci{sg.bytes, 0u, 0u, 0u, FI_DFSST | (sg.pad ? FI_OK : 0u), 0u, 0u};
      const gptr<u32x4> dst = gbl(reinterpret_cast<u32x4*>(info + sg.first_chunk + k));
      const u32x8 cv        = __builtin_bit_cast(u32x8, ci);
      dst[0]                = cv.lo;
      dst[1]                = cv.hi;
    }
    return;  // uniform per segment
  }
  // The front of the segment, nearly always its whole length stream, goes to
  // LDS while the header that describes it arrives, the symbol table behind
  // it: two round trips.  (Each lane reading its fields' words from memory, one
  // dependent load after another, chunk by chunk, took 13 us for a row group
  // and 20 us for 956 segments; now 8.7 us and 18.5 us.)
  const uint32_t rows = sg.row_count;
  const uint32_t nch  = (rows + FSST_CHUNK_ROWS - 1u) / FSST_CHUNK_ROWS;
  const uint32_t wv   = tid / WAVE;
  const uint32_t lane = lane_id();
  bool ok             = false;
  uint32_t dict_end = 0, width = 0, symoff = 0, skew = 0;
  uint32_t b0 = 0, bn = sg.bytes_size < PREP_STAGE ? sg.bytes_size : PREP_STAGE;  // staged: bytes [b0, b0 + bn)
  __syncthreads();  // the previous segment's use of sm is done
  if (sg.bytes_size >= 16u) {
    skew     = block_issue<NT>(sm.fields, seg, bn);
    dict_end = su32(seg + 4);
    width    = su32(seg + 8);
    symoff   = su32(seg + 12);
    ok       = dict_end <= sg.bytes_size && symoff < dict_end && width <= 32u;
  }
  import_symtab(seg, sg.bytes_size, symoff, ok, tab, sm);  // waits for both

  // chunk bounds: wave w sums chunks w, w + NT / WAVE, ..., 16 fields per lane; a
  // stream that leaves the segment (malformed) is read from memory, bounded
  const uint64_t stream_end = 16u + ((uint64_t{rows} * width + 7u) >> 3);
  const bool inside         = ok && width && stream_end <= sg.bytes_size;
  uint32_t carry            = 0;
  for (uint32_t k0 = 0; k0 < nch;) {
    uint32_t cnt = nch - k0 < NT ? nch - k0 : NT;
    if (inside) {
      if (k0) {  // the next piece of the stream
        b0 = 16u + 128u * width * k0;  // 1024 fields take 128 * width bytes
        bn = stream_end - b0 < PREP_STAGE ? static_cast<uint32_t>(stream_end - b0) : PREP_STAGE;
        skew = block_stage<NT>(sm.fields, seg + b0, bn);
        __syncthreads();
      }
      if (b0 + bn < stream_end) {  // the chunks that are staged whole
        const uint32_t whole = (b0 + bn - 16u) / (128u * width) - k0;
        cnt                  = whole < cnt ? whole : cnt;
      }
    }
    if (ok)
      for (uint32_t k = k0 + wv; k < k0 + cnt; k += NT / WAVE) {
        const uint32_t r0 = k * FSST_CHUNK_ROWS;
        const uint32_t r1 = rows - r0 < FSST_CHUNK_ROWS ? rows : r0 + FSST_CHUNK_ROWS;
        const uint32_t f0 = r0 + 16u * lane < r1 ? r0 + 16u * lane : r1;
        const uint32_t f1 = f0 + 16u < r1 ? f0 + 16u : r1;
        bool hg           = false;
        uint32_t s        = 0;
        if (inside) {
          uint32_t mx      = 0;
          const uint64_t p = 8u * (uint64_t{skew} + 16u - b0) + uint64_t{f0} * width;  // modulo 2^64: f0's bit is staged
          s                = lds_fields_sum(sm.fields, static_cast<uint32_t>(p), f1 - f0, width, &mx);
          hg = mx >= ROW_HUGE;
        } else {
          s = fields_sum(seg + 16, end, f0, f1, width, &hg);
        }
        const uint32_t tt = __builtin_amdgcn_readlane(wave_incl_sum_u32(s), WAVE - 1);
        const bool any_hg = ballot(hg) != 0;
        if (lane == 0) {
          sm.sum[k - k0]  = tt;
          sm.huge[k - k0] = any_hg ? 1u : 0u;
        }
      }
    __syncthreads();
    const uint32_t v  = (ok && tid < cnt) ? sm.sum[tid] : 0u;
    uint32_t T        = 0;
    const uint32_t ex = block_excl_scan<NT / WAVE>(v, sm.wave, &T);
    if (tid < cnt) {
      const uint32_t k  = k0 + tid;
      const uint32_t r1 = rows - k * FSST_CHUNK_ROWS < FSST_CHUNK_ROWS ? rows : (k + 1u) * FSST_CHUNK_ROWS;
      uint32_t flags    = 0;
      if (ok) {
        flags = width | FI_OK;
        if (seg + 16 + ((uint64_t{r1} * width + 7u) >> 3) <= end) flags |= FI_LFAST;
        if (sm.huge[tid]) flags |= FI_HUGE;
      }
      FsstChunkInfo ci;
      ci.bytes      = seg;
      ci.c_lo       = carry + ex;
      ci.c_hi       = carry + ex + v;
      ci.dict_end   = dict_end;
      ci.flags      = flags;
      ci.bytes_size = sg.bytes_size;
      ci.pad        = 0;
      const gptr<u32x4> dst = gbl(reinterpret_cast<u32x4*>(info + sg.first_chunk + k));
      const u32x8 cv        = __builtin_bit_cast(u32x8, ci);
      dst[0]                = cv.lo;
      dst[1]                = cv.hi;
    }
    carry += T;
    k0 += cnt;
    __syncthreads();  // sum[], huge[] and fields[] are read before the next piece refills them
  }
}

// ---- chunk decode ----

// The compressed-length fields of rows r and r + 1 (0 past the chunk's rows);
// lw: the fields staged in LDS from bit bit0 when they all lie inside the
// segment (lfast), read without a branch around them.
__device__ __forceinline__ void fsst_fields2(const uint32_t* lw, uint32_t bit0, bool lfast, const uint8_t* seg,
                                             const uint8_t* end, uint32_t row_begin, uint32_t width, uint32_t r,
                                             uint32_t rows, uint32_t& a, uint32_t& b)
{
  if (lfast) {
    a = lds_bits32(lw, bit0 + r * width, width);
    b = lds_bits32(lw, bit0 + (r + 1u) * width, width);
  } else {
    a = stream_bits32(seg + 16, end, uint64_t{row_begin + r} * width, width);
    b = stream_bits32(seg + 16, end, uint64_t{row_begin + r + 1u} * width, width);
  }
  a = r < rows ? a : 0u;
  b = r + 1u < rows ? b : 0u;
}

// The segment's symbol table and the chunk's length fields on their way to
// LDS (LDS-direct loads); returns bit0 of fsst_fields2.
__device__ __forceinline__ uint32_t fsst_issue_front(FsstSmem& sm, const FsstSymTab* tab, bool lfast,
                                                     const uint8_t* seg, uint32_t row_begin, uint32_t rows,
                                                     uint32_t width)
{
  block_issue<FSST_THREADS>(reinterpret_cast<uint32_t*>(sm.sym), reinterpret_cast<const uint8_t*>(tab),
                            sizeof(FsstSymTab));
  if (!lfast) return 0;
  const uint64_t b0 = (uint64_t{row_begin} * width) >> 3;
  const uint64_t b1 = (uint64_t{row_begin + rows} * width + 7u) >> 3;
  const uint32_t h  = block_issue<FSST_THREADS>(reinterpret_cast<uint32_t*>(sm.out), seg + 16 + b0,
                                               static_cast<uint32_t>(b1 - b0));
  return h * 8u + static_cast<uint32_t>((uint64_t{row_begin} * width) & 7u);
}

// A row that has bytes starts at stage position y.
__device__ __forceinline__ void fsst_mark_row(FsstSmem& sm, uint32_t y)
{
  __hip_atomic_fetch_or(&sm.bits[y >> 5], 1u << (y & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// A run's chars from its walked groups: window by window when they pass
// FSST_WINDOW.  The window is cleared for the first one, and sm.dec[] is
// complete.  `get_base()` gives the chars offset of the run (it
// is called once, after the first window's ORs, and synchronises the
// workgroup).
template <class GetBase>
__device__ __forceinline__ void fsst_emit_run(FsstGroup (&gr)[GROUPS_PER_THR], FsstSmem& sm, uint32_t y_hi,
                                              const bool (&lits)[GROUPS_PER_THR], uint32_t T, uint8_t* chars,
                                              uint64_t chars_cap, GetBase&& get_base)
{
  const uint32_t tid = threadIdx.x;
  // the groups' bytes are taken apart again, not kept from the first walk in
  // a register each
#pragma unroll
  for (uint32_t k = 0; k < GROUPS_PER_THR; ++k)
#pragma unroll
    for (uint32_t d = 0; d < 4; ++d) __asm__ volatile("" : "+v"(gr[k].q[d]), "+v"(gr[k].p[d]));
  if (T <= FSST_WINDOW) {
#pragma unroll
    for (uint32_t k = 0; k < GROUPS_PER_THR; ++k)
      fsst_group_emit<false>(gr[k], sm, k * FSST_THREADS + tid, y_hi, lits[k], 0u);
    const uint64_t at = get_base();
    if (at < chars_cap)
      window_store(sm, reinterpret_cast<uintptr_t>(chars) + at,
                   at + T <= chars_cap ? T : static_cast<uint32_t>(chars_cap - at));
    return;
  }
  uint64_t base = 0;
#pragma unroll 1
  for (uint32_t w0 = 0; w0 < T; w0 += FSST_WINDOW) {
    const uint32_t nw = T - w0 < FSST_WINDOW ? T - w0 : FSST_WINDOW;
    if (w0) {
      __syncthreads();  // the stores have read the window
      window_clear(sm, nw);
      __syncthreads();
    }
#pragma unroll
    for (uint32_t k = 0; k < GROUPS_PER_THR; ++k)
      fsst_group_emit<true>(gr[k], sm, k * FSST_THREADS + tid, y_hi, lits[k], w0);
    if (w0) __syncthreads();
    else base = get_base();
    const uint64_t at = base + w0;
    if (at >= chars_cap) return;
    window_store(sm, reinterpret_cast<uintptr_t>(chars) + at,
                 at + nw <= chars_cap ? nw : static_cast<uint32_t>(chars_cap - at));
  }
}

// A chunk that is not one run: several runs, all walked for their decoded
// lengths first and again, each before it is emitted; or (malformed, or a row
// that no run holds) the row-wise path.  A call with scalar arguments, as
// plain_chunk.
__device__ __attribute__((noinline)) void fsst_chunk_runs(const uint8_t* seg, uint32_t bytes_size, uint32_t dict_end,
                                                          uint32_t flags, uint32_t c_lo, uint32_t c_hi,
                                                          uint32_t row_begin, uint32_t rows, uint32_t col_row,
                                                          const FsstSymTab* __restrict__ tab, uint32_t c,
                                                          uint32_t n_chunks, FsstState* __restrict__ st,
                                                          int32_t* __restrict__ offsets, uint8_t* __restrict__ chars,
                                                          uint64_t chars_cap, uint32_t total_rows, uint32_t spin_limit,
                                                          LdsPtr<FsstSmem> smp)
{
  FsstSmem& sm         = *(FsstSmem*)smp;
  const uint32_t tid   = threadIdx.x;
  fsst_lookback_begin(c, st, spin_limit);
  const uint8_t* end   = seg + bytes_size;
  const uint32_t width = flags & FI_WIDTH;
  const bool lfast     = width && (flags & FI_LFAST);
  const uint32_t bit0  = fsst_issue_front(sm, tab, lfast, seg, row_begin, rows, width);
  __builtin_amdgcn_s_waitcnt(WAITCNT_VMEM_DONE);
  __syncthreads();
  const uint32_t* lw = reinterpret_cast<const uint32_t*>(sm.out);
  const uint32_t r0 = 2u * tid, r1 = r0 + 1u;
  uint32_t cl0, cl1;
  fsst_fields2(lw, bit0, lfast, seg, end, row_begin, width, r0, rows, cl0, cl1);
  const uint32_t ne0 = cl0 ? 1u : 0u, ne1 = cl1 ? 1u : 0u;  // rows with bytes
  constexpr uint32_t RUN_MAX = FSST_CSTAGE - 15u;            // whatever the run's alignment
  const uint32_t wide        = cl0 > RUN_MAX || cl1 > RUN_MAX ? 1u << 16 : 0u;
  uint32_t x0, n0, x_all, n_all;
  block_excl_scan2(cl0 + cl1, ne0 + ne1 + wide, sm.wave, x0, n0, x_all, n_all);
  const uint32_t x1 = x0 + cl0, x2 = x1 + cl1;
  // Rows shorter than 1 MiB keep the prefix sums from wrapping, so they rise
  // from c_lo to c_hi.
  if ((flags & FI_HUGE) || c_hi < c_lo || c_hi > dict_end || n_all >> 16) {
    if (tid == 0) sm.comp[0] = c_lo;
    if (r0 < rows) sm.comp[r0 + 1u] = c_lo + x1;
    if (r1 < rows) sm.comp[r1 + 1u] = c_lo + x2;
    __syncthreads();
    const uint32_t T    = fsst_lengths_rows(sm, seg, dict_end, rows);
    const uint64_t base = fsst_lookback(c, n_chunks, T, st, spin_limit, sm);
    fsst_offsets(FsstChunk{0u, row_begin, rows, col_row}, c, n_chunks, rows, T, base, offsets, total_rows, sm);
    if (T == 0 || base >= chars_cap) return;
    fsst_emit_rows(sm, seg, dict_end, rows, T, base, chars, chars_cap);
    return;
  }
  n0 &= 0xFFFFu;
  const uint32_t n1 = n0 + ne0;
  if (tid == 0) sm.len[FSST_ESC] = LEN_ESC;
  // the run: rows [ra, rb), compressed bytes [xa, xb) of the chunk, nb rows
  // with bytes below rb; t_before decoded bytes of the chunk precede it
  uint32_t ra = 0, rb = 0, xa = 0, xb = 0, nb = 0, o0 = 0, o1 = 0;
  uint64_t t_before = 0, base = 0;
  bool measured     = false;
#pragma unroll 1
  for (;;) {
    // as many rows as fit; the last of them tells where the run ends
    __syncthreads();  // the previous run's users of LDS are done
    const bool f0       = r0 >= ra && r0 < rows && x1 - xa <= RUN_MAX;
    const bool f1       = r1 >= ra && r1 < rows && x2 - xa <= RUN_MAX;
    const uint32_t fits = static_cast<uint32_t>(__builtin_popcountll(ballot(f0)) + __builtin_popcountll(ballot(f1)));
    if (lane_id() == 0) sm.part[tid >> 6] = fits;
    for (uint32_t i = tid; i < FSST_CSTAGE / 32u; i += FSST_THREADS) sm.bits[i] = 0u;
    __syncthreads();
    rb = ra + __builtin_amdgcn_readlane(row_incl_sum_u32(sm.part[lane_id() & (FSST_WAVES - 1u)]), FSST_WAVES - 1u);
    if (r0 == rb - 1u || r1 == rb - 1u) {
      sm.wave[0] = r0 == rb - 1u ? x1 : x2;
      sm.wave[1] = r0 == rb - 1u ? n1 : n1 + ne1;
    }
    __syncthreads();
    xb = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(sm.wave[0])));
    nb = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(sm.wave[1])));
    const bool some      = xb != xa;
    const uintptr_t sa   = reinterpret_cast<uintptr_t>(seg + dict_end - c_lo - xb);
    const uint32_t c_h   = some ? static_cast<uint32_t>(sa & 15u) : 0u;
    const uint32_t y_hi  = some ? c_h + (xb - xa) : 0u;
    const uint8_t* stage = some ? reinterpret_cast<const uint8_t*>(sa - c_h)
                                : reinterpret_cast<const uint8_t*>(fsst_zero_group);
    FsstGroup gr[GROUPS_PER_THR];
    uint32_t prev[GROUPS_PER_THR];
    fsst_load_groups(gr, prev, stage, y_hi);
    const bool in0 = r0 >= ra && r0 < rb, in1 = r1 >= ra && r1 < rb;
    if (in0 && ne0) fsst_mark_row(sm, y_hi - (x1 - xa));
    if (in1 && ne1) fsst_mark_row(sm, y_hi - (x2 - xa));
    __syncthreads();
    bool lits[GROUPS_PER_THR];
    const uint32_t T = fsst_walk_lengths(gr, sm, prev, c_h, y_hi, stage, lits);
    __syncthreads();
    // as in fsst_chunk, for the rows that are the run's
    if (in0) {
      const uint32_t e0 = run_prefix(sm, y_hi - (x0 - xa)), e1 = run_prefix(sm, y_hi - (x1 - xa));
      o0 = static_cast<uint32_t>(t_before) + T - e0;
      if (ne0) sm.dec[nb - n0] = T - e0 - e1;
    }
    if (in1) {
      const uint32_t e1 = run_prefix(sm, y_hi - (x1 - xa)), e2 = run_prefix(sm, y_hi - (x2 - xa));
      o1 = static_cast<uint32_t>(t_before) + T - e1;
      if (ne1) sm.dec[nb - n1] = T - e1 - e2;
    }
    if (tid == 0) sm.dec[0] = T;
    __syncthreads();
    window_clear(sm, T < FSST_WINDOW ? T : FSST_WINDOW);
    __syncthreads();
    if (measured) {
      fsst_emit_run(gr, sm, y_hi, lits, T, chars, chars_cap, [&]() -> uint64_t {
        __syncthreads();
        return base + t_before;
      });
      if (rb >= rows) return;
    }
    t_before += T;
    ra = rb;
    xa = xb;
    if (rb < rows) continue;
    measured = true;
    fsst_lookback_publish(c, t_before, st, spin_limit);
    base = fsst_lookback_wait(c, n_chunks, t_before, st, spin_limit, sm);
    fsst_row_offsets(c, n_chunks, col_row, rows, t_before, base, o0, o1, offsets, total_rows);
    ra = xa  = 0;
    t_before = 0;
  }
}

// Decode chunk `c` (its position in the column's chunk order) with the
// calling workgroup.  Every thread must call it, after a workgroup barrier
// that follows any earlier use of `sm` (the callers' claim of the chunk ends
// with one), so the first loads issue without waiting.  `ci` and `tab` are the
// segment pre-pass's output for the chunk and its segment (unused for a chunk
// of uncovered rows).
//
// One memory round trip brings the symbol table and the chunk's
// compressed-length fields to LDS (LDS-direct loads) and its compressed bytes
// to registers; a second is the look-back for the column-wide chars offset.
__device__ __forceinline__ void fsst_chunk(const FsstChunk ch, const FsstChunkInfo ci, const FsstSymTab* tab,
                                           uint32_t c, uint32_t n_chunks, FsstState* __restrict__ st,
                                           int32_t* __restrict__ offsets, uint8_t* __restrict__ chars,
                                           uint64_t chars_cap, uint32_t total_rows, uint32_t spin_limit, FsstSmem& sm)
{
  const uint32_t tid  = threadIdx.x;
  const bool ok       = ch.seg != FSST_GAP && (ci.flags & FI_OK);
  const uint32_t rows = ch.rows;
  if (ok && (ci.flags & (FI_DICT | FI_UNC | FI_DFSST))) {  // uniform per chunk
    const PlainArgs args{ci.bytes,  ci.bytes_size, ci.dict_end, ci.flags, ci.c_lo, ci.c_hi, ch.row_begin, rows,
                         ch.col_row, c, n_chunks, st, offsets, chars, chars_cap, total_rows, spin_limit};
    plain_chunk<ROWS_PER_THR>(args, sm);
    return;
  }
  // No row has bytes: none of a segment's, or of one with a bad header, or none that
  // is not empty or NULL.  (Rows shorter than 1 MiB do not wrap their sum.)  1 M such
  // rows took 69 us, and 86 us in a batch, as a run of no bytes, which is called; so
  // 29 us and 39 us.
  if (!ok || (!(ci.flags & FI_HUGE) && ci.c_hi == ci.c_lo)) {
    const uint64_t base = fsst_lookback(c, n_chunks, 0u, st, spin_limit, sm);
    for (uint32_t r = tid; r < rows; r += FSST_THREADS)
      gbl(offsets)[ch.col_row + r] = static_cast<int32_t>(static_cast<uint32_t>(base));
    if (c == n_chunks - 1u && tid == 0) gbl(offsets)[total_rows] = static_cast<int32_t>(static_cast<uint32_t>(base));
    return;
  }
  // Rows are stored back to front ending at dict_end: the chunk's bytes are
  // [dict_end - c_hi, dict_end - c_lo).  One run holds them nearly always.
  const uint8_t* seg = ci.bytes;
  const uint32_t C   = ci.c_hi - ci.c_lo;
  const uintptr_t ca = reinterpret_cast<uintptr_t>(seg + ci.dict_end - ci.c_hi);
  const uint32_t c_h = static_cast<uint32_t>(ca & 15u);
  if ((ci.flags & FI_HUGE) || ci.c_hi < ci.c_lo || ci.c_hi > ci.dict_end || C > FSST_CSTAGE - c_h) {
    fsst_chunk_runs(seg, ci.bytes_size, ci.dict_end, ci.flags, ci.c_lo, ci.c_hi, ch.row_begin, rows, ch.col_row, tab, c,
                    n_chunks, st, offsets, chars, chars_cap, total_rows, spin_limit, (LdsPtr<FsstSmem>)(&sm));
    return;
  }
  const uint8_t* end   = seg + ci.bytes_size;
  const uint32_t width = ci.flags & FI_WIDTH;
  const bool lfast     = width && (ci.flags & FI_LFAST);
  const uint32_t y_hi  = c_h + C;
  const uint8_t* stage = reinterpret_cast<const uint8_t*>(ca - c_h);
  const uint32_t bit0  = fsst_issue_front(sm, tab, lfast, seg, ch.row_begin, rows, width);
  // The groups' loads go out last and unconditionally, so the wait below
  // leaves exactly these 2 * GROUPS_PER_THR loads in flight: the compressed
  // prefix runs while they arrive.
  __builtin_amdgcn_sched_barrier(0);
  FsstGroup gr[GROUPS_PER_THR];
  uint32_t prev[GROUPS_PER_THR];
  fsst_load_groups(gr, prev, stage, y_hi);
  for (uint32_t i = tid; i < FSST_CSTAGE / 32u; i += FSST_THREADS) sm.bits[i] = 0u;
  static_assert(GROUPS_PER_THR == 2, "the wait below leaves the groups' four loads in flight");
  __asm__ volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // ---- rows: compressed lengths (fsst.cu:132-188) and starts; thread t owns
  // rows 2t, 2t + 1 ----
  static_assert(ROWS_PER_THR == 2, "the staged path's row arithmetic");
  const uint32_t* lw = reinterpret_cast<const uint32_t*>(sm.out);
  uint32_t cl0, cl1;
  fsst_fields2(lw, bit0, lfast, seg, end, ch.row_begin, width, 2u * tid, rows, cl0, cl1);
  const uint32_t ne0 = cl0 ? 1u : 0u, ne1 = cl1 ? 1u : 0u;  // rows with bytes
  uint32_t all;
  const uint32_t pre = block_excl_scan_lds((cl0 + cl1) | (ne0 + ne1) << PK_LEN, sm.wave, &all);
  // stage positions: row 2t ends at ya, row 2t + 1 at yb and starts at yc
  const uint32_t ya = y_hi - (pre & ((1u << PK_LEN) - 1u)), yb = ya - cl0, yc = yb - cl1;
  if (ne0) fsst_mark_row(sm, yb);
  if (ne1) fsst_mark_row(sm, yc);
  if (tid == 0) sm.len[FSST_ESC] = LEN_ESC;
  lds_barrier();

  // ---- first walk ----
  bool lits[GROUPS_PER_THR];
  const uint32_t T = fsst_walk_lengths(gr, sm, prev, c_h, y_hi, stage, lits);
  // The aggregate is published now; the look-back's wait, and the offsets,
  // come once the first window's chars are in LDS.
  fsst_lookback_publish(c, T, st, spin_limit);
  lds_barrier();

  // ---- rows: output positions.  A row's chars follow those of the rows below
  // it, which lie after it in storage order ----
  const uint32_t e0 = run_prefix(sm, ya), e1 = run_prefix(sm, yb), e2 = run_prefix(sm, yc);
  const uint32_t k0 = (all >> PK_LEN) - (pre >> PK_LEN);  // one past row 2t's rank
  if (ne0) sm.dec[k0] = T - e0 - e1;        // output position T - e0, prefix e1
  if (ne1) sm.dec[k0 - ne0] = T - e1 - e2;
  if (tid == 0) sm.dec[0] = T;  // bytes before the first row's, which decode to nothing
  lds_barrier();
  window_clear(sm, T < FSST_WINDOW ? T : FSST_WINDOW);
  lds_barrier();

  // ---- second walk ----
  fsst_emit_run(gr, sm, y_hi, lits, T, chars, chars_cap, [&]() -> uint64_t {
    const uint64_t base = fsst_lookback_wait(c, n_chunks, T, st, spin_limit, sm);
    fsst_row_offsets(c, n_chunks, ch.col_row, rows, T, base, T - e0, T - e1, offsets, total_rows);
    return base;
  });
}

}  // namespace sdr
