// bf16 / fp16 MFMA paths of scatter2scatter and groupXtY for gfx950.
//
// One workgroup owns one BM x BN output tile that never straddles two experts and walks the contraction in
// slices of 64: global -> LDS directly (double buffered, or a ring of stages for the memory-bound small-row
// classes), or global -> registers -> LDS in the one-wave-per-SIMD form of the 256 x 256 class (mainloop_rs)
// -> MFMA 16x16x32 -> LDS-staged epilogue with 16-byte global accesses.
// Operands whose contraction axis is contiguous in memory ("direct": gathered X rows, weights stored
// (N,K)) sit in LDS as [row][64] with a 16-byte XOR swizzle and are read with ds_read_b128; operands
// whose contraction axis is strided ("transposed": weights stored (K,N), both operands of X^T dY) sit
// as [64][cols] and are read with ds_read_b64_tr_b16, which hands each lane four consecutive
// contraction elements of one column.
//
// Counterparts in the reference: _scatter2scatter + _compute_expert_block
// (scattermoe/kernels/ops.py:11-42, 50-118) and _groupXtY + _xty_and_bias (ops.py:242-366).
#pragma once
#include "common.hpp"

// Tunables (measured on the Mixtral-shape workload unless noted):
//   ROWS*_BELOW  average rows per expert under which the 32-, 64-, 128- and 256-row ring-buffered tile classes
//                are used (weight-streaming regime; see dispatch_s2s)
//   GM_RING      tile rows that visit a tile column back to back in the ring classes' order (1: -15 %, 4: -4 %)
//   STRIPE_BELOW average rows per expert under which the 256x256 class uses that order too (Mixtral shape, 1536
//                tokens: 1.68 -> 1.37 ms for the two forward launches; neutral at 4096, 2 % slower at 8192)
//   GM_S2S       row super-tiles per raster band of scatter2scatter (4: +3 % on the layer-2 shaped launches)
//   GM_XTY       the same for groupXtY (4: 1-2 % over unbanded on all three training workloads)
static constexpr int ROWS32_BELOW = 16, ROWS64_BELOW = 52, ROWS128_BELOW = 112, ROWS256_BELOW = 224;
static constexpr int GM_RING = 8;
static constexpr int STRIPE_BELOW = 1024;
// Whole launches below this many rows per expert are taken in chunks of neighbouring tiles per XCD (find_tile_chunked)
// where the experts' loads are even: an XCD then reads the token rows of its own experts only (column stripes: all rows,
// eight times over the fabric) and streams through one contiguous piece of the weights.  One chunk per XCD where the
// launch is a stream over the weights, else as many as there are rounds, so that the XCDs stay at neighbouring experts.
// Whole layers, us, stripes or super tiles -> chunks: 128 experts d = 2048, F = 768, forward of 60 / 200 / 2000 / 6000 /
// 10000 tokens 216 -> 205, 238 -> 227, 380 -> 350, 694 -> 677, 1032 -> 982; 32 experts d = F = 2880, 48 tokens 261 ->
// 252, training step of 1501 / 3000 tokens 1617 -> 1574, 2653 -> 2525; 8 experts d = 4096, F = 14336, training step of
// 6000 tokens 11996 -> 11728.  Uneven loads keep the other order (taken in chunks, loads falling as 1 / rank^1.8: 1607 -> 1681).
// Even is judged by tile rows or blocks of 64: experts of one tile row each may still differ in its height.  One launch with
// loads of 60 to 250 rows, experts in no order, chunks against stripes: 32 experts 2880 -> 2880 147 / 161, 2880 -> 2 x 2880 240 / 265;
// 64, 2048 -> 2048 144 / 152; 128, 2048 -> 1536 198 / 229, 768 -> 2048 122 / 128; with the experts sorted by load (the heavy
// ones then share an XCD) 161 / 154, 261 / 263, 150 / 159, 229 / 229, 138 / 124.
// Above 2048 rows per expert: even (128 experts x 2048 rows 8538 -> 8546).
static constexpr int CHUNK_BELOW = 3072;
static constexpr int GM_S2S = 4;
static constexpr int GM_XTY = 4;
static constexpr int XTY_GATHER_MAX_N = 6144;   // widest dY for which groupXtY gathers the rows of X itself
static constexpr int REMAINDER_ROWS = 128;      // last tiles of at most this many rows leave a product that cuts them off (cut_tails)
#include <type_traits>
#include <algorithm>
#include <math.h>

namespace smoe {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

static constexpr int BK = 64;               // contraction slice per stage

// Weight layouts whose kernels a source instantiates: 1 K-contiguous, 2 N-contiguous, 3 both (sources compile side by side)
#ifndef SMOE_LAYOUTS
#define SMOE_LAYOUTS 3
#endif

// Products are 16 x 16 x 32, not 32 x 32 x 16: the launches run at the power cap, and the smaller shape moves a quarter of the
// accumulators per instruction through the matrix cores for twice the operands.  Nothing but independent instructions on random
// operands in registers, one wave per SIMD: 1.80 PFLOP/s with 32 x 32 x 16, 2.01 with 16 x 16 x 32.  One of these adds up its
// 32 products in the order of two of those: the same bits.
template <typename T> struct Mfma;
template <> struct Mfma<bf16_t> {
  static __device__ __forceinline__ f32x4 run(i32x4 a, i32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ void in_place(i32x4 a, i32x4 b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ float sum8(i32x4 a) {
    const bf16x8 v = __builtin_bit_cast(bf16x8, a);
    return (((float)v[0] + (float)v[1]) + ((float)v[2] + (float)v[3])) +
           (((float)v[4] + (float)v[5]) + ((float)v[6] + (float)v[7]));
  }
};
template <> struct Mfma<f16_t> {
  static __device__ __forceinline__ f32x4 run(i32x4 a, i32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ void in_place(i32x4 a, i32x4 b, f32x4& c) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  }
  static __device__ __forceinline__ float sum8(i32x4 a) {
    const f16x8 v = __builtin_bit_cast(f16x8, a);
    return (((float)v[0] + (float)v[1]) + ((float)v[2] + (float)v[3])) +
           (((float)v[4] + (float)v[5]) + ((float)v[6] + (float)v[7]));
  }
};

// The accumulators of a 32 x 32 block of the output: four 16 x 16 products, q[2 r + c] the one at (16 r, 16 c).  The MFMAs are
// issued with the operands swapped (column operand first), so a lane holds, of group g, four consecutive columns of one row.
struct Block {
  f32x4 q[4];
  __device__ __forceinline__ float operator[](int e) const { return q[e >> 2][e & 3]; }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int g = 0; g < 4; ++g) q[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  }
};
__device__ __forceinline__ int block_row(int lane, int g) { return 16 * (g >> 1) + (lane & 15); }
__device__ __forceinline__ int block_col(int lane, int g) { return 16 * (g & 1) + 4 * (lane >> 4); }

typedef __attribute__((address_space(3))) char lds_char;

__device__ __forceinline__ unsigned lds_address(const char* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
__device__ __forceinline__ unsigned wave_uniform_id() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}
__device__ __forceinline__ i32x4 lds_read16(const char* p) { return *(const i32x4*)p; }
__device__ __forceinline__ void lds_write16(char* p, i32x4 v) { *(i32x4*)p = v; }
__device__ __forceinline__ s16x4 lds_read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
}

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void glb_void_t;

// 16 bytes per lane straight from global memory into LDS: lane i of the wave lands at dst + 16*i.
// Issued as inline assembly on purpose: for the builtin the compiler assumes that every later LDS read
// may alias the in-flight transfer and waits for it (vmcnt(0)) before the first ds_read, which would
// serialise the prefetch of slice k+1 with the MFMAs of slice k.  The main loop waits explicitly instead.
// `lds_addr` is the wave-uniform byte address inside the workgroup's LDS allocation; the global address is
// a wave-uniform 64-bit base (scalar registers) plus a 32-bit per-lane byte offset.  This addressing form
// matters: the same load with a full 64-bit address in each lane costs the issuing wave so much issue time
// that the matrix pipe starves (measured: +50% run time for 8 such loads per 32 MFMAs, against no
// measurable cost for the scalar-base form).
// STREAM: the non-temporal hint, for an operand the launch reads exactly once (the weights of the memory-bound
// classes), so that it does not displace the rows that are read again and again.
template <bool STREAM = false>
__device__ __forceinline__ void load_to_lds16(const char* base_uniform, unsigned off, unsigned lds_addr) {
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(lds_addr), "v"(off), "s"(base_uniform)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds_addr), "v"(off), "s"(base_uniform)
                 : "memory", "m0");
}
__device__ __forceinline__ const char* make_uniform(const char* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (const char*)(((uint64_t)hi << 32) | lo);
}

// Both operand kinds fill a 64-deep LDS tile of EXT*128 bytes in LINEAR order of 16-byte pieces: piece
// p = j*NT + t is copied by thread t in round j (a wave's 64 pieces are contiguous, which is what the
// direct-to-LDS load needs).  Which global piece lands in LDS piece p is where the two kinds differ:
// the XOR swizzles below are applied on the global side.

// ---- operand with contiguous contraction axis: LDS tile [EXT][64], 128 B per row ------------------------
// piece p = (row, phys) holds contraction chunk c = phys ^ f(row).  A ds_read_b128 takes its lanes in groups of 16 that are not
// consecutive (0-3, 12-15, 20-23, 24-27; 4-11, 16-19, 28-31; ...): of a fragment of 16 rows, eight rows of one chunk and the eight
// others of the chunk next to it, which this f puts into 16 different 16-byte bank groups (16 cycles per fragment with four
// waves reading; 32 with an f that separates 16 rows of one chunk).
__device__ __forceinline__ int direct_swz(int row) { return row & 7; }

template <int EXT, int NT, bool STREAM = false>
struct DirectOp {
  static constexpr int PIECES = EXT * 8;
  static constexpr int R = PIECES / NT;
  static constexpr int LDS_BYTES = EXT * 128;
  static constexpr int DS_PER_FRAG = 1;
  static_assert(PIECES % NT == 0, "tile must be a whole number of rounds");
  const char* base;        // wave-uniform global address all rows are relative to
  unsigned off[R];         // byte offset of this thread's piece of load slot j at contraction 0
  // Load slot j carries round (j + rot) % R of the tile.  The workgroups of a super tile that share a panel use
  // different rotations, each starting with the rows it is the designated first toucher of: those L2 misses
  // then start earliest, and the other sharers ask for the same lines later in their own queues, when the
  // fill is under way or done, instead of piling onto a miss that has only just been issued.
  int rot = 0;
  __device__ __forceinline__ int rnd(int j) const { const int r = j + rot; return r >= R ? r - R : r; }
  // `row_off(row)` returns the byte offset (from `b`) of element (row, k = 0) of the tile's row `row`
  template <typename F>
  __device__ __forceinline__ void init(const char* b, F row_off) {
    base = make_uniform(b);
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int p = rnd(j) * NT + t, row = p >> 3;
      off[j] = (unsigned)row_off(row) + (((p & 7) ^ direct_swz(row)) << 4);
    }
  }
  __device__ __forceinline__ void issue_one(unsigned tile, int k0, int j) const {
    load_to_lds16<STREAM>(base + (int64_t)k0 * 2, off[j], tile + wave_uniform_id() * 1024 + rnd(j) * NT * 16);
  }
  // The same pieces into registers: what the loads of a slice have in common, here its byte offset (whole slices only; past the
  // last one: that one again), and where a piece belongs in the LDS tile
  typedef int Slice;
  __device__ __forceinline__ Slice slice(int k0, int kend) const { return min(k0, kend - BK) * 2; }
  __device__ __forceinline__ i32x4 load_piece(Slice s, int j) const {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, -1, 0x00020000);
    return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off[j], s, STREAM ? 2 : 0));
  }
  __device__ __forceinline__ int piece_lds(int j) const { return (rnd(j) * NT + (int)threadIdx.x) * 16; }
  __device__ __forceinline__ void issue(unsigned tile, int k0) const {
#pragma unroll
    for (int j = 0; j < R; ++j) issue_one(tile, k0, j);
  }
  // Partial last slice: pieces past `kend` are fetched from contraction 0 of the same row (always valid
  // memory) and overwritten with zeros by the same thread once its loads have landed.
  __device__ __forceinline__ void issue_tail_one(unsigned tile, int k0, int kend, int j) const {
    const int p = rnd(j) * NT + threadIdx.x;
    const int c = (p & 7) ^ direct_swz(p >> 3);
    const bool ok = k0 + c * 8 < kend;
    load_to_lds16<STREAM>(base, ok ? off[j] + (unsigned)k0 * 2 : off[j] - (c << 4),
                  tile + wave_uniform_id() * 1024 + rnd(j) * NT * 16);
  }
  __device__ __forceinline__ void issue_tail(unsigned tile, int k0, int kend) const {
#pragma unroll
    for (int j = 0; j < R; ++j) issue_tail_one(tile, k0, kend, j);
  }
  __device__ __forceinline__ void zero_tail(char* tile, int k0, int kend) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int p = rnd(j) * NT + t;
      const int c = (p & 7) ^ direct_swz(p >> 3);
      if (k0 + c * 8 >= kend) lds_write16(tile + p * 16, i32x4{0, 0, 0, 0});
    }
  }
  // fragment of MFMA operand rows [base, base+16), contraction step ks (32 elements)
  static __device__ __forceinline__ i32x4 frag(const char* tile, int base, int ks) {
    const int l = lane_id();
    return lds_read16(tile + (base + (l & 15)) * 128 + (((4 * ks + (l >> 4)) ^ direct_swz(l & 15)) << 4));
  }
  // only operands that gather their contraction rows have anything to do here (see TransOp)
  __device__ __forceinline__ void fetch_rows(int, int) {}
  __device__ __forceinline__ void stage_rows(int) {}
  __device__ __forceinline__ void take_rows(int) {}
};

// ---- operand with strided contraction axis: LDS tile [64][EXT], read transposed --------------------------
// Row kr of the tile is EXT*2 bytes = G granules of 64 B (32 columns).  A ds_read_b64_tr_b16 phase touches
// half a granule (16 columns) in 4 consecutive rows and in the 4 rows 8 further down; storing granule g of row kr at position
// g ^ (kr & 3), its halves exchanged in every second 8 rows, spreads those 8 accesses over all 64 banks.
__device__ __forceinline__ int trans_piece(int kr, int phys) {      // logical 16-byte piece of row kr at position phys
  return phys ^ ((kr & 3) << 2) ^ ((kr >> 2) & 2);
}
// GATHER: the contraction rows are not consecutive in memory but picked through an index vector (row r of the
// operand is row rows[r] / fan of the source matrix).  The 64 rows of a slice are looked up once per workgroup, not
// once per thread (vector-ALU work in this loop comes straight out of the matrix pipe's time): thread t < 64 fetches
// the index of row t one slice ahead (`fetch_rows`, an ordinary load that the main loop's wait covers), turns it into
// a byte offset and puts it into LDS before the loop's barrier (`stage_rows`); after the barrier every thread picks
// the offsets of its own load slots up from there (`take_rows`).
// LEAN: one offset register for all load slots whose pieces differ by whole rows only, the rows between them added in scalar
// registers (weight gradients: 128 registers per wave, or 256 accumulators, leave no room for one per slot).
template <int EXT, int NT, bool STREAM = false, bool GATHER = false, bool LEAN = false>
struct TransOp {
  static constexpr int CPR = EXT / 8;                  // 16-byte pieces per contraction row
  static constexpr int PIECES = 64 * CPR;
  static constexpr int R = PIECES / NT;
  static constexpr int RS = EXT * 2;                   // LDS row stride, bytes
  static constexpr int DS_PER_FRAG = 2;
  static constexpr int LDS_BYTES = 64 * RS;
  static_assert(PIECES % NT == 0 && EXT % 128 == 0, "unsupported transposed tile width");
  const char* base;    // wave-uniform global address of (contraction 0, column 0 of the tile)
  static constexpr int SLOT_ROWS = NT / CPR;           // contraction rows between load slots
  static constexpr int OFFS = LEAN && !GATHER ? (SLOT_ROWS % 16 == 0 ? 1 : 2) : R;
  static_assert(SLOT_ROWS % 8 == 0 || OFFS == R, "two kinds of rows");
  unsigned off[OFFS];  // byte offset of this thread's piece of load slot j within the first slice
                       // (GATHER: within the slice that is issued next)
  // (rot is 0 where OFFS < R) what load slot j adds to off[j % OFFS]
  __device__ __forceinline__ unsigned slot_off(int j) const { return OFFS == R ? 0u : (unsigned)(j / OFFS * OFFS * SLOT_ROWS) * (unsigned)ld; }
  int rot = 0;         // load slot j carries round (j + rot) % R (see DirectOp)
  __device__ __forceinline__ int rnd(int j) const { const int r = j + rot; return r >= R ? r - R : r; }
  int64_t ld;          // bytes between contraction rows
  // GATHER only
  const int64_t* rows; // wave-uniform: index vector, already offset to the first contraction row
  unsigned fan;
  unsigned colb;       // byte offset of this thread's pieces inside their contraction rows (the rows of its load slots
                       // differ by multiples of 16, which the swizzle does not see)
  static_assert(!GATHER || NT / CPR % 16 == 0, "one column offset per thread");
  unsigned next_row;   // thread t < 64: index of contraction row t of the slice after the one being issued
  unsigned* srow;      // LDS, [2][64]: byte offsets of the rows of the slice to be issued next, by slice parity
  // contraction row inside a slice that load slot j of this thread carries
  __device__ __forceinline__ int slot_row(int j) const { return (rnd(j) * NT + (int)threadIdx.x) / CPR; }
  // columns >= valid_cols are clamped to column 0 (they only feed outputs that are never stored)
  __device__ __forceinline__ void init(const char* b, int64_t ld_bytes, int valid_cols) {
    init_cols(b, ld_bytes, [&](int tc) { return tc < valid_cols ? tc : 0; });
  }
  // `col_of(tc)`: element column (relative to `b`, a multiple of 8, always inside the allocation) that tile
  // column tc (a multiple of 8) is fetched from
  template <typename F>
  __device__ __forceinline__ void init_cols(const char* b, int64_t ld_bytes, F col_of) {
    base = make_uniform(b);
    ld = ld_bytes;
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < OFFS; ++j) {
      const int p = rnd(j) * NT + t;
      const int kr = p / CPR, phys = p % CPR;
      const int cc = trans_piece(kr, phys);
      if constexpr (GATHER) colb = (unsigned)col_of(cc * 8) * 2;
      else off[j] = (unsigned)(kr * ld_bytes) + (unsigned)col_of(cc * 8) * 2;
    }
  }
  // GATHER: `b` is (row 0, column 0 of the tile) of the SOURCE matrix, `r` the index vector at the operand's first
  // contraction row, `klen` the number of contraction rows, `lds_rows` 2 x 64 words of LDS.  Ends with the first
  // slice's offsets taken (one workgroup barrier inside).
  __device__ __forceinline__ void init_gather(const char* b, int64_t ld_bytes, int valid_cols, const int64_t* r,
                                              int fan_out, int klen, unsigned* lds_rows) {
    rows = (const int64_t*)make_uniform((const char*)r);
    fan = (unsigned)fan_out;
    srow = lds_rows;
    init(b, ld_bytes, valid_cols);
    fetch_rows(0, klen);
    stage_rows(0);
    __syncthreads();
    take_rows(0);
  }
  // index of row t of the slice at contraction k0 (rows past the end repeat the last row: their data is zeroed in LDS)
  __device__ __forceinline__ void fetch_rows(int k0, int klen) {
    if constexpr (GATHER) {
      if (wave_uniform_id() == 0) {
        int r = k0 + (int)threadIdx.x;
        r = r < klen ? r : klen - 1;
        next_row = r >= 0 ? (unsigned)rows[r] : 0u;
      }
    }
  }
  // before the barrier of the iteration that issues slice number `slice`
  __device__ __forceinline__ void stage_rows(int slice) {
    if constexpr (GATHER) {
      if (wave_uniform_id() == 0) srow[(slice & 1) * 64 + threadIdx.x] = (unsigned)((int64_t)(next_row / fan) * ld);
    }
  }
  // after that barrier
  __device__ __forceinline__ void take_rows(int slice) {
    if constexpr (GATHER) {
#pragma unroll
      for (int j = 0; j < R; ++j) off[j] = srow[(slice & 1) * 64 + slot_row(j)] + colb;
    }
  }
  __device__ __forceinline__ void issue_one(unsigned tile, int k0, int j) const {
    if constexpr (GATHER) load_to_lds16<STREAM>(make_uniform(base), off[j], tile + wave_uniform_id() * 1024 + rnd(j) * NT * 16);
    else load_to_lds16<STREAM>(base + (int64_t)k0 * ld + slot_off(j), off[j % OFFS], tile + wave_uniform_id() * 1024 + rnd(j) * NT * 16);
  }
  // The same pieces into registers (not for gathered rows): what the loads of a slice have in common, here a buffer descriptor
  // that ends with row kend - 1, so that contraction rows from there on read as zeros (a row's pieces lie inside its first `ld`
  // bytes; past the last slice: an empty one), and where a piece belongs in the LDS tile
  struct Slice { const char* base; int bytes; };
  __device__ __forceinline__ Slice slice(int k0, int kend) const {
    return Slice{make_uniform(base + (int64_t)k0 * ld), __builtin_amdgcn_readfirstlane(min(max(kend - k0, 0), BK) * (int)ld)};
  }
  __device__ __forceinline__ i32x4 load_piece(Slice s, int j) const {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)s.base, 0, s.bytes, 0x00020000);
    return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off[j % OFFS] + slot_off(j)), 0, STREAM ? 2 : 0));      // (a scalar offset would come off the range)
  }
  __device__ __forceinline__ int piece_lds(int j) const { return (rnd(j) * NT + (int)threadIdx.x) * 16; }
  __device__ __forceinline__ void issue(unsigned tile, int k0) const {
#pragma unroll
    for (int j = 0; j < R; ++j) issue_one(tile, k0, j);
  }
  // Partial last slice: contraction rows past `kend` are fetched from row 0 of the slice (always valid
  // memory) and overwritten with zeros by the same thread once its loads have landed.
  __device__ __forceinline__ void issue_tail_one(unsigned tile, int k0, int kend, int j) const {
    if constexpr (GATHER) {
      issue_one(tile, k0, j);          // rows past the end already point at the last valid row
    } else {
      const int kr = slot_row(j);
      const bool ok = k0 + kr < kend;
      load_to_lds16<STREAM>(base + (int64_t)k0 * ld, off[j % OFFS] + slot_off(j) - (ok ? 0u : (unsigned)(kr * ld)),
                    tile + wave_uniform_id() * 1024 + rnd(j) * NT * 16);
    }
  }
  __device__ __forceinline__ void issue_tail(unsigned tile, int k0, int kend) const {
#pragma unroll
    for (int j = 0; j < R; ++j) issue_tail_one(tile, k0, kend, j);
  }
  __device__ __forceinline__ void zero_tail(char* tile, int k0, int kend) const {
    const int t = threadIdx.x;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int p = rnd(j) * NT + t;
      if (k0 + p / CPR >= kend) lds_write16(tile + p * 16, i32x4{0, 0, 0, 0});
    }
  }
  // Each 16-lane block transposes a 4 (contraction) x 16 (columns) patch: lane r of the block points at
  // contraction row r/4, columns 4*(r%4)..+3 and receives column r, contraction 0..3.  Block b covers the contraction
  // elements 8*b..; a second read 4 rows further down completes the 8 elements per lane the MFMA expects
  // (k = 8*(lane/16) + 0..7).
  static __device__ __forceinline__ i32x4 frag(const char* tile, int base, int ks) {
    const int l = lane_id();
    const int b = l >> 4, r = l & 15;
    const int kr = ks * 32 + 8 * b + (r >> 2);
    const int unit = (base >> 4) ^ ((r >> 2) << 1) ^ (b & 1);      // 32 bytes; (kr & 3) == r >> 2, (kr >> 3 & 1) == (b & 1)
    const char* p = tile + kr * RS + (unit << 5) + (r & 3) * 8;
    const s16x4 lo = lds_read_tr(p);
    const s16x4 hi = lds_read_tr(p + 4 * RS);
    const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(i32x4, v);
  }
};

// 16 bytes per lane from global memory into LDS through a buffer descriptor: as load_to_lds16, but a lane whose offset lies
// beyond the descriptor's range reads zeros (the rows behind an expert's last one, without a branch and without a second
// write to LDS).  `soff`: a scalar byte offset on top of the lanes' own.
__device__ __forceinline__ void buffer_to_lds16(i32x4 rsrc, unsigned off, unsigned soff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_addr), "v"(off), "s"(rsrc), "s"(soff)
               : "memory", "m0");
}
__device__ __forceinline__ i32x4 buffer_rsrc(const void* base, unsigned bytes) {
  const uint64_t v = (uint64_t)base;
  i32x4 r = {(int)__builtin_amdgcn_readfirstlane((unsigned)v), (int)__builtin_amdgcn_readfirstlane((unsigned)(v >> 32)),
             (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000};
  asm volatile("s_nop 4" : "+s"(r));      // an assembly load may follow: five wait states behind the instructions above
  return r;
}

// A lane offset that every descriptor of a weight gradient's gathered or short operand rejects, with any instruction or scalar offset on top of it (ranges stay
// below 2 GiB: the launchers check).
static constexpr unsigned OUT_OF_RANGE = 0x80000000u;
// ---- operand with strided contraction axis whose contraction may end anywhere (weight gradients of mainloop_pair) --------
// The LDS layout of TransOp, filled through a buffer descriptor that ends with the last contraction row: what lies behind it
// reads as zeros, without a pass over LDS afterwards.  GATHER: row r of the operand is row rows[r] / fan of the source matrix;
// lane t of every wave looks up row t of a slice, two slices ahead of its loads (fetch_rows, an ordinary load that the main
// loop's wait covers), turns it into a byte offset while the slice before is multiplied (stage_rows), and the lanes pick the
// offsets of their own pieces from each other (take_rows): no LDS, no barrier.
template <int EXT, int NT, bool GATHER>
struct RowsOp {
  typedef TransOp<EXT, NT> Layout;
  static constexpr int R = Layout::R, LDS_BYTES = Layout::LDS_BYTES, DS_PER_FRAG = Layout::DS_PER_FRAG, CPR = Layout::CPR;
  static_assert(NT / CPR % 8 == 0, "one column offset per thread, or one for each of two kinds of load slots");
  static constexpr int COLS = NT / CPR % 16 == 0 ? 1 : 2;
  const char* base;        // wave-uniform: (contraction 0, column 0 of the tile); GATHER: of the source matrix
  i32x4 rsrc;              // of the slice to be issued next
  unsigned off[R];
  unsigned ld, colb[COLS]; // bytes (of load slot j: colb[j % COLS])
  int klen;
  // GATHER only
  const int64_t* rows;
  unsigned fan, next_row, row_off;
  __device__ __forceinline__ void init_cols(const char* b, int64_t ld_bytes, int valid_cols, int k) {
    base = make_uniform(b);
    ld = (unsigned)ld_bytes;
    klen = k;
#pragma unroll
    for (int j = 0; j < COLS; ++j) {
      const int tc = trans_piece((j * NT + (int)threadIdx.x) / CPR, (int)threadIdx.x % CPR) * 8;
      colb[j] = tc < valid_cols ? tc * 2 : 0;              // (such columns only feed outputs that are never stored)
    }
  }
  __device__ __forceinline__ void init(const char* b, int64_t ld_bytes, int valid_cols, int k) {
    init_cols(b, ld_bytes, valid_cols, k);
#pragma unroll
    for (int j = 0; j < R; ++j) off[j] = (unsigned)((j * NT + (int)threadIdx.x) / CPR) * ld + colb[j % COLS];
    take_rows(0);
  }
  // `span`: bytes from `b` to the end of the source matrix
  __device__ __forceinline__ void init_gather(const char* b, int64_t ld_bytes, int valid_cols, int k, const int64_t* r,
                                              int fan_out, unsigned span) {
    init_cols(b, ld_bytes, valid_cols, k);
    rows = r;
    fan = (unsigned)fan_out;
    next_row = 0;
    rsrc = buffer_rsrc(base, span);
    fetch_rows(0);
    const unsigned first = next_row;
    fetch_rows(BK);
    const unsigned second = next_row;
    fetch_rows(2 * BK);
    const unsigned third = next_row;
    next_row = first;
    stage_rows(0);
    take_rows(0);
    next_row = second;
    stage_rows(1);
    next_row = third;
  }
  // row indices of the slice at contraction k0
  __device__ __forceinline__ void fetch_rows(int k0) {
    if constexpr (GATHER) {
      const int r = k0 + lane_id();
      if (r < klen) next_row = (unsigned)rows[r];
    }
  }
  // what has been fetched becomes the offsets of slice number `slice`
  __device__ __forceinline__ void stage_rows(int slice) {
    if constexpr (GATHER) row_off = slice * BK + lane_id() < klen ? next_row / fan * ld : OUT_OF_RANGE;
  }
  // slice number `slice` is the next to be issued
  __device__ __forceinline__ void take_rows(int slice) {
    if constexpr (GATHER) {
      asm volatile("" : "+v"(next_row));                   // (the compiler's wait for it: here, with nothing in flight)
#pragma unroll
      for (int j = 0; j < R; ++j)
        off[j] = (unsigned)__builtin_amdgcn_ds_bpermute((j * NT + (int)threadIdx.x) / CPR * 4, (int)row_off) + colb[j % COLS];
    } else {
      const int left = klen - slice * BK;
      rsrc = buffer_rsrc(base + (int64_t)slice * BK * ld, left > 0 ? (unsigned)min(left, BK) * ld : 0u);
    }
  }
  __device__ __forceinline__ void issue_one(unsigned tile, int, int j) const {
    buffer_to_lds16(rsrc, off[j], 0, tile + wave_uniform_id() * 1024 + j * NT * 16);
  }
  static __device__ __forceinline__ i32x4 frag(const char* tile, int b, int ks) { return Layout::frag(tile, b, ks); }
};

// One slice of both operands, load slots interleaved (A0 B0 A1 B1 ...) so that the rows each operand starts
// with (see `rot`) are requested first.
template <class AOp, class BOp>
__device__ __forceinline__ void issue_slice(const AOp& A, const BOp& B, unsigned dst, int k0) {
  constexpr int RM = AOp::R > BOp::R ? AOp::R : BOp::R;
#pragma unroll
  for (int j = 0; j < RM; ++j) {
    if (j < AOp::R) A.issue_one(dst, k0, j);
    if (j < BOp::R) B.issue_one(dst + AOp::LDS_BYTES, k0, j);
  }
}
template <class AOp, class BOp>
__device__ __forceinline__ void issue_slice_tail(const AOp& A, const BOp& B, unsigned dst, int k0, int kend) {
  constexpr int RM = AOp::R > BOp::R ? AOp::R : BOp::R;
#pragma unroll
  for (int j = 0; j < RM; ++j) {
    if (j < AOp::R) A.issue_tail_one(dst, k0, kend, j);
    if (j < BOp::R) B.issue_tail_one(dst + AOp::LDS_BYTES, k0, kend, j);
  }
}

// WG_: workgroups per CU the registers have to leave room for (LDS permitting)
// PAIR_: two workgroups per CU that fill its LDS between them (mainloop_pair)
// ONCE_: the tile is its expert's only one in its column: nobody else reads its weights (see s2s_tile)
template <int BM_, int BN_, int WM_, int WN_, int NS_ = 2, bool RS_ = false, int WG_ = 1, bool PAIR_ = false, bool ONCE_ = false>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_;
  static constexpr int NS = NS_;                      // LDS stages (2: double buffer, more: ring)
  static constexpr bool RS = RS_;                     // operands travel global -> registers -> LDS (mainloop_rs)
  static constexpr int WG = WG_;
  static constexpr bool PAIR = PAIR_, ONCE = ONCE_;
  // the same tile with U blocks of 32 rows per wave
  template <int U> using Height = Tile<U * 32 * WM_, BN_, WM_, WN_, NS_, RS_, WG_, PAIR_, ONCE_>;
  typedef Tile<BM_, BN_, WM_, WN_, NS_, RS_, WG_, PAIR_, true> Once;
  static constexpr int NW = WM * WN, NT = NW * 64;
  static constexpr int WAVES_PER_SIMD = WG_ * NW / 4 > 0 ? WG_ * NW / 4 : 1;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int FM = WTM / 32, FN = WTN / 32;
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be a multiple of a 32x32 block");
};

// A wave's products of a slice where fragments are read while others are multiplied.  A step of 32 contraction elements needs
// 2 FM fragments of the row operand and 2 FN of the column operand (16 rows each), too many registers to hold twice.  It goes in
// four quarters, each half of the row fragments times half of the column fragments, in an order in which a half is read during
// the quarter before the one that needs it, into registers whose last use was the quarter before that: row halves 0 0 1 1,
// column halves 0 1 1 0 in a slice's first step, 1 0 0 1 in its second.
// Quarter Q = 0..7 of a slice:
template <int Q>
struct Quarter {
  static constexpr int STEP = Q >> 2, C = Q & 3;
  static constexpr int A = C >> 1, B = (C == 0 || C == 3 ? 0 : 1) ^ STEP;            // halves that it multiplies
  // the half that is read meanwhile: of the row (else the column) operand, which half, of which step (2: next slice, step 0)
  static constexpr bool READ_A = C == 1 || C == 2;
  static constexpr int READ_HALF = READ_A ? (C == 1 ? 1 : 0) : 1 ^ STEP;
  static constexpr int READ_STEP = C < 2 ? STEP : STEP + 1;
};
template <typename T, class TL, int Q>
__device__ __forceinline__ void quarter_products(Block (&acc)[TL::FM][TL::FN], const i32x4 (&fa)[2 * TL::FM], const i32x4 (&fb)[2 * TL::FN]) {
#pragma unroll
  for (int u = 0; u < TL::FM * TL::FN; ++u) {
    const int i = Quarter<Q>::A * TL::FM + u / TL::FN, j = Quarter<Q>::B * TL::FN + u % TL::FN;
    f32x4& c = acc[i >> 1][j >> 1].q[2 * (i & 1) + (j & 1)];
    c = Mfma<T>::run(fb[j], fa[i], c);
  }
}
// Fragment number f of the half that is read in quarter Q, from the stage at `ta`, `tb`.
template <class TL, class AOp, class BOp, int Q>
__device__ __forceinline__ void quarter_read(const char* ta, const char* tb, int wm, int wn, int f, i32x4 (&fa)[2 * TL::FM],
                                             i32x4 (&fb)[2 * TL::FN]) {
  typedef Quarter<Q> Qu;
  constexpr int step = Qu::READ_STEP & 1;
  if constexpr (Qu::READ_A) {
    const int i = Qu::READ_HALF * TL::FM + f;
    fa[i] = AOp::frag(ta, wm * TL::WTM + i * 16, step);
  } else {
    const int j = Qu::READ_HALF * TL::FN + f;
    fb[j] = BOp::frag(tb, wn * TL::WTN + j * 16, step);
  }
}

// Main loop shared by both kernels.  acc[i][j] is the 32x32 block (i, j) of this wave's tile.
// Full 64-deep slices travel global -> LDS directly (no registers, no ds_write) one slice ahead of the
// MFMAs; a trailing partial slice is zero-filled in LDS after it has landed.
// If `rowsum`, rs[i] additionally accumulates, per lane, the sum of the lane's own 8 contraction elements of
// A-fragment i; adding lanes l, l+16, l+32 and l+48 afterwards gives the sum over the contraction of A row l%16.
template <typename T, class TL, class AOp, class BOp, int Q, bool CAN_ROWSUM>
__device__ __forceinline__ void mainloop_quarter(const char* ta, const char* tb, int wm, int wn, bool rowsum,
                                                 Block (&acc)[TL::FM][TL::FN], float (&rs)[2 * TL::FM],
                                                 i32x4 (&fa)[2 * TL::FM], i32x4 (&fb)[2 * TL::FN]) {
  typedef Quarter<Q> Qu;
  // (four workgroups per CU hide a wave's wait for its row fragments, and have no registers to read them ahead)
  constexpr bool LATE_A = TL::WG > 2;
  constexpr int NF = Qu::READ_STEP == 2 || (LATE_A && Qu::READ_A) ? 0 : Qu::READ_A ? TL::FM : TL::FN;
  if constexpr (LATE_A && Q > 0 && (Qu::C & 1) == 0) {
#pragma unroll
    for (int i = 0; i < TL::FM; ++i)
      fa[Qu::A * TL::FM + i] = AOp::frag(ta, wm * TL::WTM + (Qu::A * TL::FM + i) * 16, Qu::STEP);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int f = 0; f < NF; ++f) quarter_read<TL, AOp, BOp, Q>(ta, tb, wm, wn, f, fa, fb);
  quarter_products<T, TL, Q>(acc, fa, fb);
  if (CAN_ROWSUM && rowsum && (Qu::C & 1) == 0) {
#pragma unroll
    for (int i = 0; i < TL::FM; ++i) rs[Qu::A * TL::FM + i] += Mfma<T>::sum8(fa[Qu::A * TL::FM + i]);
  }
  // Interleave: the LDS reads are spread between the first MFMAs.
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    __builtin_amdgcn_sched_group_barrier(0x100, Qu::READ_A ? AOp::DS_PER_FRAG : BOp::DS_PER_FRAG, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
  }
  if constexpr (TL::FM * TL::FN > NF) __builtin_amdgcn_sched_group_barrier(0x008, TL::FM * TL::FN - NF, 0);
  __builtin_amdgcn_sched_barrier(0);
}
template <typename T, class TL, class AOp, class BOp, bool CAN_ROWSUM>
__device__ __forceinline__ void mainloop(AOp& A, BOp& B, int klen, char* lds, bool rowsum,
                                         Block (&acc)[TL::FM][TL::FN], float (&rs)[2 * TL::FM]) {
  constexpr int STAGE = AOp::LDS_BYTES + BOp::LDS_BYTES;
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const int nfull = klen / BK;
  const bool tail = (klen % BK) != 0;
  const int nk = nfull + (tail ? 1 : 0);
  const unsigned lds_u = lds_address(lds);
  if (nfull > 0) issue_slice(A, B, lds_u, 0);
  else if (tail) issue_slice_tail(A, B, lds_u, 0, klen);
  A.fetch_rows(BK, klen);            // gathered operands: row indices of the slice after the one just issued
  B.fetch_rows(BK, klen);
  for (int kt = 0; kt < nk; ++kt) {
    char* cur = lds + (TL::NS == 1 ? 0 : (kt & 1) * STAGE);
    const unsigned nxt = lds_u + (TL::NS == 1 ? 0 : ((kt + 1) & 1) * STAGE);
    if (TL::NS == 1 && kt > 0) {
      // one stage: slice kt is requested once everyone is done with slice kt - 1; the other workgroups of the CU
      // multiply meanwhile
      __syncthreads();
      A.take_rows(kt);
      B.take_rows(kt);
      if (kt < nfull) issue_slice(A, B, lds_u, kt * BK);
      else issue_slice_tail(A, B, lds_u, kt * BK, klen);
      A.fetch_rows((kt + 1) * BK, klen);
      B.fetch_rows((kt + 1) * BK, klen);
    }
    __builtin_amdgcn_s_waitcnt(0);   // this thread's direct loads of slice kt have landed in LDS
    if (tail && kt == nfull) {
      A.zero_tail(cur, kt * BK, klen);
      B.zero_tail(cur + AOp::LDS_BYTES, kt * BK, klen);
    }
    A.stage_rows(kt + 1);
    B.stage_rows(kt + 1);
    __syncthreads();                 // ... everyone's have, and everyone is done reading `nxt`
    if constexpr (TL::NS > 1) {
      A.take_rows(kt + 1);
      B.take_rows(kt + 1);
      if (kt + 1 < nfull) issue_slice(A, B, nxt, (kt + 1) * BK);
      else if (tail && kt + 1 == nfull) issue_slice_tail(A, B, nxt, (kt + 1) * BK, klen);
      if (kt + 2 < nk) {
        A.fetch_rows((kt + 2) * BK, klen);
        B.fetch_rows((kt + 2) * BK, klen);
      }
    }
    const char* ta = cur;
    const char* tb = cur + AOp::LDS_BYTES;
    i32x4 fa[2 * TL::FM], fb[2 * TL::FN];
#pragma unroll
    for (int i = 0; i < TL::FM; ++i) fa[i] = AOp::frag(ta, wm * TL::WTM + i * 16, 0);
#pragma unroll
    for (int j = 0; j < TL::FN; ++j) fb[j] = BOp::frag(tb, wn * TL::WTN + j * 16, 0);
    mainloop_quarter<T, TL, AOp, BOp, 0, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 1, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 2, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 3, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 4, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 5, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 6, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
    mainloop_quarter<T, TL, AOp, BOp, 7, CAN_ROWSUM>(ta, tb, wm, wn, rowsum, acc, rs, fa, fb);
  }
}

// Main loop of the one-wave-per-SIMD class (4 waves, wave tiles of up to 128 x 128): operands travel global ->
// registers -> LDS.  A burst of loads at the top of a slice holds the waves that issue it off the matrix pipe until
// the memory pipeline has taken all of them (it takes one 1 KB wave-load per ~17 cycles and CU), and loads spread over
// the slice leave the late ones too little time to land when LDS is the only place they can land in: here every
// thread's pieces of a slice (16 in a 256 x 256 tile) sit in registers for up to two slices, which LDS has no room for.
//   set S = (kt + 1) & 1 holds slice kt + 1: its pieces are written to the other LDS stage during the first six of
//   slice kt's eight quarters (ds_write_b128, spread evenly: behind every sixth MFMA) and each is reloaded with slice kt + 3 two
//   quarters later (the last of them in the first two quarters of the next slice), one load per 8 MFMAs throughout;
//   one barrier per slice, after six quarters: behind it the first fragments of slice kt + 1 are read while the
//   last two quarters are multiplied.
// Whole 64-deep slices (the launchers check) or operands that read as zeros behind their last contraction row.  One slice is
// enough (a contraction part may have no more): what is loaded ahead past the last one, that one again (DirectOp) or zeros (TransOp),
// is written to LDS and not multiplied.
//
// A thread's pieces of a slice in the order they are written and reloaded: the operands alternate while the row
// operand (the smaller one in a tile of fewer than 256 rows) has pieces left.
template <class TL, class AOp, class BOp>
struct RsPlan {
  static constexpr int BOTH = AOp::R < BOp::R ? AOp::R : BOp::R;
  static constexpr int N = AOp::R + BOp::R;                       // pieces per thread and slice
  static constexpr int NM = TL::FM * TL::FN;                      // MFMAs per quarter of a step (Quarter), eight of them per slice
  static constexpr int L = (N + 3) / 4;                           // loads per two quarters (the first two: what is left)
  static constexpr bool is_b(int q) { return q >= 2 * BOTH ? BOp::R > AOp::R : (q & 1) != 0; }
  static constexpr int index(int q) { return q < 2 * BOTH ? q >> 1 : q - BOTH; }
  // pieces written before quarter Q, the first six
  static constexpr int written(int Q) { return N * Q / 6; }
  static_assert(written(2) >= L && written(4) >= 2 * L && N >= 3 * L, "a piece is reloaded after it has been written");
  // Places in a quarter: behind which MFMA fragment, write or load number i is issued.  An MFMA takes four issue slots, one of them
  // its own, so memory instructions, their waits and scalar work go behind different ones.
  static constexpr int read_at(int i, int NF) { return 2 * NF <= NM ? 2 * i : i; }
  static constexpr int write_at(int i) { return NM - 2 - 3 * i > 0 ? NM - 2 - 3 * i : 0; }
  static constexpr int load_at(int i) { return NM * (2 * i + 1) / 4 + (NM >= 8 ? 1 : 0); }
  // LDS: the two stages of the row operand, then those of the column operand, so that the instructions' offset fields reach from
  // one stage to the other (one set of addresses)
  static constexpr int A_STAGE = AOp::LDS_BYTES, B0 = 2 * AOp::LDS_BYTES, B_STAGE = BOp::LDS_BYTES;
};

// What the loads of the next slices have in common: at the start of slice kt of parity P, a[P], b[P] of slice kt + 2, the other
// ones of slice kt + 3.
template <class AOp, class BOp>
struct RsSlices {
  typename AOp::Slice a[2];
  typename BOp::Slice b[2];
};

template <typename T, class TL, class AOp, class BOp, int P, int Q, int N>
__device__ __forceinline__ void rs_quarter(const AOp& A, const BOp& B, char* lds, char* lds_b, int kt, int kend,
                                           RsSlices<AOp, BOp>& sl, int wm, int wn,
                                           Block (&acc)[TL::FM][TL::FN], i32x4 (&g)[2][N],
                                           i32x4 (&fa)[2 * TL::FM], i32x4 (&fb)[2 * TL::FN]) {
  typedef RsPlan<TL, AOp, BOp> Plan;
  typedef Quarter<Q> Qu;
  constexpr int NM = Plan::NM, S = P ^ 1;
  constexpr int NF = Qu::READ_A ? TL::FM : TL::FN;
  static_assert(NF <= NM, "at most one fragment read behind an MFMA");
  // fragments are read from the stage being multiplied, in the last two quarters from the stage just filled
  constexpr int src = Qu::READ_STEP == 2 ? S : P;
  // pieces written to the other stage; pieces loaded in two quarters: the last ones of the other set (slice kt + 2), then a third
  // each of the others of this one (slice kt + 3)
  constexpr int w0 = Plan::written(Q), nw = Q < 6 ? Plan::written(Q + 1) - w0 : 0;
  constexpr int H = Q >> 1, SET = H == 0 ? P : S;
  constexpr int q0 = H == 0 ? 3 * Plan::L : (H - 1) * Plan::L, nl2 = H == 0 ? N - 3 * Plan::L : Plan::L;
  constexpr int l0 = q0 + nl2 * (Q & 1) / 2, nl = q0 + nl2 * ((Q & 1) + 1) / 2 - l0;
  static_assert(nw <= 3 && nl <= 2, "places");
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const int i = Qu::A * TL::FM + m / TL::FN, j = Qu::B * TL::FN + m % TL::FN;
    Mfma<T>::in_place(fb[j], fa[i], acc[i >> 1][j >> 1].q[2 * (i & 1) + (j & 1)]);
#pragma unroll
    for (int f = 0; f < NF; ++f)
      if (Plan::read_at(f, NF) == m)
        quarter_read<TL, AOp, BOp, Q>(lds + src * Plan::A_STAGE, lds_b + src * Plan::B_STAGE, wm, wn, f, fa, fb);
#pragma unroll
    for (int f = 0; f < nw; ++f)
      if (Plan::write_at(nw - 1 - f) == m) {
        const int q = w0 + f;
        if (Plan::is_b(q)) lds_write16(lds_b + S * Plan::B_STAGE + B.piece_lds(Plan::index(q)), g[S][q]);
        else lds_write16(lds + S * Plan::A_STAGE + A.piece_lds(Plan::index(q)), g[S][q]);
      }
#pragma unroll
    for (int f = 0; f < nl; ++f)
      if (Plan::load_at(f) == m) {
        const int q = l0 + f;
        g[SET][q] = Plan::is_b(q) ? B.load_piece(sl.b[SET], Plan::index(q)) : A.load_piece(sl.a[SET], Plan::index(q));
      }
    if (Q == 2 && m == NM / 2 - 1) sl.a[P] = A.slice((kt + 4) * BK, kend);
    if (Q == 3 && m == NM / 2 - 1) sl.b[P] = B.slice((kt + 4) * BK, kend);
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (Q == 5) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // this thread's pieces are in LDS, its reads of this stage done
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <typename T, class TL, class AOp, class BOp, int P, int N>
__device__ __forceinline__ void rs_slice(const AOp& A, const BOp& B, char* lds, char* lds_b, int kt, int kend,
                                         RsSlices<AOp, BOp>& sl, int wm, int wn,
                                         Block (&acc)[TL::FM][TL::FN], i32x4 (&g)[2][N],
                                         i32x4 (&fa)[2 * TL::FM], i32x4 (&fb)[2 * TL::FN]) {
  __builtin_amdgcn_sched_barrier(0);
  rs_quarter<T, TL, AOp, BOp, P, 0, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 1, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 2, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 3, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 4, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 5, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 6, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
  rs_quarter<T, TL, AOp, BOp, P, 7, N>(A, B, lds, lds_b, kt, kend, sl, wm, wn, acc, g, fa, fb);
}

template <typename T, class TL, class AOp, class BOp>
__device__ __forceinline__ void mainloop_rs(const AOp& A, const BOp& B, int klen, char* lds, Block (&acc)[TL::FM][TL::FN]) {
  typedef RsPlan<TL, AOp, BOp> Plan;
  constexpr int N = Plan::N;
  static_assert(BK == 64, "eight quarters per slice");
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  // A partial last slice only with operands that zero-fill (TransOp); without any contraction rows one slice of
  // zeros is multiplied (no branch around the loop: 256 accumulator registers would have to be merged behind it).
  const int nk = max(1, (klen + BK - 1) / BK);
  i32x4 g[2][N];
  i32x4 fa[2 * TL::FM], fb[2 * TL::FN];
  RsSlices<AOp, BOp> sl = {{A.slice(0, klen), A.slice(BK, klen)}, {B.slice(0, klen), B.slice(BK, klen)}};
  auto load = [&](int set, int q) {
    return Plan::is_b(q) ? B.load_piece(sl.b[set], Plan::index(q)) : A.load_piece(sl.a[set], Plan::index(q));
  };
  // the column operand's stages from an address of their own (kept from being folded into constants): an instruction's offset
  // field does not reach them from the row operand's
  unsigned second = Plan::B0;
  asm volatile("" : "+v"(second));
  char* lds_b = lds + second;
#pragma unroll
  for (int q = 0; q < N; ++q) g[0][q] = load(0, q);
#pragma unroll
  for (int q = 0; q < N; ++q) g[1][q] = load(1, q);
  sl.a[0] = A.slice(2 * BK, klen), sl.b[0] = B.slice(2 * BK, klen);
  sl.a[1] = A.slice(3 * BK, klen), sl.b[1] = B.slice(3 * BK, klen);
#pragma unroll
  for (int q = 0; q < N; ++q) {
    if (Plan::is_b(q)) lds_write16(lds_b + B.piece_lds(Plan::index(q)), g[0][q]);
    else lds_write16(lds + A.piece_lds(Plan::index(q)), g[0][q]);
  }
#pragma unroll
  for (int q = 0; q < 3 * Plan::L; ++q) g[0][q] = load(0, q);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  // what the first quarter multiplies
#pragma unroll
  for (int i = 0; i < TL::FM; ++i) fa[i] = AOp::frag(lds, wm * TL::WTM + i * 16, 0);
#pragma unroll
  for (int j = 0; j < TL::FN; ++j) fb[j] = BOp::frag(lds_b, wn * TL::WTN + j * 16, 0);
  int kt = 0;
  for (; kt + 1 < nk; kt += 2) {
    rs_slice<T, TL, AOp, BOp, 0, N>(A, B, lds, lds_b, kt, klen, sl, wm, wn, acc, g, fa, fb);
    rs_slice<T, TL, AOp, BOp, 1, N>(A, B, lds, lds_b, kt + 1, klen, sl, wm, wn, acc, g, fa, fb);
  }
  if (kt < nk) rs_slice<T, TL, AOp, BOp, 0, N>(A, B, lds, lds_b, kt, klen, sl, wm, wn, acc, g, fa, fb);
  // (the compiler does not know how long the products above, being assembly, take to write their accumulators: 19 wait states at
  // the most; they are read by assembly, see stage_accumulators)
  asm volatile("s_nop 15\n\ts_nop 3");
}

// Main loop of the class with two workgroups of four waves per CU (256 x 128 tiles, wave tiles of up to 128 x 64).  Its
// point is what happens outside the loop: a tile is looked up, waits for its first slice and is rounded and stored while
// the other workgroup of the CU multiplies, which a 256 x 256 tile that has the CU to itself cannot hide (17 to 23 K cycles of
// them against 2 400 to 2 900 per slice).  80 KB of LDS each: two stages of the row operand, one of the column operand, whose
// fragments of a whole slice are read into registers (32 of them) ahead of the products, so that the next slice's pieces
// can be on their way into the same stage while they run.  The burst of reads and the two barriers around it fall into the
// other workgroup's products.
// Whole 64-deep slices only (the launcher checks), or operands that read as zeros behind their last contraction row (RowsOp).
// `rowsum` and rs as in mainloop.
static constexpr int PAIR_STAGE = 32 * 1024, PAIR_B = 2 * PAIR_STAGE, PAIR_LDS = PAIR_B + 16 * 1024;
template <typename T, class TL, class AOp, class BOp, bool ROWS>
__device__ __forceinline__ void mainloop_pair(AOp& A, BOp& B, int klen, char* lds, bool rowsum, Block (&acc)[TL::FM][TL::FN],
                                              float (&rs)[2 * TL::FM]) {
  static_assert(AOp::LDS_BYTES <= PAIR_STAGE && BOp::LDS_BYTES <= PAIR_LDS - PAIR_B, "LDS");
  constexpr int KS = 2 * (BK / 32), LOADS = AOp::R + BOp::R, PER_STEP = (LOADS + KS - 2) / (KS - 1);      // (all of them up front: 2 % slower)
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const unsigned lds_u = lds_address(lds);
  const int nk = ROWS ? max(1, (klen + BK - 1) / BK) : klen / BK;      // (no rows: one slice of zeros)
#pragma unroll
  for (int j = 0; j < BOp::R; ++j) B.issue_one(lds_u + PAIR_B, 0, j);
#pragma unroll
  for (int j = 0; j < AOp::R; ++j) A.issue_one(lds_u, 0, j);
  auto slice = [&](int kt, auto more) {
    const unsigned par = (unsigned)(kt & 1) * PAIR_STAGE;
    const char* ta = lds + par;
    const char* tb = lds + PAIR_B;
    const unsigned na = lds_u + (PAIR_STAGE - par);
    // this thread's pieces of slice kt have landed, everyone's have, and everyone is done with slice kt - 1
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ROWS && decltype(more)::value) {
      A.take_rows(kt + 1);
      B.take_rows(kt + 1);
    }
    // half of the row fragments of a step of 32 at a time, the next half read meanwhile
    i32x4 fa[2][TL::FM], fb[BK / 32][2 * TL::FN];
    auto row_frag = [&](int h, int i) { return AOp::frag(ta, wm * TL::WTM + ((h & 1) * TL::FM + i) * 16, h >> 1); };
#pragma unroll
    for (int j = 0; j < 2 * TL::FN; ++j) fb[0][j] = BOp::frag(tb, wn * TL::WTN + j * 16, 0);
#pragma unroll
    for (int i = 0; i < TL::FM; ++i) fa[0][i] = row_frag(0, i);
#pragma unroll
    for (int j = 0; j < 2 * TL::FN; ++j) fb[1][j] = BOp::frag(tb, wn * TL::WTN + j * 16, 1);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // everyone has the column operand's fragments
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);                       // ahead of the other workgroup's reads (1 to 2 %)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int c = ks & 1, n = c ^ 1;
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int q = ks * PER_STEP; q < (ks + 1) * PER_STEP && q < LOADS; ++q) {
          if (q < BOp::R) B.issue_one(lds_u + PAIR_B, (kt + 1) * BK, q);
          else A.issue_one(na, (kt + 1) * BK, q - BOp::R);
        }
        if constexpr (ROWS) {
          if (ks == 1) {
            A.stage_rows(kt + 2);
            B.stage_rows(kt + 2);
          }
          if (ks == KS - 1) {
            A.fetch_rows((kt + 3) * BK);
            B.fetch_rows((kt + 3) * BK);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (ks + 1 < KS) {
#pragma unroll
        for (int i = 0; i < TL::FM; ++i) fa[n][i] = row_frag(ks + 1, i);
      }
#pragma unroll
      for (int i = 0; i < TL::FM; ++i)
#pragma unroll
        for (int j = 0; j < 2 * TL::FN; ++j) {
          const int r = c * TL::FM + i;
          f32x4& d = acc[r >> 1][j >> 1].q[2 * (r & 1) + (j & 1)];
          d = Mfma<T>::run(fb[ks >> 1][j], fa[c][i], d);
        }
      if (ROWS && rowsum) {
#pragma unroll
        for (int i = 0; i < TL::FM; ++i) rs[c * TL::FM + i] += Mfma<T>::sum8(fa[c][i]);
      }
      if (ks + 1 < KS) {
#pragma unroll
        for (int i = 0; i < TL::FM; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, AOp::DS_PER_FRAG, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * TL::FM * TL::FN - TL::FM, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  for (int kt = 0; kt + 1 < nk; ++kt) slice(kt, std::true_type());
  slice(nk - 1, std::false_type());
}

// Main loop of the small-row (decode) tile class: memory bound, so what matters is bytes in flight.  The
// slices travel through a ring of NS stages; NS-1 slices are on their way while one is being multiplied.
template <typename T, class TL, class AOp, class BOp>
__device__ __forceinline__ void mainloop_ring(const AOp& A, const BOp& B, int klen, char* lds,
                                              Block (&acc)[TL::FM][TL::FN]) {
  constexpr int STAGE = AOp::LDS_BYTES + BOp::LDS_BYTES;
  constexpr int NS = TL::NS;
  constexpr int LOADS = AOp::R + BOp::R;               // direct loads per thread and slice
  static_assert((NS - 2) * LOADS <= 63, "vmcnt cannot count that many loads in flight");
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const int nfull = klen / BK;
  const bool tail = (klen % BK) != 0;
  const int nk = nfull + (tail ? 1 : 0);
  const unsigned lds_u = lds_address(lds);
#define SMOE_RING_ISSUE(s, slot)                                              \
  do {                                                                        \
    const unsigned dst_ = lds_u + (slot) * STAGE;                             \
    if ((s) < nfull) issue_slice(A, B, dst_, (s) * BK);                       \
    else if ((s) < nk) issue_slice_tail(A, B, dst_, (s) * BK, klen);          \
  } while (0)
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) SMOE_RING_ISSUE(s, s);
  int slot = 0;                                        // stage of slice kt
  for (int kt = 0; kt < nk; ++kt) {
    // slice kt has landed; the NS-2 younger slices may stay in flight (loads complete in issue order).
    // Near the end fewer are in flight, so wait for everything there.
    if (kt + NS - 2 < nk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    char* cur = lds + slot * STAGE;
    if (tail && kt == nfull) {
      A.zero_tail(cur, kt * BK, klen);
      B.zero_tail(cur + AOp::LDS_BYTES, kt * BK, klen);
    }
    __syncthreads();                 // everyone's part of slice kt is there; everyone is done with slice kt-1
    const int prev = slot == 0 ? NS - 1 : slot - 1;
    SMOE_RING_ISSUE(kt + NS - 1, prev);
    i32x4 fa[BK / 32][2 * TL::FM], fb[BK / 32][2 * TL::FN];
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
#pragma unroll
      for (int i = 0; i < 2 * TL::FM; ++i) fa[ks][i] = AOp::frag(cur, wm * TL::WTM + i * 16, ks);
#pragma unroll
      for (int j = 0; j < 2 * TL::FN; ++j) fb[ks][j] = BOp::frag(cur + AOp::LDS_BYTES, wn * TL::WTN + j * 16, ks);
    }
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks)
#pragma unroll
      for (int i = 0; i < 2 * TL::FM; ++i)
#pragma unroll
        for (int j = 0; j < 2 * TL::FN; ++j) {
          f32x4& c = acc[i >> 1][j >> 1].q[2 * (i & 1) + (j & 1)];
          c = Mfma<T>::run(fb[ks][j], fa[ks][i], c);
        }
    slot = slot + 1 == NS ? 0 : slot + 1;
  }
#undef SMOE_RING_ISSUE
}

// Store the wave's accumulators: per group of four (see Block) one 8-byte store instead of four 2-byte stores.  dst[m] is the element offset of output row m of the tile (or -1),
// columns n0 + [0, BN) clipped to ncols (contiguous); optional bias (already offset to the expert), stride sb.
template <typename T, class TL>
__device__ __forceinline__ void epilogue(const Block (&acc)[TL::FM][TL::FN], T* __restrict__ out,
                                         const int64_t* dst, int n0, int ncols,
                                         const T* __restrict__ bias, int64_t sb) {
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const bool base_ok = ((uintptr_t)out & 7) == 0;
#pragma unroll
  for (int i = 0; i < TL::FM; ++i) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t d = dst[wm * TL::WTM + i * 32 + block_row(l, g)];
#pragma unroll
      for (int j = 0; j < TL::FN; ++j) {
        const int n = n0 + wn * TL::WTN + j * 32 + block_col(l, g);
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[i][j][g * 4 + e];
          if (bias != nullptr && n + e < ncols) v[e] += to_f32(bias[(int64_t)(n + e) * sb]);
        }
        if (d < 0) continue;
        if (base_ok && n + 3 < ncols && ((d + n) & 3) == 0) {
          T4 p;
#pragma unroll
          for (int e = 0; e < 4; ++e) p[e] = from_f32<T>(v[e]);
          *(T4*)(out + d + n) = p;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < ncols) out[d + n + e] = from_f32<T>(v[e]);
        }
      }
    }
  }
}

// ---- epilogues that go through LDS ------------------------------------------------------------------
// Two floats rounded to the storage type by one instruction (element-wise casts cost a conversion and a merge per
// element); same rounding as the scalar cast.  `set_pair` puts the pair into elements 2k, 2k + 1 of a vector.
template <typename T, typename V>
__device__ __forceinline__ void set_pair(V& v, int k, float a, float b) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef T T2 __attribute__((ext_vector_type(2)));
  const T2 r = __builtin_convertvector((f32x2_t){a, b}, T2);
  v[2 * k] = r[0];
  v[2 * k + 1] = r[1];
}

// After the main loop the operand buffers are free.  The accumulators (transposed blocks, see `epilogue`) are
// rounded to the storage type and written to LDS as a row-major BM x BN tile, so that the global traffic of the
// epilogue can be 16 bytes per lane with a wave covering whole 128-byte lines: 16-byte piece c of row r sits at
// chunk c ^ (r & (CPR-1)) of the row (192 columns: c ^ (r & 7)), which keeps both the 8-byte column-strided writes and the 16-byte
// row-major reads free of bank conflicts.
template <class TL>
__device__ __forceinline__ int staged_addr(int row, int col) {
  constexpr int CPR = TL::BN / 8;
  constexpr int SWZ = (CPR & (CPR - 1)) == 0 ? CPR - 1 : 7;
  return row * (TL::BN * 2) + (((col >> 3) ^ (row & SWZ)) << 4) + ((col & 7) << 1);
}

// The thread's index, for what comes behind the main loop: the one-wave-per-SIMD form, and four workgroups per CU, have no
// registers to hold what the compiler would derive from it ahead of the loop.
template <class TL>
__device__ __forceinline__ int late_thread() {
  int t = (int)threadIdx.x;
  if constexpr (TL::RS || TL::WG > 2) asm volatile("" : "+v"(t));
  return t;
}
// Four accumulators where they are used.  One wave per SIMD: assembly, behind the wait at the main loop's end (left to the compiler,
// all accumulators are copied to vector registers ahead of it).
template <class TL>
__device__ __forceinline__ f32x4 accumulators(const f32x4& q) {
  if constexpr (!TL::RS) return q;
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float x;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"(q[e]));
    v[e] = x;
  }
  return v;
}

// `bias_of(tile_col)` returns the value to add to that column (0 without bias).
template <typename T, class TL, typename BF>
__device__ __forceinline__ void stage_accumulators(const Block (&acc)[TL::FM][TL::FN], char* lds, BF bias_of,
                                                   float* sbias) {
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int tx = late_thread<TL>(), wave = tx >> 6, l = tx & 63;
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  // One wave per SIMD: the additions per column come from LDS (written here, one column per thread), so that the
  // walk over the 256 accumulator registers below is one straight piece of code without loads or branches.
  if constexpr (TL::RS) {
    for (int t = tx; t < TL::BN; t += TL::NT) sbias[t] = bias_of(t);
  }
  __syncthreads();                                   // every wave is done reading operands
#pragma unroll
  for (int j = 0; j < TL::FN; ++j) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int col = wn * TL::WTN + j * 32 + block_col(l, c);
      float bv[4];
      if constexpr (TL::RS) {
        const f32x4 b4 = *(const f32x4*)(sbias + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[e] = b4[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[e] = bias_of(col + e);
      }
#pragma unroll
      for (int i = 0; i < 2 * TL::FM; ++i) {
        const int g = 2 * (i & 1) + c, row = wm * TL::WTM + (i >> 1) * 32 + block_row(l, g);
        const f32x4 q = accumulators<TL>(acc[i >> 1][j].q[g]);
        T4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = from_f32<T>(q[e] + bv[e]);
        *(T4*)(lds + staged_addr<TL>(row, col)) = v;
      }
    }
  }
  __syncthreads();
}

// What is added to output column n; to column tc of a tile of the fused forward GLU (hidden columns from nh0).
template <typename T>
__device__ __forceinline__ float plain_bias(const T* __restrict__ bias, int64_t sb, int ncols, int n) {
  return bias != nullptr && n < ncols ? to_f32(bias[(int64_t)n * sb]) : 0.0f;
}
template <typename T, class TL>
__device__ __forceinline__ float glu_bias(const S2SArgs& a, const T* __restrict__ bias, int nh0, int tc) {
  constexpr int HALF = TL::WTN / 2;
  const int j = tc % TL::WTN;
  const int hc = nh0 + (tc / TL::WTN) * HALF + j % HALF;
  return bias != nullptr && hc < a.N ? to_f32(bias[(int64_t)(hc + (j >= HALF ? a.N : 0)) * a.sbn]) : 0.0f;
}

// Fused gated-linear-unit epilogues (rows in grouped order: output row = row0 + m).
// Forward: the column operand of the tile is laid out so that each wave owns WTN/2 "first half" columns
// (accumulator blocks j < FN/2) and the matching WTN/2 "second half" columns (blocks j + FN/2).  Both are
// rounded to the storage type first and the hidden value is computed from the rounded values, i.e. the same
// arithmetic as storing the pre-activation and running the stand-alone pass over it.
template <typename T, class TL>
__device__ __forceinline__ void epilogue_glu_fwd(const Block (&acc)[TL::FM][TL::FN], const S2SArgs& a, int row0,
                                                 int rows, int nh0, const T* __restrict__ bias) {
  if constexpr (TL::FN % 2 == 0) {
    typedef T T4 __attribute__((ext_vector_type(4)));
    constexpr int FH = TL::FN / 2;
    const int wave = threadIdx.x >> 6, l = lane_id();
    const int wm = wave / TL::WN, wn = wave % TL::WN;
    const int F = a.N;
    const bool gf = (a.act & 1) != 0;
    T* pre = (T*)a.Y;
    T* hid = (T*)a.H;
    const bool vec_ok = (((uintptr_t)pre | (uintptr_t)hid) & 7) == 0 && ((a.sym | a.shm | F) & 3) == 0;
#pragma unroll
    for (int i = 0; i < TL::FM; ++i) {
#pragma unroll
      for (int j = 0; j < FH; ++j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int m = wm * TL::WTM + i * 32 + block_row(l, g);
          const int64_t row = row0 + m;
          const int n = nh0 + wn * (TL::WTN / 2) + j * 32 + block_col(l, g);
          T first[4], second[4], h[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v1 = acc[i][j][g * 4 + e], v2 = acc[i][j + FH][g * 4 + e];
            if (bias != nullptr && n + e < F) {
              v1 += to_f32(bias[(int64_t)(n + e) * a.sbn]);
              v2 += to_f32(bias[(int64_t)(F + n + e) * a.sbn]);
            }
            first[e] = from_f32<T>(v1);
            second[e] = from_f32<T>(v2);
            const float lin = to_f32(gf ? second[e] : first[e]), gat = to_f32(gf ? first[e] : second[e]);
            h[e] = from_f32<T>(glu_h(a.act, gat, lin));
          }
          if (m >= rows) continue;
          if (vec_ok && n + 3 < F) {
            if (pre != nullptr) {
              *(T4*)(pre + row * a.sym + n) = T4{first[0], first[1], first[2], first[3]};
              *(T4*)(pre + row * a.sym + F + n) = T4{second[0], second[1], second[2], second[3]};
            }
            *(T4*)(hid + row * a.shm + n) = T4{h[0], h[1], h[2], h[3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (n + e >= F) continue;
              if (pre != nullptr) {
                pre[row * a.sym + n + e] = first[e];
                pre[row * a.sym + F + n + e] = second[e];
              }
              hid[row * a.shm + n + e] = h[e];
            }
          }
        }
      }
    }
  }
}

// Backward: the product is d(hidden); it is rounded to the storage type and turned into d(pre-activation)
// with the saved pre-activation, exactly as the stand-alone pass would do from a stored d(hidden).
template <typename T, class TL>
__device__ __forceinline__ void epilogue_glu_bwd(const Block (&acc)[TL::FM][TL::FN], const S2SArgs& a, int row0,
                                                 int rows, int n0) {
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const int F = a.N;
  const bool gf = (a.act & 1) != 0;
  const T* pre = (const T*)a.aux;
  T* dpre = (T*)a.Y;
  const bool vec_ok = (((uintptr_t)pre | (uintptr_t)dpre) & 7) == 0 && ((a.sym | a.saux | F) & 3) == 0;
#pragma unroll
  for (int i = 0; i < TL::FM; ++i) {
#pragma unroll
    for (int j = 0; j < TL::FN; ++j) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int m = wm * TL::WTM + i * 32 + block_row(l, g);
        const int64_t row = row0 + m;
        const int n = n0 + wn * TL::WTN + j * 32 + block_col(l, g);
        if (m >= rows || n >= F) continue;
        const bool vec = vec_ok && n + 3 < F;
        T p1[4], p2[4], o1[4], o2[4];
        if (vec) {
          const T4 v1 = *(const T4*)(pre + row * a.saux + n), v2 = *(const T4*)(pre + row * a.saux + F + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) { p1[e] = v1[e]; p2[e] = v2[e]; }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool ok = n + e < F;
            p1[e] = ok ? pre[row * a.saux + n + e] : from_f32<T>(0.0f);
            p2[e] = ok ? pre[row * a.saux + F + n + e] : from_f32<T>(0.0f);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float dv = to_f32(from_f32<T>(acc[i][j][g * 4 + e]));
          const float lin = to_f32(gf ? p2[e] : p1[e]), gat = to_f32(gf ? p1[e] : p2[e]);
          float f_lin, f_gat;
          glu_grad(a.act, dv, gat, lin, f_lin, f_gat);
          const T d_lin = from_f32<T>(f_lin), d_gat = from_f32<T>(f_gat);
          o1[e] = gf ? d_gat : d_lin;
          o2[e] = gf ? d_lin : d_gat;
        }
        if (vec) {
          *(T4*)(dpre + row * a.sym + n) = T4{o1[0], o1[1], o1[2], o1[3]};
          *(T4*)(dpre + row * a.sym + F + n) = T4{o2[0], o2[1], o2[2], o2[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (n + e >= F) continue;
            dpre[row * a.sym + n + e] = o1[e];
            dpre[row * a.sym + F + n + e] = o2[e];
          }
        }
      }
    }
  }
}

// Plain store through LDS: dst[m] is the element offset of output row m of the tile (or -1).
// Output tiles are written once and not read again by the launch: stored with the non-temporal hint so that they
// do not displace operand panels in the L2 (c4: -1 % step time, c2: -0.2 %).
template <typename V>
__device__ __forceinline__ void stream_store(const V& v, V* p) { __builtin_nontemporal_store(v, p); }

// 16-byte store through a buffer descriptor: the hardware drops it when `offset` (bytes) lies beyond the descriptor's
// range, so a piece outside the tile's valid part needs no branch around its store.  That matters where loads are in
// flight across the stores: stores and loads share one counter, and behind a store that a branch may have skipped
// the compiler can only wait for everything, the prefetched loads of the next group included.
template <typename V>
__device__ __forceinline__ void range_checked_store(const V& v, __amdgpu_buffer_rsrc_t r, unsigned offset) {
  static_assert(sizeof(V) == 16, "16-byte pieces");
  typedef unsigned u32x4_st __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_st, v), r, (int)offset, 0, 2 /* non-temporal */);
}
// Descriptor over the valid rows of a tile's output: `row_bytes` per row from `base` on.
// (Base and range are the same for every lane; saying so keeps the compiler from wrapping each store into a loop
// over the distinct descriptors of the wave.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rows_rsrc(void* base, int rows, int64_t row_bytes) {
  const int64_t span = (int64_t)rows * row_bytes;
  const int range = __builtin_amdgcn_readfirstlane(span < 0xffffffffLL ? (int)(unsigned)span : -1);
  return __builtin_amdgcn_make_buffer_rsrc((void*)make_uniform((const char*)base), 0, range, 0x00020000);
}

template <typename T, class TL>
__device__ __forceinline__ void epilogue_staged(const Block (&acc)[TL::FM][TL::FN], T* __restrict__ out,
                                                const int64_t* dst, int n0, int ncols, const T* __restrict__ bias,
                                                int64_t sb, char* lds) {
  const int tx = late_thread<TL>();
  typedef T T8 __attribute__((ext_vector_type(8)));
  constexpr int CPR = TL::BN / 8, PIECES = TL::BM * CPR, PP = PIECES / TL::NT;
  static_assert(PIECES % TL::NT == 0, "pieces must divide evenly");
  if constexpr (!TL::RS)
    stage_accumulators<T, TL>(acc, lds, [&](int tc) { return plain_bias<T>(bias, sb, ncols, n0 + tc); }, nullptr);
  // In groups: the row offsets of a group, then its pieces, are read from LDS back to back before the first of its
  // stores (written as one conditional store per piece, every piece would wait for two LDS round trips of its own)
  constexpr int GRP = PP % 16 == 0 ? 16 : PP % 8 == 0 ? 8 : PP % 6 == 0 ? 6 : PP;
  static_assert(PP % GRP == 0, "groups must divide the pieces");
#pragma unroll
  for (int q0 = 0; q0 < PP; q0 += GRP) {
    int64_t d[GRP];
    T8 v[GRP];
#pragma unroll
    for (int g = 0; g < GRP; ++g) d[g] = dst[((q0 + g) * TL::NT + tx) / CPR];
#pragma unroll
    for (int g = 0; g < GRP; ++g) {
      const int p = (q0 + g) * TL::NT + tx;
      v[g] = *(const T8*)(lds + staged_addr<TL>(p / CPR, (p % CPR) * 8));
    }
#pragma unroll
    for (int g = 0; g < GRP; ++g) asm volatile("" : "+v"(v[g]), "+v"(d[g]));      // keeps the reads above the branches
#pragma unroll
    for (int g = 0; g < GRP; ++g) {
      const int n = n0 + (((q0 + g) * TL::NT + tx) % CPR) * 8;
      if (d[g] >= 0 && n < ncols) stream_store(v[g], (T8*)(out + d[g] + n));
    }
  }
}

// Forward GLU through LDS: both halves staged (tile column order: per wave block WTN/2 first-half columns, then
// the matching second-half columns); per 16-byte piece of hidden columns two LDS reads, three coalesced stores.
template <typename T, class TL>
__device__ __forceinline__ void epilogue_glu_fwd_staged(const Block (&acc)[TL::FM][TL::FN], const S2SArgs& a,
                                                        int row0, int rows, int nh0, const T* __restrict__ bias,
                                                        char* lds) {
  {
    const int tx = late_thread<TL>();
    typedef T T8 __attribute__((ext_vector_type(8)));
    constexpr int HALF = TL::WTN / 2;
    constexpr int CPR = TL::BN / 16, PIECES = TL::BM * CPR, PP = PIECES / TL::NT;
    static_assert(PIECES % TL::NT == 0 && HALF % 8 == 0, "pieces must divide evenly");
    const int F = a.N;
    if constexpr (!TL::RS) stage_accumulators<T, TL>(acc, lds, [&](int tc) { return glu_bias<T, TL>(a, bias, nh0, tc); }, nullptr);
    T* pre = (T*)a.Y;
    T* hid = (T*)a.H;
    // a group's LDS reads are issued back to back ahead of its arithmetic and stores (see epilogue_staged)
    constexpr int GRP = PP % 8 == 0 ? 8 : PP % 4 == 0 ? 4 : PP;
    static_assert(PP % GRP == 0, "groups must divide the pieces");
    // which half holds the gate is the same for the whole launch: one copy of the loop for each case instead of a
    // select per element (the accumulators are in LDS by now, so the branch has nothing to carry)
    auto pieces = [&](auto gate_first) {
    const bool gf = gate_first;       // a constant in the two copies of the one-wave-per-SIMD class
#pragma unroll
    for (int q0 = 0; q0 < PP; q0 += GRP) {
      T8 v1[GRP], v2[GRP];
#pragma unroll
      for (int g = 0; g < GRP; ++g) {
        const int p = (q0 + g) * TL::NT + tx;
        const int row = p / CPR, hc = (p % CPR) * 8;          // hidden column inside the tile
        const int tc = (hc / HALF) * TL::WTN + hc % HALF;     // tile column of the first-half value
        v1[g] = *(const T8*)(lds + staged_addr<TL>(row, tc));
        v2[g] = *(const T8*)(lds + staged_addr<TL>(row, tc + HALF));
      }
#pragma unroll
      for (int g = 0; g < GRP; ++g) asm volatile("" : "+v"(v1[g]), "+v"(v2[g]));
#pragma unroll
      for (int g = 0; g < GRP; ++g) {
        const int p = (q0 + g) * TL::NT + tx;
        const int row = p / CPR, n = nh0 + (p % CPR) * 8;
        if (row >= rows || n >= F) continue;
        const T8 first = v1[g], second = v2[g];
        T8 h;
#pragma unroll
        for (int e = 0; e < 8; e += 2)
          set_pair<T>(h, e / 2, glu_h(a.act, to_f32(gf ? first[e] : second[e]), to_f32(gf ? second[e] : first[e])),
                      glu_h(a.act, to_f32(gf ? first[e + 1] : second[e + 1]), to_f32(gf ? second[e + 1] : first[e + 1])));
        const int64_t r = row0 + row;
        if (pre != nullptr) {
          stream_store(first, (T8*)(pre + r * a.sym + n));
          stream_store(second, (T8*)(pre + r * a.sym + F + n));
        }
        stream_store(h, (T8*)(hid + r * a.shm + n));
      }
    }
    };
    // (the 8-wave classes, with half the registers per wave, keep one copy and select per element: two copies
    // there cost 130 spilled registers)
    if constexpr (!TL::RS) pieces((a.act & 1) != 0);
    else if ((a.act & 1) != 0) pieces(std::true_type());
    else pieces(std::false_type());
  }
}

// Backward through LDS: d(hidden) tile staged, then every thread handles 16-byte pieces (8 columns of one row):
// two coalesced 16-byte loads of the saved pre-activation, two coalesced 16-byte stores of its gradient.
template <typename T, class TL>
__device__ __forceinline__ void epilogue_glu_bwd_staged(const Block (&acc)[TL::FM][TL::FN], const S2SArgs& a,
                                                        int row0, int rows, int n0, char* lds) {
  const int tx = late_thread<TL>();
  typedef T T8 __attribute__((ext_vector_type(8)));
  constexpr int CPR = TL::BN / 8, PIECES = TL::BM * CPR, PP = PIECES / TL::NT;
  constexpr int GRP = PP % 8 == 0 ? 4 : PP % 4 == 0 ? 2 : PP % 6 == 0 ? 3 : (PP >= 2 ? PP / 2 : 1);    // pieces per group, two in flight
  static_assert(PIECES % TL::NT == 0 && (PP == 1 || PP % (2 * GRP) == 0), "pieces must divide evenly");
  if constexpr (!TL::RS) stage_accumulators<T, TL>(acc, lds, [](int) { return 0.0f; }, nullptr);
  const int F = a.N;
  const T* pre = (const T*)a.aux;
  T* dpre = (T*)a.Y;
  const __amdgpu_buffer_rsrc_t out_rows = tile_rows_rsrc(dpre + (int64_t)row0 * a.sym, rows, a.sym * 2);
  // The saved pre-activation of the next group of pieces is on its way while the current group is worked on (loads of
  // rows and columns outside the tile's valid part are redirected to its first row / column and their results dropped).
  // One copy of the loop for each position of the gate half (see epilogue_glu_fwd_staged).
  auto pieces = [&](auto gate_first) {
  const bool gf = gate_first;       // a constant in the two copies of the one-wave-per-SIMD class
  T8 p1[2][GRP], p2[2][GRP];
  auto fetch = [&](auto buf, int q0) {
#pragma unroll
    for (int u = 0; u < GRP; ++u) {
      const int p = (q0 + u) * TL::NT + tx;
      const int row = p / CPR, n = n0 + (p % CPR) * 8;
      const T* src = pre + (int64_t)(row0 + (row < rows ? row : 0)) * a.saux + (n < F ? n : 0);
      // read exactly once per step: the non-temporal hint keeps it from displacing operand panels in the L2 (-0.3 %)
      p1[decltype(buf)::value][u] = __builtin_nontemporal_load((const T8*)src);
      p2[decltype(buf)::value][u] = __builtin_nontemporal_load((const T8*)(src + F));
    }
  };
  auto work = [&](auto buf, int q0) {
    T8 dh[GRP];
#pragma unroll
    for (int u = 0; u < GRP; ++u) {
      const int p = (q0 + u) * TL::NT + tx;
      dh[u] = *(const T8*)(lds + staged_addr<TL>(p / CPR, (p % CPR) * 8));
    }
#pragma unroll
    for (int u = 0; u < GRP; ++u) {
      const int p = (q0 + u) * TL::NT + tx;
      const int row = p / CPR, n = n0 + (p % CPR) * 8;
      T8 o1, o2;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float f_lin[2], f_gat[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const T v1 = p1[decltype(buf)::value][u][e + h], v2 = p2[decltype(buf)::value][u][e + h];
          glu_grad(a.act, to_f32(dh[u][e + h]), to_f32(gf ? v1 : v2), to_f32(gf ? v2 : v1), f_lin[h], f_gat[h]);
        }
        set_pair<T>(o1, e / 2, gf ? f_gat[0] : f_lin[0], gf ? f_gat[1] : f_lin[1]);
        set_pair<T>(o2, e / 2, gf ? f_lin[0] : f_gat[0], gf ? f_lin[1] : f_gat[1]);
      }
      const unsigned at = row < rows && n < F ? (unsigned)(((int64_t)row * a.sym + n) * 2) : 0xffffffffu;
      range_checked_store(o1, out_rows, at);
      range_checked_store(o2, out_rows, at == 0xffffffffu ? at : at + (unsigned)F * 2);
    }
  };
  fetch(std::integral_constant<int, 0>(), 0);
  // two trips per pass: at the head of a loop the compiler waits for every outstanding load and store
#pragma unroll 2
  for (int q0 = 0; q0 < PP; q0 += 2 * GRP) {
    if constexpr (PP > 1) fetch(std::integral_constant<int, 1>(), q0 + GRP);
    work(std::integral_constant<int, 0>(), q0);
    if constexpr (PP > 1) {
      if (q0 + 2 * GRP < PP) fetch(std::integral_constant<int, 0>(), q0 + 2 * GRP);
      work(std::integral_constant<int, 1>(), q0 + GRP);
    }
  }
  };
  if constexpr (!TL::RS) pieces((a.act & 1) != 0);
  else if ((a.act & 1) != 0) pieces(std::true_type());
  else pieces(std::false_type());
}

// gpt-oss forward through LDS: the tile holds BN consecutive columns of the pre-activation, i.e. BN/2 (gate, up)
// pairs per row; per 16-byte piece one LDS read, one 16-byte store of the pre-activation (if wanted) and one
// 8-byte store of four hidden values.
template <typename T, class TL>
__device__ __forceinline__ void epilogue_oss_fwd_staged(const Block (&acc)[TL::FM][TL::FN], const S2SArgs& a,
                                                        int row0, int rows, int n0, const T* __restrict__ bias,
                                                        char* lds) {
  const int tx = late_thread<TL>();
  typedef T T8 __attribute__((ext_vector_type(8)));
  typedef T T4 __attribute__((ext_vector_type(4)));
  constexpr int CPR = TL::BN / 8, PIECES = TL::BM * CPR, PP = PIECES / TL::NT;
  static_assert(PIECES % TL::NT == 0, "pieces must divide evenly");
  if constexpr (!TL::RS)
    stage_accumulators<T, TL>(acc, lds, [&](int tc) { return plain_bias<T>(bias, a.sbn, a.N, n0 + tc); }, nullptr);
  T* pre = (T*)a.Y;
  T* hid = (T*)a.H;
  constexpr int GRP = PP % 16 == 0 ? 16 : PP % 8 == 0 ? 8 : PP;      // LDS reads of a group back to back (see epilogue_staged)
  static_assert(PP % GRP == 0, "groups must divide the pieces");
#pragma unroll
  for (int q0 = 0; q0 < PP; q0 += GRP) {
    T8 vs[GRP];
#pragma unroll
    for (int g = 0; g < GRP; ++g) {
      const int p = (q0 + g) * TL::NT + tx;
      vs[g] = *(const T8*)(lds + staged_addr<TL>(p / CPR, (p % CPR) * 8));
    }
#pragma unroll
    for (int g = 0; g < GRP; ++g) asm volatile("" : "+v"(vs[g]));
#pragma unroll
    for (int g = 0; g < GRP; ++g) {
      const int p = (q0 + g) * TL::NT + tx;
      const int row = p / CPR, n = n0 + (p % CPR) * 8;
      if (row >= rows || n >= a.N) continue;
      const T8 v = vs[g];
      T4 h;
#pragma unroll
      for (int e = 0; e < 4; e += 2)
        set_pair<T>(h, e / 2, oss_h(to_f32(v[2 * e]), to_f32(v[2 * e + 1]), a.alpha, a.limit),
                    oss_h(to_f32(v[2 * e + 2]), to_f32(v[2 * e + 3]), a.alpha, a.limit));
      const int64_t r = row0 + row;
      if (pre != nullptr) stream_store(v, (T8*)(pre + r * a.sym + n));
      stream_store(h, (T4*)(hid + r * a.shm + n / 2));
    }
  }
}

// gpt-oss backward through LDS: d(hidden) tile staged; per piece of 8 hidden columns two 16-byte loads of the saved
// pre-activation pairs and two 16-byte stores of their gradient.
template <typename T, class TL>
__device__ __forceinline__ void epilogue_oss_bwd_staged(const Block (&acc)[TL::FM][TL::FN], const S2SArgs& a,
                                                        int row0, int rows, int n0, char* lds) {
  const int tx = late_thread<TL>();
  typedef T T8 __attribute__((ext_vector_type(8)));
  constexpr int CPR = TL::BN / 8, PIECES = TL::BM * CPR, PP = PIECES / TL::NT;
  constexpr int GRP = PP % 8 == 0 ? 4 : PP % 4 == 0 ? 2 : PP % 6 == 0 ? 3 : (PP >= 2 ? PP / 2 : 1);    // pieces per group, two in flight
  static_assert(PIECES % TL::NT == 0 && (PP == 1 || PP % (2 * GRP) == 0), "pieces must divide evenly");
  if constexpr (!TL::RS) stage_accumulators<T, TL>(acc, lds, [](int) { return 0.0f; }, nullptr);
  const int F = a.N;
  const T* pre = (const T*)a.aux;
  T* dpre = (T*)a.Y;
  const __amdgpu_buffer_rsrc_t out_rows = tile_rows_rsrc(dpre + (int64_t)row0 * a.sym, rows, a.sym * 2);
  // next group's saved pre-activation pairs on their way while the current group is worked on (see epilogue_glu_bwd_staged)
  T8 p1[2][GRP], p2[2][GRP];
  auto fetch = [&](auto buf, int q0) {
#pragma unroll
    for (int u = 0; u < GRP; ++u) {
      const int p = (q0 + u) * TL::NT + tx;
      const int row = p / CPR, n = n0 + (p % CPR) * 8;
      const T* src = pre + (int64_t)(row0 + (row < rows ? row : 0)) * a.saux + 2 * (n < F ? n : 0);
      p1[decltype(buf)::value][u] = *(const T8*)src;
      p2[decltype(buf)::value][u] = *(const T8*)(src + 8);
    }
  };
  auto work = [&](auto buf, int q0) {
    T8 dh[GRP];
#pragma unroll
    for (int u = 0; u < GRP; ++u) {
      const int p = (q0 + u) * TL::NT + tx;
      dh[u] = *(const T8*)(lds + staged_addr<TL>(p / CPR, (p % CPR) * 8));
    }
#pragma unroll
    for (int u = 0; u < GRP; ++u) {
      const int p = (q0 + u) * TL::NT + tx;
      const int row = p / CPR, n = n0 + (p % CPR) * 8;
      const T8 v1 = p1[decltype(buf)::value][u], v2 = p2[decltype(buf)::value][u];
      T8 o1, o2;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float dg, du;
        oss_grad(to_f32(v1[2 * e]), to_f32(v1[2 * e + 1]), to_f32(dh[u][e]), a.alpha, a.limit, dg, du);
        set_pair<T>(o1, e, dg, du);
        oss_grad(to_f32(v2[2 * e]), to_f32(v2[2 * e + 1]), to_f32(dh[u][4 + e]), a.alpha, a.limit, dg, du);
        set_pair<T>(o2, e, dg, du);
      }
      const unsigned at = row < rows && n < F ? (unsigned)(((int64_t)row * a.sym + 2 * n) * 2) : 0xffffffffu;
      range_checked_store(o1, out_rows, at);
      range_checked_store(o2, out_rows, at == 0xffffffffu ? at : at + 16u);
    }
  };
  fetch(std::integral_constant<int, 0>(), 0);
  // two trips per pass: at the head of a loop the compiler waits for every outstanding load and store
#pragma unroll 2
  for (int q0 = 0; q0 < PP; q0 += 2 * GRP) {
    if constexpr (PP > 1) fetch(std::integral_constant<int, 1>(), q0 + GRP);
    work(std::integral_constant<int, 0>(), q0);
    if constexpr (PP > 1) {
      if (q0 + 2 * GRP < PP) fetch(std::integral_constant<int, 0>(), q0 + 2 * GRP);
      work(std::integral_constant<int, 1>(), q0 + GRP);
    }
  }
}

// XCD-aware tile order.  Workgroup ids are dealt round-robin to the 8 XCDs (private L2 each), so the 32
// workgroups an XCD runs side by side are the ids x, x+8, ..., x+248 of one 256-block; they are mapped to
// one 8 x 4 "super tile" of output tiles.  Per 64-deep slice that group touches 8 row panels + 4 column
// panels for 32 tiles' worth of operands, i.e. 3/8 of the requests miss the XCD's L2 instead of 9/16 for
// a 16 x 2 arrangement and 33/64 for 32 x 1 (measured at the Mixtral shape: 13.3 GB fetched from the
// memory side per launch against 20.5 GB for 16 x 2).  Super tiles are numbered row-super fastest so that
// the XCDs working at the same time share column panels through the memory-side cache.
struct Raster {
  static constexpr int SM = 8, SN = 4;
  int m_tiles, n_tiles, m_supers, n_supers, supers, gm;
  int striped;                             // 1: column-striped order of the memory-bound classes (see make_striped)
  int chunked = 0;                         // 1, 2: order of find_tile_chunked (2: in rounds) before this one
  int once = 0;                            // weights of experts of one tile row bypass the caches (see reads_weights_once)
  int64_t grid_size;                       // host side only: number of workgroups (may exceed what a launch takes)
  __host__ int64_t grid() const { return grid_size; }
  // (ml, nl): position of the tile inside its super tile
  template <int SN_ = SN>
  __host__ __device__ __forceinline__ bool map(int pid, int& m, int& n, int& ml, int& nl) const {
    const int x = pid & 7, i = pid >> 3;
    if (striped) {
      // Columns of a group of gm tile rows, one group after another, are dealt to the XCDs in eights, one each: no XCD has more
      // than one column group more than another, and none has workgroups without a tile between those with one (they leave at
      // once, but the CUs are dealt out by turns: 8 of every 16 put two tiles on every second CU).  Which of the eight an XCD takes
      // moves on with the groups; an XCD that keeps the same columns of all experts is slower (16 experts, 346 rows as 1 / rank^1.8,
      // 2688 -> 2 x 7168, 112 columns 144 -> 152 us).
      const int m_lo = i % gm, j = i / gm;
      const int u = 8 * j + ((x + 8 * j / n_tiles) & 7), g = u / n_tiles;
      m = g * gm + m_lo;
      n = u - g * n_tiles;
      ml = nl = 0;
      return m < m_tiles && n < n_tiles;
    }
    // The 8 supers of step j = i / 32 go to the 8 XCDs rotated by j: supers differ in how many of their tiles
    // exist (partial last column-super, empty tile rows), and a fixed assignment would give some XCDs the full
    // ones every time.
    const int j = i / (SM * SN_);
    const int s = j * 8 + ((x + j) & 7), r = i % (SM * SN_);
    if (s >= supers) return false;
    ml = r % SM;
    nl = r / SM;
    // bands of `gm` row-supers; inside a band column-super major, row-super fastest
    const int band = s / (gm * n_supers);
    const int rem = s - band * gm * n_supers;
    const int g = min(gm, m_supers - band * gm);
    m = (band * gm + rem % g) * SM + r % SM;
    n = (rem / g) * SN_ + r / SM;
    return m < m_tiles && n < n_tiles;
  }
};

// `gm`: row-supers per band.  A band's row panels (gm * 8 tiles) are reused by every column-super while the
// column panels stream past once, so the band should be small enough for its row panels to stay in the
// memory-side cache and large enough to keep all XCDs inside one band.
static Raster make_raster(int64_t m_tiles, int n_tiles, int gm, int sn = Raster::SN) {
  Raster r;
  r.m_tiles = (int)m_tiles;
  r.n_tiles = n_tiles;
  r.m_supers = (int)((m_tiles + Raster::SM - 1) / Raster::SM);
  r.n_supers = (n_tiles + sn - 1) / sn;
  r.striped = 0;
  r.gm = gm < 1 ? 1 : (gm > r.m_supers ? r.m_supers : gm);
  const int64_t supers = (int64_t)r.m_supers * r.n_supers;
  r.grid_size = (supers + 7) / 8 * 8 * Raster::SM * sn;
  r.supers = supers > 0x7fffffffLL ? 0x7fffffff : (int)supers;   // such a grid is rejected by the launchers
  return r;
}

// Order of the memory-bound (ring) classes.  The grid covers an upper bound of the tile rows, so some rows are
// empty, and which ones is known only on the device: every XCD therefore takes the same share of every group of `gm` tile
// rows, and the empty rows, which come last, cost nothing but their launch.  The rows of a group visit a tile column back to
// back on one XCD, so that an expert with several tile rows finds its weight panel in that XCD's L2.
// us, when XCD x had the columns n = x + group (mod 8) of a group, existing or not -> now: 8 experts x 584 rows, 21 tile rows in
// ten columns, 4640 -> 1272 179 -> 115 (the first XCDs had two columns in each of the groups, 42 tiles where a round is 32 per XCD);
// random launches with loads as 1 / rank^0.3 to ^1.8 of 4 to 112 rows per expert 1.03 to 1.06 times as fast, of 112 to 1000 1.02 to
// 1.07, in tiles of 192 columns 1.03 to 1.06, single ones 0.94 to 1.77; whole layers drawn at random 1.00 to 1.02 (0.98 to 1.52).
static Raster make_striped(int64_t m_tiles, int n_tiles, int gm) {
  Raster r;
  r.striped = 1;
  r.m_tiles = (int)m_tiles;
  r.n_tiles = n_tiles;
  r.gm = gm < 1 ? 1 : (gm > m_tiles ? (int)m_tiles : gm);
  r.n_supers = 0;
  r.m_supers = (int)((m_tiles + r.gm - 1) / r.gm);                       // groups of tile rows
  r.supers = 0;
  r.grid_size = ((int64_t)r.m_supers * n_tiles + 7) / 8 * 8 * r.gm;
  return r;
}

// =====================================================================================================
// scatter2scatter
// =====================================================================================================
// What the workgroup of an output tile knows before it starts on it.
struct S2STile {
  int e, row0, rows;            // expert, first row (grouped order) and number of rows
  int n_tile, n0;               // tile column and its first output column
  int m_loc, n_loc;             // place inside the super tile
  int part, klen;               // contraction part and its length
  int slot;                     // thread m < BM: slot of row m of the tile, where one is needed
};

// Columns of a tile's column operand in LDS, if it is read transposed: tiles of 192 columns keep the layout of 256 and do not
// multiply the last 64 (which repeat column 0: one more request of a piece that is there).
template <class TL>
static constexpr int column_extent = TL::BN == 192 ? 256 : TL::BN;

// One output tile; TL::BM >= rows.
template <typename T, class TL, bool B_TR>
__device__ __forceinline__ void s2s_tile(const S2SArgs& a, const S2STile& t, int n_tiles, char* lds, int64_t* sDst,
                                         const int* sSrc, float* sBias) {
  typedef DirectOp<TL::BM, TL::NT> AOp;
  // Ring classes serve launches with at most a tile row or two per expert: (nearly) every weight element is read
  // once, and with the non-temporal hint it does not push the token rows, which every workgroup of a tile row reads,
  // out of the L2s (hint extended from the 32-/64-row classes to all ring classes: Mixtral layer forward at 256 /
  // 384 / 448 tokens 0.539 -> 0.505 / 0.559 -> 0.526 / 0.711 -> 0.688 ms, neutral from 768 tokens on)
  constexpr bool W_ONCE = TL::ONCE || TL::NS > 2 || (TL::WG > 1 && !TL::PAIR);
  typedef typename std::conditional<B_TR, TransOp<column_extent<TL>, TL::NT, W_ONCE, false, TL::RS>, DirectOp<TL::BN, TL::NT, W_ONCE>>::type BOp;
  constexpr bool LAST_TILES = TL::BM == 128 && TL::BN == 256 && TL::NS == 3;
  constexpr bool CAN_SPLIT = LAST_TILES || TL::RS;
  const int glu = TL::RS ? __builtin_amdgcn_readfirstlane(a.glu) : -1;      // (as for the tile in s2s_mfma_kernel)
  const int e = t.e, row0 = t.row0, rows = t.rows, n0 = t.n0;
  const int k_first = CAN_SPLIT ? t.part * a.k_part : 0;

  AOp A;
  A.rot = TL::RS ? 0 : (t.n_loc * AOp::R / (TL::PAIR ? 2 * Raster::SN : Raster::SN)) % AOp::R;    // the row panel has SN sharers
  // Lane offsets are 32-bit: grouped input rows are taken relative to the tile's first row (so that the input may
  // be of any size), gathered ones relative to the start of the token matrix.
  const int64_t sxm = a.sxm;
  const int src0 = a.x_grouped ? row0 : 0;
  const char* Xb = (const char*)a.X + ((int64_t)src0 * sxm + k_first) * 2;
  A.init(Xb, [&](int row) { return (int64_t)(sSrc[row] - src0) * sxm * 2; });
  BOp B;
  B.rot = TL::RS ? 0 : (t.m_loc * BOp::R / Raster::SM) % BOp::R;    // the column panel has SM sharers
  const char* Wb = (const char*)a.W + ((int64_t)e * a.swe + (int64_t)k_first * (B_TR ? a.swk : 1)) * 2;
  if ((TL::RS ? glu : a.glu) == 1) {
    // tile column tc -> weight column: wave block tc / WTN, first half of the block from [0, F), second from [F, 2F)
    const int F = a.N;
    auto wcol = [&](int tc) {
      const int j = tc % TL::WTN;
      const int hc = n0 + (tc / TL::WTN) * (TL::WTN / 2) + j % (TL::WTN / 2);
      return hc < F ? hc + (j >= TL::WTN / 2 ? F : 0) : 0;
    };
    if constexpr (B_TR) {
      B.init_cols(Wb, a.swk * 2, wcol);
    } else {
      const int64_t swn = a.swn;
      B.init(Wb, [&](int row) { return (int64_t)wcol(row) * swn * 2; });
    }
  } else if constexpr (B_TR) {
    B.init(Wb + (int64_t)n0 * 2, a.swk * 2, TL::BN == 192 ? min(a.N - n0, TL::BN) : a.N - n0);
  } else {
    const int64_t swn = a.swn;
    const int N = a.N;
    B.init(Wb, [&](int row) { const int n = n0 + row < N ? n0 + row : N - 1; return (int64_t)n * swn * 2; });
  }

  Block acc[TL::FM][TL::FN];
  float rs[2 * TL::FM];
#pragma unroll
  for (int i = 0; i < TL::FM; ++i)
#pragma unroll
    for (int j = 0; j < TL::FN; ++j) acc[i][j].clear();
  if constexpr (TL::RS) mainloop_rs<T, TL, AOp, BOp>(A, B, t.klen, lds, acc);
  else if constexpr (TL::PAIR) mainloop_pair<T, TL, AOp, BOp, false>(A, B, a.K, lds, false, acc, rs);
  else if constexpr (TL::NS > 2) mainloop_ring<T, TL, AOp, BOp>(A, B, t.klen, lds, acc);
  else mainloop<T, TL, AOp, BOp, false>(A, B, a.K, lds, false, acc, rs);

  if constexpr (TL::RS) {
    if (a.ksplit > 1) {
      // This part's sums of the tile's rows, in float32 (parts_sum_kernel adds the parts)
      const int tx = late_thread<TL>(), wave = tx >> 6, l = tx & 63;
      const int wm = wave / TL::WN, wn = wave % TL::WN;
      float* P = a.partial + ((int64_t)t.part * a.L + row0) * a.N + n0;
#pragma unroll
      for (int i = 0; i < 2 * TL::FM; ++i) {
        const int m = wm * TL::WTM + i * 16 + (l & 15);
        if (m >= rows) continue;
#pragma unroll
        for (int j = 0; j < 2 * TL::FN; ++j) {
          const int n = wn * TL::WTN + (j >> 1) * 32 + block_col(l, j & 1);
          const f32x4 v = accumulators<TL>(acc[i >> 1][j >> 1].q[2 * (i & 1) + (j & 1)]);
          if (n0 + n < a.N) *(f32x4*)(P + (int64_t)m * a.N + n) = v;
        }
      }
      return;
    }
  }
  if constexpr (LAST_TILES) {
    if (a.ksplit > 1) {
      // This part's accumulators as they lie in the registers, 16 bytes per lane and store (whole 1 KB runs per
      // wave); splitk_reduce_kernel knows which output element each of them belongs to.
      f32x4* P = (f32x4*)a.partial +
                   (((int64_t)e * n_tiles + t.n_tile) * a.ksplit + t.part) * (TL::FM * TL::FN * 4 * TL::NT);
#pragma unroll
      for (int i = 0; i < TL::FM; ++i)
#pragma unroll
        for (int j = 0; j < TL::FN; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            P[((i * TL::FN + j) * 4 + g) * TL::NT + threadIdx.x] = acc[i][j].q[g];
      return;
    }
  }

  {
    int slot = t.slot;
    asm volatile("" : "+v"(slot));                          // not looked at before this point
    const int m = threadIdx.x;
    if (m < TL::BM) sDst[m] = m < rows ? (int64_t)(a.y_grouped ? row0 + m : slot) * a.sym : -1;
  }
  __syncthreads();
  const T* bias = a.b ? (const T*)a.b + (int64_t)e * a.sbe : nullptr;
  // 16-byte pieces need every row start 16-byte aligned; otherwise the lane-wise epilogues are used (the
  // one-wave-per-SIMD class is only launched on aligned outputs)
  if constexpr (TL::RS) {
    // (staged here, once for all epilogues: a copy of the walk over 256 accumulators in each costs registers ahead of them)
    stage_accumulators<T, TL>(acc, lds, [&](int tc) {
      if constexpr (TL::BN != 192) {
        if (glu == 1) return glu_bias<T, TL>(a, bias, n0, tc);
      }
      return glu == 0 || glu == 3 ? plain_bias<T>(bias, a.sbn, a.N, n0 + tc) : 0.0f;
    }, sBias);
    if (glu == 0) epilogue_staged<T, TL>(acc, (T*)a.Y, sDst, n0, a.N, bias, a.sbn, lds);
    else if (glu == 2) epilogue_glu_bwd_staged<T, TL>(acc, a, row0, rows, n0, lds);
    else if (glu == 4) epilogue_oss_bwd_staged<T, TL>(acc, a, row0, rows, n0, lds);
    if constexpr (TL::BN != 192) {                          // (192 columns: not the forward units, see narrow_columns)
      if (glu == 1) epilogue_glu_fwd_staged<T, TL>(acc, a, row0, rows, n0, bias, lds);
      else if (glu == 3) epilogue_oss_fwd_staged<T, TL>(acc, a, row0, rows, n0, bias, lds);
    }
  } else if (a.glu == 0) {
    const bool al16 = (((uintptr_t)a.Y & 15) == 0) && ((a.sym | a.N) & 7) == 0;
    if (al16) epilogue_staged<T, TL>(acc, (T*)a.Y, sDst, n0, a.N, bias, a.sbn, lds);
    else epilogue<T, TL>(acc, (T*)a.Y, sDst, n0, a.N, bias, a.sbn);
  } else if (a.glu == 1) {
    const bool al16 = ((((uintptr_t)a.Y | (uintptr_t)a.H) & 15) == 0) && ((a.sym | a.shm | a.N) & 7) == 0;
    if (al16) epilogue_glu_fwd_staged<T, TL>(acc, a, row0, rows, n0, bias, lds);
    else epilogue_glu_fwd<T, TL>(acc, a, row0, rows, n0, bias);
  } else if (a.glu == 2) {
    const bool al16 = ((((uintptr_t)a.aux | (uintptr_t)a.Y) & 15) == 0) && ((a.saux | a.sym | a.N) & 7) == 0;
    if (al16) epilogue_glu_bwd_staged<T, TL>(acc, a, row0, rows, n0, lds);
    else epilogue_glu_bwd<T, TL>(acc, a, row0, rows, n0);
  } else if (a.glu == 3) {
    epilogue_oss_fwd_staged<T, TL>(acc, a, row0, rows, n0, bias, lds);      // alignment checked by the launcher
  } else {
    epilogue_oss_bwd_staged<T, TL>(acc, a, row0, rows, n0, lds);
  }
}

// A tile of at most TL::BM = 256 rows.  An expert's last tile is partly filled: it is multiplied at the height of its rows, in
// steps of 64 (which keep the four waves, or the eight, equally busy), not as a whole tile.  (Same sums in the same order.)
// What it buys is that such tiles need no launch of their own any more (see cut_tails); a training step with many
// tiles per expert is the same with it (Mixtral shape, 16.5 tiles per expert).
template <typename T, class TL, bool B_TR>
__device__ __forceinline__ void s2s_tile_at_height(const S2SArgs& a, const S2STile& t, int n_tiles, char* lds, int64_t* sDst,
                                                   const int* sSrc, float* sBias) {
  const int h = (t.rows + 63) >> 6;
  if (h == 4) s2s_tile<T, TL, B_TR>(a, t, n_tiles, lds, sDst, sSrc, sBias);
  else if (h == 3) s2s_tile<T, typename TL::template Height<3>, B_TR>(a, t, n_tiles, lds, sDst, sSrc, sBias);
  else if (h == 2) s2s_tile<T, typename TL::template Height<2>, B_TR>(a, t, n_tiles, lds, sDst, sSrc, sBias);
  else s2s_tile<T, typename TL::template Height<1>, B_TR>(a, t, n_tiles, lds, sDst, sSrc, sBias);
}

template <typename T, class TL, bool B_TR>
__global__ __launch_bounds__(TL::NT, TL::WAVES_PER_SIMD) void s2s_mfma_kernel(S2SArgs a, Raster rast) {
  // (a workgroup that shares its CU's LDS with one other keeps its row tables where operands are to come: the source rows in
  // the second row stage, which is requested behind a barrier that follows their last reading, the output rows in the
  // column stage)
  constexpr int STAGE = (TL::BM + (B_TR ? column_extent<TL> : TL::BN)) * 128;
  static_assert(TL::BM * TL::BN * 2 <= (TL::PAIR ? PAIR_B : TL::NS * STAGE), "staged tile must fit the operand buffers");
  __shared__ __attribute__((aligned(16))) char lds[TL::PAIR ? PAIR_LDS : TL::NS * STAGE];
  __shared__ int64_t sDst_[TL::PAIR ? 1 : TL::BM];
  __shared__ int sSrc_[TL::PAIR ? 1 : TL::BM];
  __shared__ __attribute__((aligned(16))) float sBias_[TL::RS ? TL::BN : 4];
  int64_t* sDst = TL::PAIR ? (int64_t*)(lds + PAIR_B) : sDst_;
  int* sSrc = TL::PAIR ? (int*)(lds + PAIR_STAGE) : sSrc_;
  float* sBias = TL::PAIR ? nullptr : sBias_;

  // Contraction parts of the experts' last tiles: the grid is `ksplit` copies of the raster, copy c multiplies the c-th part of the
  // contraction (a raster is a multiple of 8 workgroups, so the XCD of a workgroup is still its first index modulo 8)
  constexpr bool LAST_TILES = TL::BM == 128 && TL::BN == 256 && TL::NS == 3;
  // (the parts are the grid's second dimension; no division here: the compiler would do it in the vector unit and
  // everything derived from it, loop counters and LDS addresses included, would leave the scalar registers)
  S2STile t;
  t.part = LAST_TILES ? (int)blockIdx.y : 0;
  int m_tile;
  int found = -1;
  if (TL::RS && a.ksplit > 1) {
    // Contraction parts of a whole product, at most a round of workgroups: the tiles that there are, one part after another, so
    // that every XCD, and every shader engine in it, has its share (workgroups without a tile between them, or columns in
    // stripes, and some CUs have two: 4 experts x 628 rows, 8512 -> 1664, 252 workgroups 163, 144 -> 113 us)
    const int tiles = count_tile_rows<TL::BM>(a.off, a.E) * rast.n_tiles;
    t.part = __builtin_amdgcn_readfirstlane(tiles > 0 ? (int)blockIdx.x / tiles : a.ksplit);
    if (t.part >= a.ksplit) return;
    const int in = (int)blockIdx.x - t.part * tiles;
    m_tile = __builtin_amdgcn_readfirstlane(in / rast.n_tiles);
    t.n_tile = in - m_tile * rast.n_tiles;
    t.m_loc = t.n_loc = 0;
    found = find_tile<TL::BM>(a.off, a.E, m_tile, t.e, t.row0, t.rows) ? 1 : 0;
    if (found == 0) return;
  } else if (rast.chunked) {
    t.m_loc = t.n_loc = 0;
    found = find_tile_chunked<TL::BM, TL::BM == 256 && (TL::BN == 256 || TL::RS || TL::PAIR)>(a.off, a.E, blockIdx.x, rast.n_tiles,
                                                                      rast.chunked == 2 ? TL::WG * 256 : 0,
                                                                      t.e, t.row0, t.rows, t.n_tile);
    if (found == 0) return;
  }
  t.klen = (LAST_TILES || TL::RS) && a.ksplit > 1 ? min(a.k_part, a.K - t.part * a.k_part) : a.K;
  if (found < 0 && !rast.map<TL::PAIR ? 2 * Raster::SN : Raster::SN>(blockIdx.x, m_tile, t.n_tile, t.m_loc, t.n_loc)) return;
  if (found > 0) {
    // looked up above
  } else if (a.tail_mode == 2) {
    // one tile row per expert: the rows its last 256-row tile would hold, when there are at most BM of them
    t.e = m_tile;
    if (!find_remainder<256>(a.off, a.E, t.e, TL::BM, t.row0, t.rows)) return;
  } else if (m_tile >= a.m_count ||
             !find_tile<TL::BM>(a.off, a.E, a.m_begin + m_tile, t.e, t.row0, t.rows, a.tail_mode == 1 ? REMAINDER_ROWS : 0)) {
    return;
  }
  if constexpr (TL::RS) {      // (one scalar value each, said so: ten registers of this form go to scratch memory otherwise)
    t.e = __builtin_amdgcn_readfirstlane(t.e);
    t.row0 = __builtin_amdgcn_readfirstlane(t.row0);
    t.rows = __builtin_amdgcn_readfirstlane(t.rows);
    t.n_tile = __builtin_amdgcn_readfirstlane(t.n_tile);
  }
  // first output column of the tile; the fused forward GLU tile holds BN/2 columns of each half
  t.n0 = a.glu == 1 ? t.n_tile * (TL::BN / 2) : t.n_tile * TL::BN;

  // Row tables, one tile row per thread.  The main loop needs only the source rows; where the output rows go is
  // stored after it, so that a launch whose input is grouped and whose output is not (layer-2 forward, layer-1
  // input gradient) does not wait for the index vector before its first operand loads.
  static_assert(TL::BM <= TL::NT, "one row of the tables per thread");
  t.slot = 0;                                               // idx[n] (< L, an int) where it is needed, else unused
  {
    const int m = threadIdx.x;
    if (m < TL::BM) {
      const int row = t.row0 + (m < t.rows ? m : t.rows - 1);      // tail rows re-read the last valid row
      if (!a.x_grouped || !a.y_grouped) t.slot = (int)a.idx[row];
      sSrc[m] = a.x_grouped ? row : (int)((unsigned)t.slot / (unsigned)a.fan_out);
    }
  }
  __syncthreads();
  if constexpr (TL::BM == 256 && (TL::BN == 256 || TL::RS || TL::PAIR)) {
    if constexpr (TL::RS || TL::PAIR) {
      if (rast.once && (int)a.off[t.e] - (t.e ? (int)a.off[t.e - 1] : 0) <= TL::BM) {
        s2s_tile_at_height<T, typename TL::Once, B_TR>(a, t, rast.n_tiles, lds, sDst, sSrc, sBias);
        return;
      }
    }
    s2s_tile_at_height<T, TL, B_TR>(a, t, rast.n_tiles, lds, sDst, sSrc, sBias);
  } else {
    s2s_tile<T, TL, B_TR>(a, t, rast.n_tiles, lds, sDst, sSrc, sBias);
  }
}

// Second half of a product whose last tiles were multiplied in contraction parts: one workgroup per (expert, tile
// column) with the thread layout of the 128 x 256 class, so that thread t finds the accumulators that thread t of
// every part left behind.  The parts are added in ascending order (the same result on every run), then bias,
// rounding and the scatter of the rows as in the plain epilogue.
template <typename T>
__global__ __launch_bounds__(512) void splitk_reduce_kernel(S2SArgs a, int n_tiles) {
  typedef Tile<128, 256, 2, 4, 3> TL;
  typedef T T4 __attribute__((ext_vector_type(4)));
  const int e = blockIdx.y, n_tile = blockIdx.x;
  int row0, rows;
  if (!find_remainder<256>(a.off, a.E, e, TL::BM, row0, rows)) return;
  const int wave = threadIdx.x >> 6, l = lane_id();
  const int wm = wave / TL::WN, wn = wave % TL::WN;
  const f32x4* P = (const f32x4*)a.partial + ((int64_t)e * n_tiles + n_tile) * a.ksplit * (TL::FM * TL::FN * 4 * TL::NT);
  const T* bias = a.b ? (const T*)a.b + (int64_t)e * a.sbe : nullptr;
  T* out = (T*)a.Y;
  const bool base_ok = ((uintptr_t)out & 7) == 0;
#pragma unroll
  for (int i = 0; i < TL::FM; ++i) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int m = wm * TL::WTM + i * 32 + block_row(l, g);
      if (m >= rows) continue;
      const int64_t row = row0 + m;
      const int64_t d = (a.y_grouped ? row : a.idx[row]) * a.sym;
#pragma unroll
      for (int j = 0; j < TL::FN; ++j) {
        const int n = n_tile * TL::BN + wn * TL::WTN + j * 32 + block_col(l, g);
        if (n >= a.N) continue;
        const int slot = ((i * TL::FN + j) * 4 + g) * TL::NT + threadIdx.x;
        f32x4 v = P[slot];
        for (int c = 1; c < a.ksplit; ++c) v += P[(int64_t)c * (TL::FM * TL::FN * 4 * TL::NT) + slot];
        if (bias != nullptr) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (n + q < a.N) v[q] += to_f32(bias[(int64_t)(n + q) * a.sbn]);
        }
        if (base_ok && n + 3 < a.N && ((d + n) & 3) == 0) {
          *(T4*)(out + d + n) = T4{from_f32<T>(v[0]), from_f32<T>(v[1]), from_f32<T>(v[2]), from_f32<T>(v[3])};
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (n + q < a.N) out[d + n + q] = from_f32<T>(v[q]);
        }
      }
    }
  }
}

// Second half of a product whose contraction was cut into parts as a whole: one wave per 512 columns of a row adds the parts up in
// ascending order (the same result on every run), then bias, rounding and the scatter of the row.
template <typename T>
__global__ __launch_bounds__(256) void parts_sum_kernel(S2SArgs a) {
  typedef T T8 __attribute__((ext_vector_type(8)));
  const int pieces = (a.N + 511) / 512;                               // per row, one per wave
  const int w = (int)(blockIdx.x * 4 + wave_uniform_id());
  const int row = __builtin_amdgcn_readfirstlane(w / pieces);
  const int n = ((w - row * pieces) * 64 + lane_id()) * 8;
  if (row >= (int)a.off[a.E - 1]) return;                             // (rows without an expert are written by nobody)
  int e = 0;
  if (a.b != nullptr) {
    for (int c = 0; c < a.E; c += 64) e += __popcll(__ballot(c + lane_id() < a.E && a.off[c + lane_id()] <= row));
  }
  if (n >= a.N) return;
  const float* P = a.partial + (int64_t)row * a.N + n;
  f32x4 v[2] = {*(const f32x4*)P, *(const f32x4*)(P + 4)};
  for (int c = 1; c < a.ksplit; ++c) {
    P += (int64_t)a.L * a.N;
    v[0] += *(const f32x4*)P;
    v[1] += *(const f32x4*)(P + 4);
  }
  T8 y;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float x = v[q >> 2][q & 3];
    if (a.b != nullptr) x += to_f32(((const T*)a.b)[(int64_t)e * a.sbe + (int64_t)(n + q) * a.sbn]);
    y[q] = from_f32<T>(x);
  }
  *(T8*)((T*)a.Y + (a.y_grouped ? (int64_t)row : a.idx[row]) * a.sym + n) = y;
}

static constexpr int NUM_CU = 256;
// expected number of 256-row tiles for rows spread evenly over the experts (binomial spread around the mean), rounded;
// `skip_small`: without the experts' last tiles of at most that many rows
static double expected_row_tiles(int64_t L, int E, int skip_small = 0) {
  const double avg = (double)L / E, sd = sqrt(avg * (1.0 - 1.0 / E)) + 1e-9;
  auto above = [&](double x) { return 0.5 * erfc((x - avg) / (sd * 1.41421356)); };      // P(rows > x)
  // expected ceil(rows / 256) = 1 + sum_j P(rows > 256 j); the terms more than 6 sd below the mean are 1
  const int j_lo = std::max(1, (int)((avg - 6 * sd) / 256.0));
  double per_expert = j_lo;
  for (int j = j_lo; j * 256.0 < avg + 6 * sd; ++j) per_expert += above(j * 256.0);
  if (skip_small > 0) {
    // minus P(rows mod 256 in [1, skip_small])
    for (int j = std::max(0, j_lo - 1); j * 256.0 < avg + 6 * sd; ++j)
      per_expert -= above(j * 256.0 + 0.5) - above(j * 256.0 + skip_small + 0.5);
  }
  return nearbyint(per_expert * E);
}

// An expert of one tile row has each weight read by one workgroup; with the non-temporal hint they leave the token rows in the L2s,
// as in the ring classes.  Only where the weights are more than the 256 MB of the memory-side cache: a program whose other data
// leaves them there finds them there (16 experts x 133 rows, 1024 -> 4960, 162 MB, launched again and again 46 -> 60 us; 64 x 120,
// 1024 -> 2048, 268 MB 57 -> 61).  An expert of several tile rows reads them from the L2 as often (8 x 300 rows, 4096 -> 14336 with the
// hint on its last tile 387 -> 447 us), hence by expert, asked where at least some are expected to have one.  us, without -> with the
// hint: 128 x 188 rows, 2048 -> 1536 209 -> 191, 768 -> 2048 122 -> 115; 128 x 250 rows 255 -> 230, 141 -> 130, gated 263 -> 240;
// 32 x 188 rows, 2880 -> 2880 148 -> 137, 2880 -> 5760 232 -> 227; 8 x 120 rows, 4096 -> 28672 364 -> 351, 8 x 194 475 -> 475.
static constexpr int64_t ONCE_MIN_WEIGHTS = 320ll << 20;
static constexpr int ONCE_BELOW_ROWS = 640;
static bool reads_weights_once(const S2SArgs& a) {
  return a.L / a.E < ONCE_BELOW_ROWS && (int64_t)a.E * a.K * 2 * (a.glu == 1 ? 2 : 1) * a.N >= ONCE_MIN_WEIGHTS;
}

template <typename T, class TL>
static int launch_s2s(const S2SArgs& a, bool b_tr, hipStream_t st) {
  const int bn = a.glu == 1 ? TL::BN / 2 : TL::BN;     // output columns per tile
  const int n_tiles = (a.N + bn - 1) / bn;
  const int64_t m_tiles = a.tail_mode == 2 ? a.E : std::min<int64_t>(max_tiles(a.L, a.E, TL::BM) - a.m_begin, a.m_count);
  // With only a few tile rows per expert no weight panel is shared by the tile rows of a super tile; the striped
  // order at least keeps the tile rows of one expert together on one XCD.
  const bool striped = TL::NS > 2 || a.L / a.E < STRIPE_BELOW;
  Raster r = striped ? make_striped(m_tiles, n_tiles, GM_RING) : make_raster(m_tiles, n_tiles, GM_S2S, TL::PAIR ? 2 * Raster::SN : Raster::SN);
  const bool whole = a.m_begin == 0 && a.m_count == 0x7fffffff && a.tail_mode == 0;
  const int64_t chunked = chunked_grid(m_tiles * n_tiles);
  const bool whole_parts = TL::RS && a.ksplit > 1;                      // (parts one after another, see s2s_mfma_kernel)
  if (whole_parts) r.grid_size = m_tiles * n_tiles * a.ksplit;
  else if (whole && a.L / a.E < CHUNK_BELOW && chunked <= 0x7fffffffLL) {
    r.chunked = TL::NS > 2 || (TL::WG > 1 && !TL::PAIR) || a.L / a.E < ROWS256_BELOW ? 1 : 2;
    r.grid_size = std::max(r.grid_size, chunked);
  }
  r.once = reads_weights_once(a);
  const int64_t grid = r.grid();
  const unsigned parts = a.ksplit > 1 && !whole_parts ? (unsigned)a.ksplit : 1u;
  if (grid > 0x7fffffffLL || m_tiles > 0x7fffffffLL) { set_error("smoe_scatter2scatter: grid too large"); return SMOE_ERR_RANGE; }
  if constexpr ((TL::BN % 128 == 0 || TL::RS) && (SMOE_LAYOUTS & 2)) {
    if (b_tr) {
      hipLaunchKernelGGL((s2s_mfma_kernel<T, TL, true>), dim3((unsigned)grid, parts), dim3(TL::NT), 0, st, a, r);
      return launch_status("s2s_mfma_kernel");
    }
  }
  if constexpr (SMOE_LAYOUTS & 1) hipLaunchKernelGGL((s2s_mfma_kernel<T, TL, false>), dim3((unsigned)grid, parts), dim3(TL::NT), 0, st, a, r);
  return launch_status("s2s_mfma_kernel");
}

// A launch of a few whole rounds plus a remainder of up to half a round pays a whole round for the remainder.
// Such a product is cut by tile rows: the whole rounds stay with the 256 x 256 class, the remaining tile rows go
// to a second launch of 256 x 128 tiles (twice the workgroups, 0.58 of the time).  Returns the number of tile
// rows of the first launch, 0 when the product is not split.  Plain products only (no fused unit behind them).
// Mixtral shape, 16384 tokens (8.25 rounds in the launches with 4096 output columns): layer-2 forward
// 3.47 -> 3.34 ms, layer-1 input gradient 7.03 -> 6.68 ms; 128 x 128 tiles for the remainder were slower
// (four times the workgroups at 0.75 of the time).  With few tile rows per expert the heights of the partly filled
// tiles decide, not their number (one launch is then as fast or faster: 32 experts x 262 rows, 5760 -> 2880
// 484 -> 456 us; 8 experts x 500 rows, 14336 -> 4096 631 -> 605), with many it pays (8 x 1000 rows 916 -> 884).
static constexpr int TAIL_SPLIT_MIN_AVG_ROWS = 640;
static int tail_split(const S2SArgs& a) {
  if (a.glu != 0 || a.m_begin != 0 || a.L / a.E < TAIL_SPLIT_MIN_AVG_ROWS) return 0;
  const int64_t n_full = (a.N + 255) / 256;
  const int64_t upper = max_tiles(a.L, a.E, 256);
  if (upper * n_full > 26 * NUM_CU) return 0;
  const double m = expected_row_tiles(a.L, a.E, a.tail_mode == 1 ? REMAINDER_ROWS : 0);
  const int64_t whole = (int64_t)(m * n_full) / NUM_CU;           // whole rounds
  if (whole < 2) return 0;
  const int64_t m_first = whole * NUM_CU / n_full;                // tile rows that fit the whole rounds
  const int64_t rest = ((int64_t)m - m_first) * n_full;           // expected 256 x 256 tiles of the remainder
  // (no remainder expected: the second launch still stands by for a tile row more than expected, which would
  // otherwise cost the first launch a whole round; its workgroups exit at once when there is none)
  if (m_first <= 0 || rest < 0 || upper <= m_first || rest > NUM_CU / 2 + 8) return 0;
  return (int)m_first;
}

// The 256 x 256 class.  Products with a long enough contraction run on the one-wave-per-SIMD form of it
// (mainloop_rs: Mixtral shape, per 64-deep slice 2 300-2 420 cycles against 2 890-3 000; its prologue and its
// epilogue, run by half as many threads, cost about 5 000 cycles more per tile, which a 12-slice contraction does not
// earn back: K = 768 is 5 % slower, K = 1536 even, K = 2048 is 5-8 % faster).
// Both forms add up every output element in the same order: the same bits.
static constexpr int RS_MIN_K = 1792;
static constexpr int RS_XTY_MIN_ROWS = 2048;      // groupXtY: average rows per expert from which that form is used,
static constexpr int RS_XTY_MIN_ROWS_ROUNDS = 1280, RS_XTY_ROUNDS = 4;      // and from which with so many rounds of tiles
// Whole slices, and output pieces of 16 bytes: what the one-wave-per-SIMD form and the paired tiles take.
static bool whole_pieces(const S2SArgs& a) {
  bool al16 = true;
  if (a.glu == 0) al16 = (((uintptr_t)a.Y & 15) == 0) && ((a.sym | a.N) & 7) == 0;
  else if (a.glu == 1) al16 = ((((uintptr_t)a.Y | (uintptr_t)a.H) & 15) == 0) && ((a.sym | a.shm | a.N) & 7) == 0;
  else if (a.glu == 2) al16 = ((((uintptr_t)a.aux | (uintptr_t)a.Y) & 15) == 0) && ((a.saux | a.sym | a.N) & 7) == 0;
  return al16 && a.K % BK == 0;
}
// Contractions of fewer than 1792 go in 256 x 128 tiles, two workgroups per CU (mainloop_pair).  The shorter the contraction
// the more of a 256 x 256 tile's time is what it does before and behind its loop; launches of one to three rounds gain most,
// their rounds being half as long.  590 random launches of 112 to 4000 rows per expert, K and N from 256 to 6000, plain and
// with every fused unit, against eight waves per 256 x 256 tile (us): K below 512 1.13 times as fast on average, below 1024
// 1.10, from there 1.05, one in thirty more than 3 % slower; 256 to 768 tiles of 256 x 256 1.16.  16 experts x 1000 rows,
// 1024 -> 1024 60 -> 48; 64 x 500, 512 -> 512 39 -> 34; 128 x 2048, 768 -> 2048 963 -> 943, 1536 -> 2048 1687 -> 1673.  (Both
// forms are held by the power cap there: a launch of K = 64 takes what its stores take, and every slice adds 63 us, 1.1 PFLOP/s.)
// Longer contractions: the one-wave-per-SIMD form reads half as much from LDS per product; K from 2048 0.97, 8 x 4096 rows,
// 14336 -> 4096 2957 -> 3216.
// Tiles half as wide have twice the edges, and where output rows are no whole number of 64-byte pieces (the unit memory is written
// in) two tiles share one at every edge.  What the gated units write, up to three times as wide as their products, then costs more
// than the tiles save, the more the shorter the contraction.  4400 random launches of more than half a round, times as fast (more
// than 3 % slower), even loads, rows of whole pieces / ragged: gated forward that saves its pre-activation 1.09 (3 of 357) /
// 0.97 (373 of 816; 64 experts x 230 rows, 64 -> 6952 325 -> 509 us, 32 x 699, 64 -> 2632 155 -> 223), its gradient 1.10 (2 of 328) /
// 1.02 (211 of 772; below 400 0.95), the interleaved unit's forward 1.12 (2 of 115) / 1.04 (8 of 64; from 1024 on 1.06, below 0.99), its
// gradient 1.10 / 1.08, forward passes that save nothing 1.15 / 1.11, plain 1.14 (9 of 492) / 1.08 (32 of 908; contractions of up to 128
// 1.05, 7 of 49).  Loads as 1 / rank^0.84 and 1 / rank^1.8: whole pieces 1.03 to 1.11, ragged 0.91 to 0.97 gated, 1.03 to 1.07 the others.
typedef Tile<256, 128, 2, 2, 2, false, 2, true> PairTile;
static bool takes_pairs(const S2SArgs& a) {
  if (a.K >= RS_MIN_K || !whole_pieces(a)) return false;
  const bool saves = a.Y != nullptr;
  int64_t in = (int64_t)((uintptr_t)a.Y & 63) >> 1 | (saves ? a.sym : 0);              // elements; whole pieces: multiples of 32
  if (a.glu == 1 || a.glu == 3) in |= (int64_t)((uintptr_t)a.H & 63) >> 1 | a.shm;
  if (a.glu == 1 || a.glu == 2) in |= a.N;                                        // the second half's first column
  if ((in & 31) == 0) return true;
  if ((a.glu == 1 && saves) || a.glu == 2) return false;
  return a.K >= (a.glu == 3 && saves ? 1024 : 192);
}

// Few rows per expert: tiles of 192 columns in place of 256 where they take no more rounds of a workgroup per CU, a round being a
// quarter shorter in products and weights.  Plain products and the gated units' gradients; the forward units have not been measured in
// them.  us, 256 -> 192 columns (rounds): 32 experts x 188 rows, 2880 -> 2880 149 -> 131 (1.5 -> 1.9), 5760 -> 2880
// 258 -> 240; 64 x 130, 2048 -> 2064 160 -> 146 (2.3 -> 2.8); 64 x 147, 2880 -> 1488 137 -> 120 (1.5 -> 2.0); 8 x 133, 4096 -> 5176
// 87 -> 76 (0.7 -> 0.8).  A round more loses (64 x 139, 2048 -> 1816 135 -> 141; 32 x 188, 2880 -> 5760 240 -> 254), and with several
// tile rows per expert the operands' LDS traffic per product counts (32 x 1024, 2880 -> 2880, 6 % less padding, 550 -> 574;
// 128 x 438, 4096 -> 2288 1180 -> 1345).  16 launches that take it, most of them random, before the instruction and the order of this
// class changed -> now: even loads 1.21 times as fast (1.09 to 1.32), as 1 / rank^0.3 1.16 (1.06 to 1.26), ^0.42 1.13 (0.92 to 1.26),
// ^0.84 1.10 (0.93 to 1.21), ^1.8 1.08 (0.97 to 1.18).  Under uneven loads nobody knows the tile rows here: what loses are launches whose
// last round was full to the brim (32 x 172, 3072 -> 2536, 37 tile rows for 32 expected, 518 tiles, 156 -> 169).
static constexpr int NARROW_MAX_ROUNDS = 4;
static bool narrow_columns(const S2SArgs& a) {
  if ((a.glu != 0 && a.glu != 2 && a.glu != 4) || a.m_begin != 0 || a.m_count != 0x7fffffff || a.tail_mode != 0) return false;
  if (a.L / a.E >= ROWS256_BELOW) return false;
  const double rows = expected_row_tiles(a.L, a.E);
  const int64_t wide = (int64_t)(rows * ((a.N + 255) / 256)), narrow = (int64_t)(rows * ((a.N + 191) / 192));
  const int64_t rounds = (narrow + NUM_CU - 1) / NUM_CU;
  return rounds <= NARROW_MAX_ROUNDS && rounds == (wide + NUM_CU - 1) / NUM_CU;
}
template <typename T>
int launch_narrow(const S2SArgs& a, bool b_tr, hipStream_t st);        // gemm_mfma_xty.hip

template <typename T>
static int launch_main_class(const S2SArgs& a, bool b_tr, hipStream_t st) {
  // (its buffer descriptors end with the last row of a strided operand: rows that overlap, as those of an expanded tensor, would
  // read as zeros)
  const bool apart = !b_tr || a.swk >= (a.glu == 1 ? 2 : 1) * (int64_t)a.N;
  if (a.K >= RS_MIN_K && whole_pieces(a) && apart && narrow_columns(a)) return launch_narrow<T>(a, b_tr, st);
  if (a.K >= RS_MIN_K && whole_pieces(a) && apart)
    return launch_s2s<T, Tile<256, 256, 2, 2, 2, true>>(a, b_tr, st);
  return launch_s2s<T, Tile<256, 256, 2, 4>>(a, b_tr, st);
}

// Products with many rows per expert and few tile columns (8 experts x 4096 rows x 16 tile columns) run in whole rounds
// of full tiles; the experts' last tiles of at most 128 rows would add a round of 64 to 128 workgroups that each walk
// the whole contraction.  With a caller workspace they are left to a launch of 128 x 256 tiles, one tile row per expert
// (which experts have such a tile is known only on the device: the launch covers all of them and the others'
// workgroups exit), with the contraction cut into parts, one workgroup each (tail_ksplit), and a small launch adds the
// parts up: float32 partial sums in a fixed order, so the result is the same on every run, but not the same bits as
// the unsplit product (its additions are grouped differently).  Everywhere else the last tiles stay with the others,
// at the height of their rows: next to the expert's other tiles they find the weights in the L2, which a launch of
// their own reads again (8 experts x 250 rows, 14336 -> 4096 505 -> 335 us, 4096 -> 2 x 14336 738 -> 636;
// 32 experts x 400 rows, 2880 -> 2 x 2880 541 -> 468; 128 x 250 rows, 2048 -> 2 x 768 301 -> 276).
static constexpr double REMAINDER_MIN_FLOP = 2e11;
static constexpr int REMAINDER_MIN_AVG_ROWS = 1536;
static constexpr int KSPLIT_MAX = 8;
static constexpr int KSPLIT_MIN_SLICES = 16;      // 64-deep slices a part must keep
static constexpr int64_t SPLITK_TILE_FLOATS = 128 * 256;

// Parts to cut the contraction of the last tiles into: enough for one workgroup per CU when half of the experts
// have such a tile; 1 = not split (also: no workspace, fused unit behind the product, ragged contraction).
static int tail_ksplit_for(int64_t K, int64_t N, int E, int glu) {
  if (glu != 0 || K % BK != 0) return 1;
  const int64_t n_tiles = (N + 255) / 256;
  const int64_t wgs = std::max<int64_t>(1, (int64_t)(E + 1) / 2 * n_tiles);
  int ks = 1;
  while (ks < KSPLIT_MAX && wgs * ks < NUM_CU && K % (BK * ks * 2) == 0 && K / (BK * ks * 2) >= KSPLIT_MIN_SLICES) ks *= 2;
  return ks;
}
static int64_t splitk_floats(int64_t N, int E, int ks) { return (int64_t)E * ((N + 255) / 256) * ks * SPLITK_TILE_FLOATS; }
static int tail_ksplit(const S2SArgs& a) {
  if (a.L / a.E < REMAINDER_MIN_AVG_ROWS) return 1;
  const int ks = tail_ksplit_for(a.K, a.N, a.E, a.glu);
  if (ks <= 1 || a.partial == nullptr || a.partial_floats < splitk_floats(a.N, a.E, ks)) return 1;
  return ks;
}

static bool cut_tails(const S2SArgs& a) {
  const bool whole = a.m_begin == 0 && a.m_count == 0x7fffffff && a.tail_mode == 0;
  if (!whole || 2.0 * (double)a.L * a.K * (a.glu == 1 ? 2.0 * a.N : (double)a.N) < REMAINDER_MIN_FLOP) return false;
  return tail_ksplit(a) > 1;
}

template <typename T>
static int launch_tails(const S2SArgs& a, bool b_tr, hipStream_t st) {
  typedef Tile<128, 256, 2, 4, 3> TailTile;
  S2SArgs rest = a;
  rest.tail_mode = 2;
  rest.ksplit = tail_ksplit(a);
  rest.k_part = a.K / rest.ksplit;
  if (const int rc = launch_s2s<T, TailTile>(rest, b_tr, st)) return rc;
  const int n_tiles = (a.N + 255) / 256;
  hipLaunchKernelGGL(splitk_reduce_kernel<T>, dim3((unsigned)n_tiles, (unsigned)a.E), dim3(512), 0, st, rest, n_tiles);
  return launch_status("splitk_reduce_kernel");
}

// Products of few tiles and a long contraction: the contraction of every tile is cut into parts, one workgroup of the
// one-wave-per-SIMD form each, which leave float32 sums; a second launch adds them up in a fixed order (parts_sum_kernel).  Without
// parts at most half of the CUs have a 256 x 256 tile, and 256 x 128 ring tiles hold a quarter of the loads in flight that the
// weights' stream needs.  The number of parts, and whether any, by the time that the parts and the classes below would take, in us:
// a slice of 64 costs 1.25 in a whole tile and 0.95 in a ring tile, or what the weights' stream does (5.2 and 4 TB/s); a
// workgroup's set-up and store 14 and 4; the sums their bytes at 4.5 TB/s, written and read.  Measured, us, without -> with (parts):
// 8 experts x 194 rows, 14336 -> 4096 241 -> 220 (2), 28672 -> 4096 478 -> 397 (2); 4 x 300, 14336 -> 4096 239 -> 196 (2); 2 x 500,
// 8192 -> 4096 116 -> 73 (4); 1 x 609, 10240 -> 1472 155 -> 47 (8); 8 x 200, 2048 -> 2048 33 -> 39, so not; a second round of
// workgroups loses as well (8 x 250, 14336 -> 4096 316 -> 361).  22 launches that take parts, 19 of them random, against the state
// before there were any: even loads 1.66 times as fast (1.00 to 3.05), as 1 / rank^0.3 1.73, ^0.42 1.72, ^0.84 1.69 (1.03 to 3.0), ^1.8
// 1.66 (0.94 to 2.8): of the 110 one is slower, whose loads make three tile rows more than expected and so a second round (16 x 888 rows,
// 11968 -> 280, 198 -> 211).
static constexpr int PARTS_MAX = 8;
static int part_length(int64_t K, int parts) { return (int)((K / BK + parts - 1) / parts) * BK; }
static int whole_parts_for(int64_t L, int64_t K, int64_t N, int E) {
  if (L / E < ROWS128_BELOW || K < RS_MIN_K || K % BK != 0 || N % 8 != 0) return 1;
  const double tiles = expected_row_tiles(L, E) * ((N + 255) / 256), weights = 2.0 * E * K * N * 1e-6, slices = (double)(K / BK);
  double least = 0.92 * (std::max(slices * 0.95, weights / 4.0) + 4);
  int best = 1;
  for (int p = 2; p <= PARTS_MAX && tiles * p <= NUM_CU; ++p) {
    const int len = part_length(K, p);
    if ((K + len - 1) / len != p) continue;                           // (no part is empty)
    const double t = std::max(len / BK * 1.25, weights / 5.2) + 14 + 8e-6 * L * N * p / 4.5;
    if (t < least) least = t, best = p;
  }
  return best;
}
static int whole_parts(const S2SArgs& a, bool b_tr) {
  const bool whole = a.m_begin == 0 && a.m_count == 0x7fffffff && a.tail_mode == 0;
  if (a.glu != 0 || !whole || a.partial == nullptr || !whole_pieces(a) || (b_tr && a.swk < a.N)) return 1;
  const int p = whole_parts_for(a.L, a.K, a.N, a.E);
  return a.partial_floats >= (int64_t)a.L * a.N * p ? p : 1;
}
template <typename T>
static int launch_parts(const S2SArgs& a, int parts, bool b_tr, hipStream_t st) {
  S2SArgs m = a;
  m.ksplit = parts;
  m.k_part = part_length(a.K, parts);
  if (const int rc = launch_s2s<T, Tile<256, 256, 2, 2, 2, true>>(m, b_tr, st)) return rc;
  const int64_t waves = (int64_t)a.L * ((a.N + 511) / 512);
  hipLaunchKernelGGL(parts_sum_kernel<T>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, m);
  return launch_status("parts_sum_kernel");
}

// A whole product in the 256-row classes: one launch, or whole rounds of 256 x 256 tiles plus a remainder of 256 x 128
// tiles (tail_split), the experts' sparsely filled last tiles apart (cut_tails).
template <typename T>
static int launch_main(const S2SArgs& a, bool b_tr, hipStream_t st) {
  if (takes_pairs(a)) return launch_s2s<T, PairTile>(a, b_tr, st);
  S2SArgs m = a;
  const bool tails = cut_tails(a);
  if (tails) m.tail_mode = 1;
  int rc;
  if (const int m_first = tail_split(m)) {
    S2SArgs first = m, rest = m;
    first.m_count = m_first;
    rest.m_begin = m_first;
    // both classes have 256-row tiles, hence the same numbering of the tile rows
    rc = launch_main_class<T>(first, b_tr, st);
    if (rc == 0) rc = launch_s2s<T, Tile<256, 128, 4, 2, 3>>(rest, b_tr, st);
  } else {
    rc = launch_main_class<T>(m, b_tr, st);
  }
  if (rc != 0 || !tails) return rc;
  return launch_tails<T>(a, b_tr, st);
}

static constexpr int MAIN_MIN_TILES = 160;
// Products whose 256 x 128 tiles fit one round of a workgroup per CU take those: the 256 x 256 ones would leave half of
// the chip idle for as long (us, 256 x 256 -> 256 x 128: 4 experts x 332 rows, 1280 -> 3328 36 -> 26; 8 x 1829,
// 10752 -> 448 224 -> 172; 32 x 438, 7616 -> 384 151 -> 118; 16 x 572, 10624 -> 448 191 -> 157; over 509 launches of
// 224 to 4000 rows per expert, a quarter of them at this line, 5.5 % on average; a second round of them loses).  The line
// is drawn for even loads; uneven ones go by column stripes (8 x 584 rows on average, 4640 -> 1272, 21 tile rows in ten
// columns 115 us).
static bool one_round_of_halves(const S2SArgs& a) {
  const int cols = a.glu == 1 ? 64 : 128;
  return expected_row_tiles(a.L, a.E) * ((a.N + cols - 1) / cols) <= NUM_CU;
}
static bool glu_fwd_pieces(const S2SArgs& a) {
  return a.glu != 1 || (((((uintptr_t)a.Y | (uintptr_t)a.H) & 15) == 0) && ((a.sym | a.shm | a.N) & 7) == 0);
}

// Fewer than 52 rows per expert: a stream over the weights of the experts that are hit, tiles of 64 or 32 rows.  What
// counts is weight bytes in flight across the chip, and that the filling of one tile's ring hides behind the stream of
// another: a workgroup that has the CU to itself (six 20 KB stages) leaves the memory idle
// while it looks its tile up, fills its ring and stores its result, for a tile of 512 KB (128 columns x 2048) about a
// fifth of its time.  Hence two or three workgroups per CU with shallower rings wherever the launch has that many.
// Measured (us, one 32 x 128 x 6 workgroup per CU -> now; weights streamed at):
//   128 experts x 12 rows, layer 1 of d = 2048, F = 768: 162 -> 140 (5.7 TB/s); layer 2: 91 -> 70 (5.7 TB/s)
//   32 experts x 6 rows, 2880 -> 2 x 2880 (N-contiguous): 169 -> 157 (6.8 TB/s); 2880 -> 2880: 88 -> 82
//   8 experts x 8 rows, layer 1 of d = 4096, F = 14336: 289 -> 275; 64 experts x 8 rows, 1024 -> 2 x 512: 29 -> 24
//   128 experts x 40 rows (64-row tiles, five stages -> three): 178 -> 156 and 106 -> 79
template <typename T>
static int dispatch_few_rows(const S2SArgs& a, bool b_tr, hipStream_t st) {
  const int64_t avg = a.L / a.E;
  const int bn = a.glu == 1 ? 64 : 128;                                   // output columns of a 128-wide tile
  const int64_t cols = (a.N + bn - 1) / bn, wgs = std::min<int64_t>(a.L, a.E) * cols;
  // Three two-stage workgroups per CU where that makes one round of what would be 1.5 rounds of two per CU
  // (us, two x three stages -> three x two: 64 x 11 tiles of K = 2048 80 -> 67, 16 x 44 74 -> 66, 32 x 23 of K = 2880
  // 89 -> 82, 16 x 44 of K = 4096 137 -> 124; with fewer tiles two stages are too few: 256 of K = 14336 147 -> 211), while
  // no expert is expected to need a second tile row, which would be a second round (three standard deviations; 32 x 23 of
  // K = 2880, two x three -> three x two: 40 rows per expert 91 -> 89, 44 rows 90 -> 89, 49 rows 113 -> 130)
  if (wgs > 2 * NUM_CU && wgs <= 3 * NUM_CU && avg + 3 * sqrt((double)avg) < 64) return launch_s2s<T, Tile<64, 128, 2, 2, 2, false, 3>>(a, b_tr, st);
  // Up to one workgroup per CU: deep rings.  At exactly one per CU N-contiguous weights are faster in two shallow ones
  // (us, deep -> shallow, 256 tiles: 8 x 30 rows, K = 14336 150 -> 141, K = 2048 27 -> 25; 32 x 30 rows, K = 2880 35 -> 33),
  // K-contiguous ones only with a short contraction (149 -> 153, 33.8 -> 32.7, 33.2 -> 32.2): deep.
  const bool few = b_tr ? wgs < NUM_CU : wgs <= NUM_CU;
  if (avg >= (few ? 24 : ROWS32_BELOW)) {
    if (few) return launch_s2s<T, Tile<64, 128, 2, 2, 5>>(a, b_tr, st);
    return launch_s2s<T, Tile<64, 128, 2, 2, 3, false, 2>>(a, b_tr, st);
  }
  // 32-row tiles have one column block per wave: the fused forward GLU only in its LDS-staged form (16-byte pieces)
  if (!glu_fwd_pieces(a)) return SMOE_ERR_UNSUPPORTED;
  if (!b_tr) {
    // K-contiguous weights: half-width tiles while 128-wide ones would not give every CU two workgroups (44 x 8 tiles
    // of K = 1024: 25 -> 17 us, 22 x 16 of K = 2048: 47 -> 39, 8 x 8 of K = 2816: 18 -> 16), and where 128-wide
    // columns do not divide evenly among the 8 XCDs, at most 3/4 of the last
    // row of eight in use (128 experts of K = 2048, uneven, before the stripes went on where they left off / evenly loaded, which take chunks: 9 columns 127 -> 116 /
    // 118 -> 106, 12 columns 164 -> 146 / 133 -> 131, 17 columns 214 -> 194 / 180 -> 179; 16 columns 213 -> 185 /
    // 165 -> 168, 32 columns 375 -> 356 / 329 -> 329: evenly loaded decides, being the ordinary case)
    if (wgs < 192) return launch_s2s<T, Tile<32, 64, 1, 2, 6>>(a, b_tr, st);
    if (wgs < 2 * NUM_CU || cols * 4 <= (cols + 7) / 8 * 8 * 3) return launch_s2s<T, Tile<32, 64, 1, 2, 4, false, 3>>(a, b_tr, st);
  } else if (few) {
    return launch_s2s<T, Tile<32, 128, 1, 4, 6>>(a, b_tr, st);
  }
  return launch_s2s<T, Tile<32, 128, 1, 4, 3, false, 2>>(a, b_tr, st);
}

template <typename T>
static int dispatch_s2s(const S2SArgs& a, bool b_tr, hipStream_t st) {
  // the gpt-oss epilogues exist only in their LDS-staged form (16-byte pieces)
  if (a.glu == 3 && !((((uintptr_t)a.Y & 15) | ((uintptr_t)a.H & 7)) == 0 && (a.sym & 7) == 0 && (a.shm & 3) == 0 &&
                      (a.N & 7) == 0))
    return SMOE_ERR_UNSUPPORTED;
  if (a.glu == 4 && !((((uintptr_t)a.aux | (uintptr_t)a.Y) & 15) == 0 && ((a.saux | a.sym | a.N) & 7) == 0))
    return SMOE_ERR_UNSUPPORTED;
  // the backward gated epilogues address a tile's output rows with 32-bit byte offsets from its first row
  if ((a.glu == 2 || a.glu == 4) && a.sym * 2 * 256 >= 0xffffffffLL) return SMOE_ERR_UNSUPPORTED;
  const int64_t avg = a.L / a.E;
  // 256 x 256 tiles, each at the height of its rows, from 112 rows per expert on if one tile row per expert gives most
  // CUs a workgroup (us against the 256 x 128 and 128-row ring classes: 32 experts x 125 rows, 2880 -> 2 x 2880
  // 269 -> 214, 5760 -> 2880 286 -> 254; 8 x 140, 4096 -> 11264 210 -> 181; 128 x 188, 2048 -> 768 with its gated unit's
  // gradient 168 -> 144; with half as many tiles as CUs, 8 x 188, 14336 -> 4096, 263 -> 288, even below 160 rows), from
  // 52 rows on where it makes one round of what the 128-row tiles do in two (16 x 90, 2048 -> 2 x 1408 56 -> 42; paired
  // tiles, of which twice as many make a round, up to two: 17 random launches of 52 to 112 rows 1.15 times as fast), and
  // from 224 rows on whatever the number of tiles, unless half-width ones fit one round.
  if (const int parts = whole_parts(a, b_tr); parts > 1) return launch_parts<T>(a, parts, b_tr, st);
  const int64_t tiles = (int64_t)a.E * ((a.N + (a.glu == 1 ? 127 : 255)) / (a.glu == 1 ? 128 : 256));
  if (avg >= ROWS256_BELOW && one_round_of_halves(a)) return launch_s2s<T, Tile<256, 128, 4, 2, 3>>(a, b_tr, st);
  if (avg >= ROWS256_BELOW || (avg >= ROWS128_BELOW && tiles >= MAIN_MIN_TILES) ||
      (avg >= ROWS64_BELOW && tiles > NUM_CU / 2 && tiles <= (takes_pairs(a) ? 2 : 1) * NUM_CU))
    return launch_main<T>(a, b_tr, st);
  // Below that the launch is a stream over the weights: tile height by rows per expert.  Launches with enough 256-wide
  // tile columns to fill the chip twice move half as many token rows per weight byte with 256-wide tiles as with
  // 128-wide ones (experts of about one 128-row tile, Mixtral layer 1: 448 tokens 518 -> 373 us).
  if (avg >= ROWS128_BELOW) return launch_s2s<T, Tile<256, 128, 4, 2, 3>>(a, b_tr, st);
  if (avg >= ROWS64_BELOW && tiles >= 2 * NUM_CU) return launch_s2s<T, Tile<128, 256, 2, 4, 3>>(a, b_tr, st);
  if (avg < ROWS64_BELOW) return dispatch_few_rows<T>(a, b_tr, st);
  // With one column block per wave the fused forward GLU exists only in its LDS-staged form (16-byte pieces)
  if (!glu_fwd_pieces(a)) return SMOE_ERR_UNSUPPORTED;
  return launch_s2s<T, Tile<128, 128, 2, 4, 3>>(a, b_tr, st);
}

// =====================================================================================================
// groupXtY:  OUT[e] (P x Q, Q contiguous) = sum_r  Pm[r, :]^T  Qm[r, :]   over the expert's rows
//   DW stored (E,N,K)-contiguous (the ParallelExperts layout):  P = dY (N cols), Q = X  (K cols)
//   DW stored (E,K,N)-contiguous:                              P = X  (K cols), Q = dY (N cols)
// Column sums of dY (the bias gradient) ride along: the first column of tiles adds up the dY fragments it
// already holds in registers.
// =====================================================================================================
struct XtYPlan {
  const void* P; int64_t ldp; int np;     // row-operand source: (L, np), leading dimension ldp elements
  const void* Q; int64_t ldq; int nq;     // column-operand source
  void* OUT; int64_t soe, sop;            // output: expert stride, row stride (columns contiguous)
  void* Db; int64_t sdbe, sdbn;
  const int64_t* off;
  int E;
  int db_from_p;                          // 1: dY is P (row sums of the tile), 0: dY is Q
  // X given as the token matrix it would be gathered from (row r of X = token row idx[r] / fan_out): the operand
  // that holds X (Q when db_from_p, else P) reads its rows through idx; NULL: X is already in grouped order
  const int64_t* idx;
  int fan_out;
  int64_t x_rows;                         // rows of the matrix X is gathered from
};

// Sum over the four lanes that hold a row's shares of the contraction.
__device__ __forceinline__ float sum_of_lane_groups(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// One output tile: rows p0, columns q0 of expert e.
template <typename T, class TL, bool GA, bool GB>
__device__ __forceinline__ void xty_tile(const XtYPlan& a, int e, int p0, int q0, char* lds, int64_t* sDst, unsigned* sRows,
                                         float* sBias) {
  typedef std::conditional_t<TL::PAIR, RowsOp<TL::BM, TL::NT, GA>, TransOp<TL::BM, TL::NT, false, GA, (TL::WG > 2 || TL::RS)>> AOp;
  typedef std::conditional_t<TL::PAIR, RowsOp<TL::BN, TL::NT, GB>, TransOp<TL::BN, TL::NT, false, GB, (TL::WG > 2 || TL::RS)>> BOp;
  const int r_lo = e ? (int)a.off[e - 1] : 0;
  const int r_hi = (int)a.off[e];

  auto output_rows = [&] {
    for (int m = threadIdx.x; m < TL::BM; m += TL::NT)
      sDst[m] = (p0 + m < a.np) ? (int64_t)e * a.soe + (int64_t)(p0 + m) * a.sop : -1;
    __syncthreads();
  };
  if constexpr (!TL::PAIR) output_rows();

  AOp A;
  if constexpr (TL::PAIR && GA)
    A.init_gather((const char*)a.P + (int64_t)p0 * 2, a.ldp * 2, a.np - p0, r_hi - r_lo, a.idx + r_lo, a.fan_out,
                  (unsigned)(((max(a.x_rows, (int64_t)1) - 1) * a.ldp + a.np - p0) * 2));
  else if constexpr (TL::PAIR) A.init((const char*)a.P + ((int64_t)r_lo * a.ldp + p0) * 2, a.ldp * 2, a.np - p0, r_hi - r_lo);
  else if constexpr (GA) A.init_gather((const char*)a.P + (int64_t)p0 * 2, a.ldp * 2, a.np - p0, a.idx + r_lo, a.fan_out, r_hi - r_lo, sRows);
  else A.init((const char*)a.P + ((int64_t)r_lo * a.ldp + p0) * 2, a.ldp * 2, a.np - p0);
  BOp B;           // (rotated load order measured 1.5 % slower here, so both operands keep rot = 0)
  if constexpr (TL::PAIR && GB)
    B.init_gather((const char*)a.Q + (int64_t)q0 * 2, a.ldq * 2, a.nq - q0, r_hi - r_lo, a.idx + r_lo, a.fan_out,
                  (unsigned)(((max(a.x_rows, (int64_t)1) - 1) * a.ldq + a.nq - q0) * 2));
  else if constexpr (TL::PAIR) B.init((const char*)a.Q + ((int64_t)r_lo * a.ldq + q0) * 2, a.ldq * 2, a.nq - q0, r_hi - r_lo);
  else if constexpr (GB) B.init_gather((const char*)a.Q + (int64_t)q0 * 2, a.ldq * 2, a.nq - q0, a.idx + r_lo, a.fan_out, r_hi - r_lo, sRows);
  else B.init((const char*)a.Q + ((int64_t)r_lo * a.ldq + q0) * 2, a.ldq * 2, a.nq - q0);

  Block acc[TL::FM][TL::FN];
  float rs[2 * TL::FM];
#pragma unroll
  for (int i = 0; i < TL::FM; ++i) {
    rs[2 * i] = rs[2 * i + 1] = 0.0f;
#pragma unroll
    for (int j = 0; j < TL::FN; ++j) acc[i][j].clear();
  }
  const bool want_db = a.Db != nullptr && a.db_from_p && q0 == 0;
  if constexpr (TL::RS) mainloop_rs<T, TL, AOp, BOp>(A, B, r_hi - r_lo, lds, acc);      // no bias gradient, no gather
  else if constexpr (TL::PAIR) mainloop_pair<T, TL, AOp, BOp, true>(A, B, r_hi - r_lo, lds, want_db, acc, rs);
  else mainloop<T, TL, AOp, BOp, true>(A, B, r_hi - r_lo, lds, want_db, acc, rs);
  if constexpr (TL::PAIR) output_rows();                 // (into the column stage, which nobody reads any more)

  if constexpr (TL::RS) stage_accumulators<T, TL>(acc, lds, [](int) { return 0.0f; }, sBias);
  if (TL::RS || TL::PAIR || ((((uintptr_t)a.OUT & 15) == 0) && ((a.soe | a.sop | a.nq) & 7) == 0))
    epilogue_staged<T, TL>(acc, (T*)a.OUT, sDst, q0, a.nq, nullptr, 0, lds);
  else
    epilogue<T, TL>(acc, (T*)a.OUT, sDst, q0, a.nq, nullptr, 0);

  if (want_db) {
    // lanes l, l+16, l+32 and l+48 hold a quarter of the contraction of row l%16 each; the first wave column writes the sums
    const int wave = threadIdx.x >> 6, l = lane_id();
    const int wm = wave / TL::WN, wn = wave % TL::WN;
#pragma unroll
    for (int i = 0; i < 2 * TL::FM; ++i) {
      const float tot = sum_of_lane_groups(rs[i]);
      const int p = p0 + wm * TL::WTM + i * 16 + l;
      if (wn == 0 && l < 16 && p < a.np) ((T*)a.Db)[(int64_t)e * a.sdbe + (int64_t)p * a.sdbn] = from_f32<T>(tot);
    }
  }
}

// LDS of a workgroup: operand stages, later the output tile on its way out; row tables.
template <class TL>
struct XtYLds {
  static constexpr int STAGES = TL::NS * (TL::BM + TL::BN) * 128, STAGED = TL::BM * TL::BN * 2;
  __attribute__((aligned(16))) char lds[STAGES > STAGED ? STAGES : STAGED];
  int64_t dst[TL::BM];
  unsigned rows[2 * 64];                    // row offsets of a gathered operand (see TransOp)
  __attribute__((aligned(16))) float bias[TL::RS ? TL::BN : 4];
};

// Order of a launch's tiles: super tiles (Raster) while the experts' loads are alike.  A tile costs its expert's rows, and the
// workgroup of index i runs on XCD i % 8 whatever else that one has to do: where an expert has more than twice the average
// rows, every XCD takes an eighth of every expert's tiles, one contiguous piece in bands of `band` columns, the experts with
// the most rows first.  In super tiles one XCD has all its CUs in the heaviest expert while others have none of its tiles
// (us, super tiles -> this, loads of a router with logits shifted by -1.8 log(rank), experts in any order: 32 experts, 32768 rows,
// 2880 x 2880 in 256 x 256 tiles 786 -> 626, 256 x 128 723 -> 579, 128 x 128 732 -> 640; 2880 x 5760 gathered 1692 -> 1315, 1582 ->
// 1210, 1355 -> 1246; 128 experts, 131072 rows, 2048 x 1536 gathered 1562 -> 1034, 1581 -> 1012.  The experts as they come instead
// of the largest first: 0.8 to 1.04 times as fast).  Even loads keep the super tiles: an expert's rows shared by all XCDs are
// read by each of them (128 x 2048 rows, 2048 x 1536 1600 -> 1640; 64 x 400, 1024 x 2048 138 -> 148).
struct XtYOrder {
  static constexpr int GROUPS = 4;         // groups of 64 experts that are looked through
  Raster rast;
  int p_tiles, q_tiles, band, chunk;       // chunk: tiles of an expert per XCD
  int by_rows;                             // 0: always super tiles
  template <int SN>
  __device__ __forceinline__ bool map(const XtYPlan& a, int pid, int& e, int& m, int& n) const {
    const int lane = lane_id();
    const int x = pid & 7, i = pid >> 3;
    int rows[GROUPS];
    bool uneven = false;
    if (by_rows) {
      // (where most of a super tile's columns do not exist, workgroups with no tile in either order leave first)
      if (2 * q_tiles <= SN && i / chunk >= a.E) {
        int m_tile, m_loc, n_loc;
        if (!rast.map<SN>(pid, m_tile, n, m_loc, n_loc)) return false;
      }
      const int64_t L = a.off[a.E - 1];
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        const int c = g * 64 + lane;
        rows[g] = -1;
        if (g * 64 < a.E && c < a.E) rows[g] = (int)(a.off[c] - (c ? a.off[c - 1] : 0));
        uneven = uneven || __ballot((int64_t)rows[g] * a.E > 2 * L) != 0;
      }
    }
    if (!uneven) {
      int m_tile, m_loc, n_loc;
      if (!rast.map<SN>(pid, m_tile, n, m_loc, n_loc)) return false;
      e = __builtin_amdgcn_readfirstlane(m_tile / p_tiles);
      m = m_tile - e * p_tiles;
      return true;
    }
    int nth = __builtin_amdgcn_readfirstlane(i / chunk);
    const int t = ((x + nth) & 7) * chunk + (i - nth * chunk);
    if (nth >= a.E || t >= p_tiles * q_tiles) return false;
    // the nth expert by the power of two its load reaches (finer steps and groups that hold no expert cost each tile 1.5 us)
    int size[GROUPS], most = 0;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      size[g] = rows[g] < 0 ? -1 : 32 - __clz(rows[g]);
      most = max(most, size[g]);
    }
    e = 0;
    for (int s = __builtin_amdgcn_readfirstlane(wave_max(most)); s >= 0 && nth >= 0; --s) {
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        if (g * 64 >= a.E) break;
        const unsigned long long q = __ballot(size[g] == s);
        const int have = __popcll(q);
        if (nth >= 0 && nth < have)
          e = g * 64 + __ffsll((long long)__ballot(size[g] == s && __popcll(q & ((1ull << lane) - 1)) == nth)) - 1;
        nth -= have;
      }
    }
    e = __builtin_amdgcn_readfirstlane(e);
    const int per_band = p_tiles * band;
    const int b = __builtin_amdgcn_readfirstlane(t / per_band);
    const int width = min(band, q_tiles - b * band), in = t - b * per_band;
    m = __builtin_amdgcn_readfirstlane(in / width);
    n = b * band + in - m * width;
    return true;
  }
};

template <typename T, class TL, bool GA, bool GB>
__global__ __launch_bounds__(TL::NT, TL::WAVES_PER_SIMD) void xty_mfma_kernel(XtYPlan a, XtYOrder order) {
  int e, m, n;
  if constexpr (TL::PAIR) {
    __shared__ __attribute__((aligned(16))) char lds[PAIR_LDS];
    if (!order.map<TL::PAIR ? 2 * Raster::SN : Raster::SN>(a, blockIdx.x, e, m, n)) return;
    xty_tile<T, TL, GA, GB>(a, e, m * TL::BM, n * TL::BN, lds, (int64_t*)(lds + PAIR_B), nullptr, nullptr);
  } else {
    __shared__ XtYLds<TL> s;
    if (!order.map<TL::PAIR ? 2 * Raster::SN : Raster::SN>(a, blockIdx.x, e, m, n)) return;
    xty_tile<T, TL, GA, GB>(a, e, m * TL::BM, n * TL::BN, s.lds, s.dst, s.rows, s.bias);
  }
}

}  // namespace smoe
#include "xty_rows.hpp"
namespace smoe {

// Bias gradient when dY is the column operand: column sums per expert segment.  A workgroup owns 256 columns of one
// expert: 32 column threads (16 bytes = 8 columns each) x 8 row lanes; every thread adds up the rows r = lane
// (mod 8) of the segment, then the 8 partial sums of a column are added in a fixed order (deterministic).
template <typename T>
__global__ __launch_bounds__(256) void colsum_kernel(const T* __restrict__ DY, int64_t ld, int N,
                                                    const int64_t* __restrict__ off, T* __restrict__ Db,
                                                    int64_t sdbe, int64_t sdbn) {
  typedef T T8 __attribute__((ext_vector_type(8)));
  __shared__ float part[8][256];
  const int e = blockIdx.y;
  const int c8 = threadIdx.x & 31, rg = threadIdx.x >> 5;
  const int n = (blockIdx.x * 32 + c8) * 8;
  const int r_lo = e ? (int)off[e - 1] : 0, r_hi = (int)off[e];
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (n < N) {
    int r = r_lo + rg;
    for (; r + 56 < r_hi; r += 64) {                   // eight loads in flight: a load at a time is all latency
      T8 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = *(const T8*)(DY + (int64_t)(r + 8 * u) * ld + n);
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int q = 0; q < 8; ++q) s[q] += to_f32(v[u][q]);
    }
    for (; r < r_hi; r += 8) {
      const T8 v = *(const T8*)(DY + (int64_t)r * ld + n);
#pragma unroll
      for (int q = 0; q < 8; ++q) s[q] += to_f32(v[q]);
    }
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) part[rg][c8 * 8 + q] = s[q];
  __syncthreads();
  const int col = blockIdx.x * 256 + threadIdx.x;
  if (col < N) {
    float t = 0.0f;
#pragma unroll
    for (int g = 0; g < 8; ++g) t += part[g][threadIdx.x];
    Db[(int64_t)e * sdbe + (int64_t)col * sdbn] = from_f32<T>(t);
  }
}

static XtYPlan xty_plan(const XtYArgs& a) {
  XtYPlan p;
  const bool k_contig = a.sdwk == 1;     // output rows = N index
  if (k_contig) {
    p.P = a.DY; p.ldp = a.sdym; p.np = a.N;
    p.Q = a.X; p.ldq = a.sxm; p.nq = a.K;
    p.sop = a.sdwn;
  } else {
    p.P = a.X; p.ldp = a.sxm; p.np = a.K;
    p.Q = a.DY; p.ldq = a.sdym; p.nq = a.N;
    p.sop = a.sdwk;
  }
  p.OUT = a.DW; p.soe = a.sdwe;
  p.Db = a.Db; p.sdbe = a.sdbe; p.sdbn = a.sdbn;
  p.off = a.off; p.E = a.E;
  p.db_from_p = k_contig ? 1 : 0;
  p.idx = a.idx; p.fan_out = a.fan_out;
  p.x_rows = a.L / (a.idx ? a.fan_out : 1);
  return p;
}

static constexpr int XTY_STORE_ROWS = 96;        // rows per expert below which a weight gradient is bound by its stores
static constexpr int XTY_SMALL_ROWS = 256;       // ... and up to which it goes in small tiles (xty_few_rows)

// `grid`: workgroups.  Each order has its own number; a launch that may take either has to cover both.
template <class TL>
static XtYOrder xty_order(const XtYPlan& p, int64_t L, int64_t& grid) {
  XtYOrder r;
  r.p_tiles = (p.np + TL::BM - 1) / TL::BM;
  r.q_tiles = (p.nq + TL::BN - 1) / TL::BN;
  r.band = TL::PAIR ? 2 * Raster::SN : Raster::SN;
  r.rast = make_raster((int64_t)p.E * r.p_tiles, r.q_tiles, GM_XTY, r.band);
  // Few rows are little of what a tile costs, and to ask whether loads are even is the more of it: up to 256 rows per expert, even loads
  // 0.94 to 0.99 of the time without the order (78 of 176 random launches more than 3 % slower), as 1 / rank^0.84 and ^1.8 0.97 to 1.07
  // (128 x 24 rows, 2048 x 1536 145 -> 158 us).  So is one column of 256 wide tiles, each alone on its CU: 0.96 (41 of 72), uneven 1.02.
  r.by_rows = p.E <= 64 * XtYOrder::GROUPS && L / p.E > XTY_SMALL_ROWS && !(TL::BN == 256 && r.q_tiles == 1);
  const int64_t chunk = ((int64_t)r.p_tiles * r.q_tiles + 7) / 8;
  r.chunk = (int)chunk;
  grid = r.by_rows ? std::max(r.rast.grid(), chunk * p.E * 8) : r.rast.grid();
  return r;
}

template <typename T, class TL>
static int launch_xty(const XtYArgs& a, hipStream_t st) {
  const bool k_contig = a.sdwk == 1;
  const XtYPlan p = xty_plan(a);
  int64_t grid;
  const XtYOrder r = xty_order<TL>(p, a.L, grid);
  if (grid > 0x7fffffffLL) { set_error("smoe_groupXtY: grid too large"); return SMOE_ERR_RANGE; }
  if constexpr (TL::RS) hipLaunchKernelGGL((xty_mfma_kernel<T, TL, false, false>), dim3((unsigned)grid), dim3(TL::NT), 0, st, p, r);
  else if (a.idx == nullptr) hipLaunchKernelGGL((xty_mfma_kernel<T, TL, false, false>), dim3((unsigned)grid), dim3(TL::NT), 0, st, p, r);
  else if (k_contig) hipLaunchKernelGGL((xty_mfma_kernel<T, TL, false, true>), dim3((unsigned)grid), dim3(TL::NT), 0, st, p, r);
  else hipLaunchKernelGGL((xty_mfma_kernel<T, TL, true, false>), dim3((unsigned)grid), dim3(TL::NT), 0, st, p, r);
  return launch_status("xty_mfma_kernel");
}

// Which tiles a weight gradient is cut into.  A 256 x 256 tile has a CU to itself and the memory idles while it is
// looked up, waits for its first slice and is stored; with few rows per expert that is most of its time.  Small tiles
// (128 x 128, one 32 KB stage, four workgroups per CU; the stores of one run under the loads and products of the
// others) pay for it with twice the operand traffic through LDS, so they win below a number of rows (both sides
// measured alone, us: 32 experts 2880 x 5760, 100 / 188 / 300 / 400 rows each: 314 -> 225, 407 -> 335, 493 -> 455,
// 594 -> 579; 128 experts 2048 x 1536: 223 -> 168, 286 -> 242, 371 -> 364, 462 -> 477; 8 experts 14336 x 4096:
// 257 -> 191, 316 -> 270, 390 -> 370, 480 -> 489.  Inside a training step, at its lower clock: 32 x 188 rows, 2880 x 2880
// 248 -> 212; even at 280).  Gathered rows as well: 34 random launches of 128 to 256 rows per expert 256 x 256 -> small
// 1.23 times as fast.
// But with few rows per expert the launch is all stores.  Output rows that are no whole number of 64-byte pieces (the unit
// memory is written in) share one at every tile edge; twice the edges cost more than small tiles save, in launches of more than
// 512 large tiles: 50 random ones of 2 to 96 rows per expert 256 x 256 -> small 0.92 times as fast (161 of whole pieces 1.28;
// us: 16 experts x 22 rows, (11024, 2416) 278 -> 311, 128 x 34, (1064, 4144) 384 -> 475).
static constexpr int XTY_STORE_TILES = 512;
static bool xty_few_rows(const XtYArgs& a) {
  const int64_t rows = a.L / a.E, tiles = (int64_t)a.E * ((a.N + 255) / 256) * ((a.K + 255) / 256);
  if (rows > XTY_SMALL_ROWS) return false;
  const int64_t pitch = a.sdwk == 1 ? a.sdwn : a.sdwk;                    // elements between output rows
  const bool pieces = ((uintptr_t)a.DW & 63) == 0 && ((pitch | a.sdwe) & 31) == 0;
  return pieces || rows >= XTY_STORE_ROWS || tiles <= XTY_STORE_TILES;
}
// The same small tiles, whatever the number of rows, where the 256 x 256 ones leave the chip idle: at most 5/8 of a
// round of one per CU, or a second round up to 9/16 full (1600 rows per expert, plain / gathered, us: 128 tiles
// 56 -> 38 / 45 -> 37, 160 tiles 59 -> 50 / 51 -> 48, 320 tiles 102 -> 77 / 96 -> 84, 384 tiles 105 -> 90 / 100 -> 90;
// but 192 tiles 56 -> 57 / 48 -> 58, 256 tiles 64 -> 60 / 55 -> 61, 512 tiles 110 -> 112 / 105 -> 116).
// They request every operand byte twice as often, so they lose once the operands are no longer served from the 256 MB
// memory-side cache, or the rows are so many that the large tiles' shorter loop outweighs the idle CUs (us, 256 x 256
// with one wave per SIMD -> small, whole products of E x (N, K) by rows per expert):
//   second round: 8 x (1536, 1536) 4096 rows 200 -> 183, 6000 rows (295 MB) 283 -> 286, 8192 rows 372 -> 397;
//     4 x (2048, 2304) 8192 rows (143 MB) 366 -> 365; 8 x (1536, 2048) 4096 rows 216 -> 205, 8192 rows 410 -> 479;
//     2 x (3072, 4096) 5000 rows 262 -> 244, 8192 rows (235 MB) 406 -> 425; 4 x (2560, 2560), 400 tiles, 1024 rows
//     67 -> 60, 2048 rows 109 -> 111, 3072 rows 150 -> 166, 4096 rows 205 -> 220, 8192 rows 390 -> 579
//   129 to 160 tiles: 8 x (1024, 1280) 6000 rows 153 -> 142, 8192 rows (302 MB) 205 -> 216; 17 x (512, 1024) 5000 rows
//     130 -> 114, 6000 rows (313 MB) 155 -> 160; 16 x (768, 768) 8192 rows (402 MB) 177 -> 216
//   up to 128 tiles: 8 x (1024, 1024) 16384 rows (537 MB) 402 -> 349, 12 x (512, 1024) 16384 rows 399 -> 348, but experts
//     of few tiles stream too much per product: 32 x (512, 512) 4096 rows 93 -> 73, 8192 rows (537 MB) 171 -> 183
//     (gathered, against eight waves: 219 -> 199)
// and for experts of one or two tiles beside many others: 128 x (256, 256) 512 / 1600 rows 19 -> 20, 42 -> 49; 53 x (256, 768)
// 1024 / 2048 rows 33 -> 36, 54 -> 66; 64 x (256, 512) 2048 rows 49 -> 40.
static bool xty_idle_chip(const XtYArgs& a, bool rs_form) {
  const int64_t per_expert = (int64_t)((a.N + 255) / 256) * ((a.K + 255) / 256), tiles = a.E * per_expert;
  const int64_t rows = a.L / a.E;
  const bool cached = (int64_t)a.L * (a.N + a.K) * 2 <= (256ll << 20);
  if (tiles <= 128) return cached ? per_expert > 1 || tiles <= 64 : per_expert >= 6 || !rs_form;
  if (per_expert < 4) return false;
  if (tiles <= 160) return cached;
  if (tiles <= 256 || tiles > 400) return false;
  return rows <= (tiles > 384 ? 1536 : !cached ? 3072 : tiles > 320 ? 5120 : 8192);
}

// One operand in registers, the other streamed past it (xty_rows.hpp), us against 128 x 128 tiles over 390 random launches with
// output rows on whole lines.  From 96 rows per expert on: even loads of 110 to 220 rows 1.07 to 1.31 times as fast; below 64
// 0.96 (both are bound by their stores there), 64 to 96 1.00 to 1.07.  Up to 224: experts beyond 256 rows go in tiles, two
// workgroups per CU where a launch of nothing but tiles has four (even loads of 250 rows, half of them beyond: 0.95, 1190
// rows 0.85).  At least 256 tiles of 256 x 256: smaller launches have too few units (16 x 142 rows, 1472 x 512 11 -> 13).
// 5650 random launches within those lines, even loads / as 1 / rank^0.42, ^0.84, ^1.8 (more than 3 % slower): the held operand is a
// panel of 256 output rows, of which narrow outputs leave most empty, two thirds and more of them multiplied for nothing; and
// what unevenness puts beyond 256 rows is then a chain of slices for a few workgroups.  Up to 128 rows 0.80 / 0.66 / 0.76 / 1.1 (100 of 102, 104
// of 121 ...), to 256 0.99 / 0.80 / 0.85 / 1.1, to 384 1.15 / 0.95 / 1.01 / 1.14, beyond 1.21 to 1.38 / 1.0 to 1.16 / 1.0 to 1.06 / 1.2 to 1.3.
// With few experts one of them has most of the rows: 8 experts 1.24 / 1.05 / 0.94 (53 of 85) / 0.96, 4 1.23 / 1.10 / 1.02 / 0.92, 16
// 1.24 / 1.04 / 0.97 / 1.08, 32 1.25 / 1.04 / 1.03 / 1.18, more 1.23 to 1.3 / 1.1 / 1.1 / 1.2.
static constexpr int XTY_HELD_MIN_ROWS = 96, XTY_HELD_MAX_ROWS = 224, XTY_HELD_MIN_PANEL = 384, XTY_HELD_MIN_EXPERTS = 16;
static bool xty_held(const XtYArgs& a) {
  const XtYPlan p = xty_plan(a);
  const int64_t rows = a.L / a.E;
  if (rows < XTY_HELD_MIN_ROWS || rows > XTY_HELD_MAX_ROWS || a.E < XTY_HELD_MIN_EXPERTS || p.np < XTY_HELD_MIN_PANEL) return false;
  return (int64_t)a.E * ((a.N + 255) / 256) * ((a.K + 255) / 256) >= 256 && xty_rows_fits(p);
}

// Between them: 256 x 128 tiles, two workgroups per CU (mainloop_pair), or the small tiles again, against eight waves per
// 256 x 256 tile over 2000 random launches of 257 to 2047 rows per expert (4 to 128 experts, K and N from 256 to 8000, gathered
// and not; even / Zipf-like loads, each in the order of XtYOrder).  256 x 128, 257 to 700 rows 1.10 / 1.17 times as fast, to 1200
// 1.06 / 1.14, to 2047 1.03 / 1.11.  Not, gathered, beyond eight rounds from 1200 rows on (0.97 / 1.02: the lookups come twice as
// often), nor where the gathered operand is a single tile row (0.98 / 1.14, 10 of 29 even ones more than 3 % slower; us, 64 experts x 857
// rows, 176 x 2520 98 -> 113); nor, a single tile row, with more experts than XtYOrder looks through (uneven loads of 300 0.81 to 0.96).
// Not where an expert's output is one tile wide: two of 128 columns read the rows twice for it (30 random launches of 129 to 256
// columns, even loads 0.96, 23 more than 3 % slower; 200 x 389 rows, 2752 x 256 177 -> 205, x 765, 3072 x 192 298 -> 339).  Not from
// 2048 rows on (even loads 0.96, 17 of 27 more than 3 % slower; 200 x 3491 rows, 256 x 256 121 -> 137).  Small tiles against 256 x 128
// while the operands come from the memory-side cache, beyond one round: 257 to 700 rows, up to eight rounds 1.07 / 1.02, to 1200
// rows, up to four 1.07 / 1.02, to 2047 rows, up to two 1.07 / 1.02.
// us, 32 experts x 500 rows, 2880 x 2880 346 -> 309; 32 x 300, 2880 x 5760 gathered 504 -> 467; 16 x 1000, 1024 x 1024 35.8 -> 34.4.
// Same bits in every class.
static constexpr int XTY_PAIR_ROUND = 2 * NUM_CU;
static int64_t xty_pair_tiles(const XtYPlan& p) { return (int64_t)p.E * ((p.np + 255) / 256) * ((p.nq + 127) / 128); }
static bool xty_small_again(const XtYArgs& a) {
  const int64_t rows = a.L / a.E, tiles = xty_pair_tiles(xty_plan(a));
  if (rows <= XTY_SMALL_ROWS || rows >= RS_XTY_MIN_ROWS || (int64_t)a.L * (a.N + a.K) * 2 > (256ll << 20)) return false;
  return tiles > XTY_PAIR_ROUND && tiles <= XTY_PAIR_ROUND * (rows < 700 ? 8 : rows < 1200 ? 4 : 2);
}
static bool xty_pairs(const XtYArgs& a) {
  const XtYPlan p = xty_plan(a);
  const int64_t rows = a.L / a.E;
  const bool gathered = a.idx != nullptr;
  if (rows <= XTY_SMALL_ROWS || rows >= RS_XTY_MIN_ROWS || (p.nq > 128 && p.nq <= 256)) return false;
  if (p.np <= 256 && ((gathered && !p.db_from_p) || p.E > 64 * XtYOrder::GROUPS)) return false;
  if (gathered && rows >= 1200 && xty_pair_tiles(p) > 8 * XTY_PAIR_ROUND) return false;
  // Output pieces of 16 bytes; rows that do not overlap (the descriptors end with the last one) and, gathered, a source below
  // 2 GiB.
  if (((uintptr_t)p.OUT & 15) != 0 || ((p.soe | p.sop | p.nq) & 7) != 0 || p.ldp < p.np || p.ldq < p.nq) return false;
  return !gathered || (p.x_rows + 1) * a.sxm + a.K < (1ll << 30);
}

// One-wave-per-SIMD form: needs the LDS-staged epilogue; no gathered operand, no bias gradient in the main loop.
// Both operands are read transposed (two LDS reads per fragment), which leaves less to win than in
// scatter2scatter: Mixtral shape (4096 rows per expert) 3.28 -> 3.12 and 6.35 -> 6.20 ms, 2048 rows per expert
// (128 experts, 768 x 2048 and 2048 x 1536 outputs) 0.81 -> 0.77 and 1.55 -> 1.51 ms.  Against 256 x 128 tiles, two workgroups per
// CU, 90 random launches of 1280 to 2047 rows per expert under even and uneven loads: of four rounds and more 1.03 times as fast
// (0.97 to 1.15; 32 x 2046 rows, 2880 x 3864 1549 -> 1432 us, 16 x 1983, 3128 x 4744 1054 -> 980), of fewer 1.00 (0.82 to 1.18); of 600 to
// 1024 rows 0.95 (0.85 to 1.04).
static bool xty_one_wave(const XtYArgs& a) {
  const bool out16 = (((uintptr_t)a.DW & 15) == 0) && ((a.sdwe | (a.sdwk == 1 ? a.sdwn : a.sdwk) | (a.sdwk == 1 ? a.K : a.N)) & 7) == 0;
  const bool db_in_loop = a.Db != nullptr && a.sdwk == 1;
  // (its buffer descriptors end with an operand's last row: rows that overlap, as those of an expanded tensor, would read as zeros)
  const bool apart = a.sdym >= a.N && a.sxm >= a.K;
  const int64_t rows = a.L / a.E, tiles = (int64_t)a.E * ((a.N + 255) / 256) * ((a.K + 255) / 256);
  return a.idx == nullptr && !db_in_loop && out16 && apart &&
         (rows >= RS_XTY_MIN_ROWS || (rows >= RS_XTY_MIN_ROWS_ROUNDS && tiles >= RS_XTY_ROUNDS * NUM_CU));
}

enum class XtYClass { held, small, pairs, one_wave, large };
static XtYClass xty_class(const XtYArgs& a) {
  const bool rs_form = xty_one_wave(a);
  if (xty_held(a)) return XtYClass::held;
  if (xty_idle_chip(a, rs_form) || xty_few_rows(a) || xty_small_again(a)) return XtYClass::small;
  if (rs_form) return XtYClass::one_wave;
  return xty_pairs(a) ? XtYClass::pairs : XtYClass::large;
}

template <typename T>
static int dispatch_xty(const XtYArgs& a, hipStream_t st) {
  int rc = 0;
  switch (xty_class(a)) {
    case XtYClass::held: rc = launch_xty_rows<T>(xty_plan(a), a.L, st); break;
    case XtYClass::small: rc = launch_xty<T, Tile<128, 128, 2, 2, 1, false, 4>>(a, st); break;
    case XtYClass::pairs: rc = launch_xty<T, PairTile>(a, st); break;
    case XtYClass::one_wave: rc = launch_xty<T, Tile<256, 256, 2, 2, 2, true>>(a, st); break;
    case XtYClass::large: rc = launch_xty<T, Tile<256, 256, 2, 4>>(a, st); break;
  }
  if (rc == 0 && a.Db != nullptr && a.sdwk != 1) {
    hipLaunchKernelGGL(colsum_kernel<T>, dim3((a.N + 255) / 256, a.E), dim3(256), 0, st, (const T*)a.DY,
                       a.sdym, a.N, a.off, (T*)a.Db, a.sdbe, a.sdbn);
    rc = launch_status("colsum_kernel");
  }
  return rc;
}

}  // namespace smoe
