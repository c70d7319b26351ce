// groupXtY of experts with few rows: one operand held in registers, the other streamed past it.
// (Included by gemm_mfma.hpp; counterpart in the reference: _groupXtY, scattermoe/kernels/ops.py:242-366.)
#pragma once

namespace smoe {

static constexpr int XTY_ROWS_MAX = 256;       // rows of an expert whose operand is held: four 64-row slices in registers
static constexpr int XR_P = 256, XR_Q = 64;    // output rows of a workgroup's panel, output columns of a step
static constexpr int XR_RING = 64 * 1024, XR_OUT = 16 * 1024;      // LDS of a workgroup, two of them per CU: operand stages, output
static constexpr int XR_UNIT_STEPS = 3;        // what a unit costs before its first step, in steps (2 to 8: the same times)

// What bounds a weight gradient of few rows is not its products but the loads in front of them: a 128 x 128 tile of 188 rows is
// three slices of 64, each requested when the one before has been multiplied, and every operand byte goes through LDS once per
// tile (setup 2.1, three slices 6.9, store 3.0 us, four tiles per CU at a time).  Here a workgroup keeps 256 output rows' operand
// in registers, all of its contraction (up to 256 rows: 128 registers), and streams the other operand past it in steps of 64
// output columns, the next steps' loads in flight while one is multiplied and stored: each streamed byte is requested once per 256
// output rows, the held ones once per unit, and no load waits for a product.  Gathered rows cost nothing: their offsets are the
// same in every step.  Measured alone, us, 128 x 128 tiles -> this (written at, TB/s): 32 experts x 188 rows, 2880 x 2880
// 205 -> 154 (3.5), 2880 x 5760 338 -> 245 (4.3); 128 x 188, 768 x 2048 126 -> 94 (4.3); 8 x 188, 14336 x 4096 289 -> 215
// (4.4); 128 x 100, 2048 x 1536 186 -> 161 (5.0).  A kernel that only stores in this pattern reaches 5.2: with 100 rows and
// fewer the stores bound it, with 200 they and the matrix cores (0.8 PFLOP/s).

// Tiles for the experts of more rows, whose workgroups come first in the same launch (a launch of their own takes 16 to 31 us
// to find nothing to do).  One stage 4 to 40 % slower, 256 x 128 tiles 18 to 110 %.
typedef Tile<128, 128, 2, 2, 2, false, 2> XRAbove;
static_assert(sizeof(XtYLds<XRAbove>) <= XR_RING + XR_OUT, "LDS");

// Where the units of a launch lie: unit = (expert, chunk of column steps, row panel), panels fastest, so that the
// workgroups that run side by side on an XCD stream through the same columns; every XCD takes one contiguous piece.
struct XtYUnits {
  int panels, chunks, chunk_steps, steps, units, per_xcd;
  int workers;             // workgroups ahead of them, for the experts of more rows (xty_rows_above)
};

// One unit of an expert of at most 64 NSL rows.
template <typename T, int NSL, bool GP, bool GQ>
__device__ __forceinline__ void xty_rows_unit(const XtYPlan& a, int e, int r_lo, int rows, int p0, int step0, int nsteps,
                                              bool want_db, char* lds) {
  typedef TransOp<XR_P, 256> POp;                        // LDS layout of a 64-row slice of the held operand
  constexpr int NST = NSL >= 3 ? 2 : 4;                     // stages of the streamed operand
  constexpr int STAGE = NSL * 8192;
  constexpr int LOADS = 2 * NSL, STORES = 8;             // memory instructions of a thread per step
  static_assert(NST * STAGE <= XR_RING && 2 * POp::LDS_BYTES <= XR_RING, "LDS");
  const int t = threadIdx.x, l = lane_id();
  const int wave = wave_uniform_id();
  const unsigned lds_u = lds_address(lds);
  // byte offset of contraction row r of an operand, from its descriptor's base (gathered rows: looked up once)
  unsigned* srow = (unsigned*)(lds + XR_RING);
  if constexpr (GP || GQ) {
    const int64_t ld = GP ? a.ldp : a.ldq;
    srow[t] = t < rows ? (unsigned)((int64_t)((unsigned)a.idx[r_lo + t] / (unsigned)a.fan_out) * ld * 2) : OUT_OF_RANGE;
    __syncthreads();
  }
  auto row_off = [&](auto gathered, int r, int64_t ld) -> unsigned {
    if constexpr (decltype(gathered)::value) return srow[r];
    else return r < rows ? (unsigned)(r * ld * 2) : OUT_OF_RANGE;
  };
  auto rsrc_of = [&](auto gathered, const void* base, int64_t ld, int cols) {
    const bool g = decltype(gathered)::value;
    // (an expert without rows reads none, its lanes being out of any range; one row's range all the same, as the bounds
    // check may take a step's scalar offset off the range and must not wrap around)
    const int64_t n = max((int64_t)1, g ? a.x_rows : (int64_t)rows);
    return buffer_rsrc((const char*)base + (g ? 0 : (int64_t)r_lo * ld * 2), (unsigned)(((n - 1) * ld + cols) * 2));
  };

  // ---- the held operand: two slices at a time through LDS, then as fragments in registers
  i32x4 fa[NSL * 2][4];
  {
    const i32x4 rp = rsrc_of(std::integral_constant<bool, GP>(), a.P, a.ldp, a.np);
    const int kr = t >> 5, phys = t & 31;                // piece j of this thread: row j * 8 + kr of the slice
    const unsigned col[2] = {(unsigned)p0 * 2 + (trans_piece(kr, phys) << 4), (unsigned)p0 * 2 + (trans_piece(8 + kr, phys) << 4)};
#pragma unroll
    for (int s0 = 0; s0 < NSL; s0 += 2) {
      if (s0 > 0) __syncthreads();                       // the first two slices have been read
#pragma unroll
      for (int s = s0; s < s0 + 2 && s < NSL; ++s)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          buffer_to_lds16(rp, row_off(std::integral_constant<bool, GP>(), s * 64 + j * 8 + kr, a.ldp) + col[j & 1], 0,
                          lds_u + (s - s0) * POp::LDS_BYTES + j * 4096 + wave * 1024);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
#pragma unroll
      for (int s = s0; s < s0 + 2 && s < NSL; ++s)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
          for (int i = 0; i < 4; ++i) fa[s * 2 + ks][i] = POp::frag(lds + (s - s0) * POp::LDS_BYTES, wave * 64 + i * 16, ks);
    }
  }
  if (want_db) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float rs = 0.0f;
#pragma unroll
      for (int q = 0; q < NSL * 2; ++q) rs += Mfma<T>::sum8(fa[q][i]);
      const float tot = sum_of_lane_groups(rs);
      const int p = p0 + wave * 64 + i * 16 + l;
      if (l < 16 && p < a.np) ((T*)a.Db)[(int64_t)e * a.sdbe + (int64_t)p * a.sdbn] = from_f32<T>(tot);
    }
  }

  // ---- the streamed operand: rows of 128 bytes per step, the two 64-byte granules of a row exchanged in every second pair
  // of rows, the halves of a granule in every second eight rows (a transposing read touches half a granule of four consecutive
  // rows and of the four rows 8 further down)
  const i32x4 rq = rsrc_of(std::integral_constant<bool, GQ>(), a.Q, a.ldq, a.nq);
  unsigned qoff[LOADS];
  {
    const int kr = t >> 3, phys = t & 7;
    const unsigned col = (phys ^ ((kr << 1) & 4) ^ ((kr >> 2) & 2)) << 4;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) qoff[j] = row_off(std::integral_constant<bool, GQ>(), j * 32 + kr, a.ldq) + col;
  }
  auto issue = [&](int step, int stage) {
    const unsigned dst = lds_u + stage * STAGE + wave * 1024;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) buffer_to_lds16(rq, qoff[j], (unsigned)(step0 + step) * (XR_Q * 2), dst + j * 4096);
  };
  // fragment (columns 16 j .. 16 j + 15, contraction step q) of a stage
  const int b = l >> 4, r4 = (l & 15) >> 2;
  const char* fbase = lds + (8 * b + r4) * 128 + (l & 3) * 8;
  const int unit = ((r4 & 2) << 5) ^ ((b & 1) << 5);
  auto frag = [&](int stage, int j, int q) {
    const char* p = fbase + stage * STAGE + q * 4096 + ((j << 5) ^ unit);
    const s16x4 lo = lds_read_tr(p), hi = lds_read_tr(p + 512);
    return __builtin_bit_cast(i32x4, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // ---- output: a wave's 32 x 64 block of a step goes through 4 KB of LDS of its own (no barrier) so that it is stored in whole
  // 128-byte lines: 16-byte piece c of row r sits at piece c ^ (r / 2 % 8)
  char* out_lds = lds + XR_RING + wave * 4096;
  const int valid = a.np - p0 < XR_P ? a.np - p0 : XR_P;
  const __amdgpu_buffer_rsrc_t ro = tile_rows_rsrc((T*)a.OUT + (int64_t)e * a.soe + (int64_t)p0 * a.sop, 1,
                                                   ((int64_t)(valid - 1) * a.sop + a.nq) * 2);
  const int64_t pitch = a.sop * 2;
  const unsigned ooff = (unsigned)((wave * 64 + (l >> 3)) * pitch) + ((l & 7) << 4);
  char* wr = out_lds + (l & 15) * 128;
  const int wsw = (l >> 1) & 7, wch = 2 * (b & 1) + (b >> 1);
  const int rdrow = (l >> 3) * 128, rdch = (l & 7) ^ (l >> 4);                        // row 8 q + l / 8
  const char* rd[2] = {out_lds + rdrow + (rdch << 4), out_lds + rdrow + ((rdch ^ 4) << 4)};      // of even and odd q

  __syncthreads();                                       // everyone has the held operand in registers
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < nsteps) issue(s, s);
  int stage = 0;
  for (int step = 0; step < nsteps; ++step) {
    // The step's columns have landed once no more operations are outstanding than were issued behind their loads: loads
    // of the steps since, and the stores of as many (fewer at either end, where the count is taken lower).
    if (step + NST - 1 > nsteps) {
      if (step < NST - 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 1) * STORES) : "memory");
    } else if (step < NST - 1) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * LOADS) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * LOADS + (NST - 1) * STORES) : "memory");
    }
    __syncthreads();                                     // everyone's have, and everyone is done with the step before
    if (step + NST - 1 < nsteps) issue(step + NST - 1, stage == 0 ? NST - 1 : stage - 1);
    Block acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j].clear();
    i32x4 fb[2][2];                                      // two of the four fragments of a step of 32, the next two meanwhile
    fb[0][0] = frag(stage, 0, 0);
    fb[0][1] = frag(stage, 1, 0);
#pragma unroll
    for (int h = 0; h < NSL * 4; ++h) {
      const int c = h & 1, n = c ^ 1;
      if (h + 1 < NSL * 4) {
        fb[n][0] = frag(stage, 2 * n, (h + 1) >> 1);
        fb[n][1] = frag(stage, 2 * n + 1, (h + 1) >> 1);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4& d = acc[i >> 1][c].q[2 * (i & 1) + j];
          d = Mfma<T>::run(fb[c][j], fa[h >> 1][i], d);
        }
    }
    // A lane holds, per group of four accumulators, four consecutive columns of its output row, the lane 16 further the
    // four next to them.  Exchanging every second 16 lanes between two neighbouring groups leaves each lane with eight columns.
    const int n0 = (step0 + step) * XR_Q;
    const bool whole = n0 + XR_Q <= a.nq;
    const unsigned off = whole || n0 + ((l & 7) << 3) < a.nq ? ooff + (unsigned)n0 * 2 : OUT_OF_RANGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      typedef T T4 __attribute__((ext_vector_type(4)));
      typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
      typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          T4 lo, hi;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            set_pair<T>(lo, h, acc[i][j][r * 8 + 2 * h], acc[i][j][r * 8 + 2 * h + 1]);
            set_pair<T>(hi, h, acc[i][j][r * 8 + 4 + 2 * h], acc[i][j][r * 8 + 4 + 2 * h + 1]);
          }
          const u32x2_t u = __builtin_bit_cast(u32x2_t, lo), v = __builtin_bit_cast(u32x2_t, hi);
          const auto s0 = __builtin_amdgcn_permlane16_swap(u[0], v[0], false, false);
          const auto s1 = __builtin_amdgcn_permlane16_swap(u[1], v[1], false, false);
          *(u32x4_t*)(wr + r * 2048 + (((j * 4 + wch) ^ wsw) << 4)) = u32x4_t{s0[0], s1[0], s0[1], s1[1]};
        }
      u32x4_t w[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) w[q] = *(const u32x4_t*)(rd[q & 1] + q * 1024);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        // Whole lines with the non-temporal hint leave the operands in the L2 (32 x 188 rows, 2880 x 5760: 281 -> 244 us).
        // (No scalar offset: with one the compiler lets the next instruction overwrite the data registers, and the store
        // has been seen to write what it found in them then)
        __builtin_amdgcn_raw_buffer_store_b128(w[q], ro, (int)(off + (unsigned)((i * 32 + q * 8) * pitch)), 0, 2 /* non-temporal */);
    }
    stage = stage + 1 == NST ? 0 : stage + 1;
  }
}

// The experts with more rows than the held operand has room for: their output in 128 x 128 tiles, worker `w` of `workers`
// (a multiple of 256) takes every `workers`-th.  Which experts those are is known only here; super tiles in the order of
// Raster, over the experts that qualify.
template <typename T, bool GP, bool GQ>
__device__ __forceinline__ void xty_rows_above(const XtYPlan& a, int w, int workers, char* lds) {
  typedef XtYLds<XRAbove> Lds;
  Lds& s = *(Lds*)lds;
  const int lane = lane_id();
  const int p_tiles = (a.np + XRAbove::BM - 1) / XRAbove::BM, q_tiles = (a.nq + XRAbove::BN - 1) / XRAbove::BN;
  const int m_supers = (p_tiles + Raster::SM - 1) / Raster::SM, supers = m_supers * ((q_tiles + Raster::SN - 1) / Raster::SN);
  for (int pid = w;; pid += workers) {
    const int x = pid & 7, i = pid >> 3, j = i / (Raster::SM * Raster::SN), r = i % (Raster::SM * Raster::SN);
    const int super = j * 8 + ((x + j) & 7);
    int nth = __builtin_amdgcn_readfirstlane(super / supers), e = -1;
    const int in = super - nth * supers;
    for (int e0 = 0; e0 < a.E; e0 += 64) {                    // the expert of that rank among those that qualify
      int rows = 0;
      if (e0 + lane < a.E) rows = (int)a.off[e0 + lane] - (e0 + lane ? (int)a.off[e0 + lane - 1] : 0);
      const bool above = rows > XTY_ROWS_MAX;
      const unsigned long long q = __ballot(above);
      const int n = __popcll(q);
      if (nth < n) {
        e = e0 + __ffsll((long long)__ballot(above && __popcll(q & ((1ull << lane) - 1)) == nth)) - 1;
        break;
      }
      nth -= n;
    }
    if (e < 0) return;
    const int m = (in % m_supers) * Raster::SM + r % Raster::SM, n = (in / m_supers) * Raster::SN + r / Raster::SM;
    if (m >= p_tiles || n >= q_tiles) continue;
    xty_tile<T, XRAbove, GP, GQ>(a, e, m * XRAbove::BM, n * XRAbove::BN, s.lds, s.dst, s.rows, s.bias);
    __syncthreads();
  }
}

template <typename T, bool GP, bool GQ>
__global__ __launch_bounds__(256, 2) void xty_rows_kernel(XtYPlan a, XtYUnits n) {
  __shared__ __attribute__((aligned(16))) char lds[XR_RING + XR_OUT];
  if ((int)blockIdx.x < n.workers) {
    xty_rows_above<T, GP, GQ>(a, blockIdx.x, n.workers, lds);
    return;
  }
  const int pid = blockIdx.x - n.workers;
  const int i = pid >> 3, u = (pid & 7) * n.per_xcd + i;
  if (i >= n.per_xcd || u >= n.units) return;
  const int per_expert = n.panels * n.chunks;
  const int e = __builtin_amdgcn_readfirstlane(u / per_expert);
  const int in = u - e * per_expert;
  const int chunk = __builtin_amdgcn_readfirstlane(in / n.panels);
  const int p0 = (in - chunk * n.panels) * XR_P;
  const int r_lo = e ? (int)a.off[e - 1] : 0;
  const int rows = (int)a.off[e] - r_lo;
  if (rows > XTY_ROWS_MAX) return;
  const int step0 = chunk * n.chunk_steps;
  const int nsteps = min(n.chunk_steps, n.steps - step0);
  const bool want_db = a.Db != nullptr && a.db_from_p && chunk == 0;
  if (rows <= 64) xty_rows_unit<T, 1, GP, GQ>(a, e, r_lo, rows, p0, step0, nsteps, want_db, lds);
  else if (rows <= 128) xty_rows_unit<T, 2, GP, GQ>(a, e, r_lo, rows, p0, step0, nsteps, want_db, lds);
  else if (rows <= 192) xty_rows_unit<T, 3, GP, GQ>(a, e, r_lo, rows, p0, step0, nsteps, want_db, lds);
  else xty_rows_unit<T, 4, GP, GQ>(a, e, r_lo, rows, p0, step0, nsteps, want_db, lds);
}

// Whether the kernel takes the launch's layout: output rows that start on 128-byte lines (others share a line at every step's
// edge and are written at a third of the rate: 128 x 34 rows, 4144 x 1064 670 us against 334 in tiles), and every
// descriptor's range below 2 GiB.
static bool xty_rows_fits(const XtYPlan& p) {
  if (((uintptr_t)p.OUT & 127) != 0 || ((p.soe | p.sop) & 63) != 0 || (p.nq & 7) != 0) return false;
  auto below = [](int64_t rows, int64_t ld, int64_t cols) { return rows * ld + cols < (1ll << 30); };
  return below(XR_P, p.sop, p.nq) && below(p.idx != nullptr && !p.db_from_p ? p.x_rows : XTY_ROWS_MAX, p.ldp, p.np + XR_P) &&
         below(p.idx != nullptr && p.db_from_p ? p.x_rows : XTY_ROWS_MAX, p.ldq, p.nq + XR_Q);
}

template <typename T>
static int launch_xty_rows(const XtYPlan& p, int64_t L, hipStream_t st) {
  XtYUnits n;
  n.panels = (p.np + XR_P - 1) / XR_P;
  n.steps = (p.nq + XR_Q - 1) / XR_Q;
  // Column steps per unit: whole rounds of two units per CU, set against what a unit costs before its first step.
  const int64_t least = (int64_t)p.E * n.panels;
  int64_t best = -1;
  for (int c = 1; c <= n.steps; ++c) {
    const int len = (n.steps + c - 1) / c, chunks = (n.steps + len - 1) / len;
    if (chunks != c) continue;
    const int64_t cost = (least * chunks + 511) / 512 * (XR_UNIT_STEPS + len);
    if (best < 0 || cost < best) best = cost, n.chunks = chunks, n.chunk_steps = len;
  }
  const int64_t units = least * n.chunks;
  if (units > 0x7ffffff0LL) { set_error("smoe_groupXtY: grid too large"); return SMOE_ERR_RANGE; }
  n.units = (int)units;
  n.per_xcd = (int)((units + 7) / 8);
  n.workers = L > XTY_ROWS_MAX ? 512 : 0;
  const dim3 grid((unsigned)(n.per_xcd * 8 + n.workers));
  if (p.idx == nullptr) hipLaunchKernelGGL((xty_rows_kernel<T, false, false>), grid, dim3(256), 0, st, p, n);
  else if (p.db_from_p) hipLaunchKernelGGL((xty_rows_kernel<T, false, true>), grid, dim3(256), 0, st, p, n);
  else hipLaunchKernelGGL((xty_rows_kernel<T, true, false>), grid, dim3(256), 0, st, p, n);
  return launch_status("xty_rows_kernel");
}

}  // namespace smoe
