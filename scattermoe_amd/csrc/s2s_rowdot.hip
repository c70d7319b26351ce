// scatter2scatter for a handful of rows (single-token and few-token decode): every weight element is used by at
// most four rows, so the launch is a stream over the weights of the experts that were hit and nothing else
// matters.  No LDS tiles and no MFMA: each wave reads whole 16-byte pieces of K-contiguous weight rows with
// plain coalesced loads (a wave instruction covers 1 KB of one weight row), multiplies them with the matching
// pieces of up to four input rows by packed dot products, and the partial sums are reduced across lanes once at
// the end.  Many small waves per CU keep far more bytes in flight than the ring-buffered MFMA tiles can.
//
// Work split: a workgroup (4 waves) owns C = 8 output columns of one tile of up to R = 4 expert-sorted rows; its
// waves take the contraction pieces round-robin (piece p of 512 elements goes to wave p % 4), so the four waves
// together read 4 KB runs of each weight row.  A workgroup walks `gpw` consecutive column groups.
//
// Counterparts in the reference: _single2scatter (scattermoe/kernels/single.py:5-59), and _scatter2scatter
// (scattermoe/kernels/ops.py:50-118) for the row/column conventions, bias and the fused GLU of mlp.py:81-87.
#include "common.hpp"
#include <algorithm>

namespace smoe {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Pair;
template <> struct Pair<bf16_t> {
  typedef __bf16 v2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ float dot(unsigned a, unsigned b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
  }
};
template <> struct Pair<f16_t> {
  typedef _Float16 v2 __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ float dot(unsigned a, unsigned b, float c) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
  }
};

// v of the lane whose id differs in bit OFF, OFF = 8 / 4 / 2 / 1 (row rotation, swizzle, quad permutations: one
// instruction each, where a general shuffle first builds a lane address)
template <int OFF>
__device__ __forceinline__ float lane_xor(float v) {
  static_assert(OFF == 8 || OFF == 4 || OFF == 2 || OFF == 1, "inside a row of 16 lanes");
  const int i = __float_as_int(v);
  if constexpr (OFF == 4) return __int_as_float(__builtin_amdgcn_ds_swizzle(i, (4 << 10) | 0x1f));
  else return __int_as_float(__builtin_amdgcn_update_dpp(0, i, OFF == 8 ? 0x128 : OFF == 2 ? 0x4e : 0xb1, 0xf, 0xf, true));
}

// Sum each of the N per-lane values over the 64 lanes of the wave: every one of the first log2(N) steps halves the
// number of values a lane carries (the lane keeps the half selected by one bit of its id and adds the partner's copy
// of it), the remaining steps are exchanges of the one value left.  Afterwards lane l holds the total of value
// l / (64 / N) in v[0].  A value is added up by the same tree of lanes whatever N is.
template <int HALF, int OFF, int N>
__device__ __forceinline__ void transpose_sum_step(float (&v)[N], int lane) {
  if constexpr (OFF >= 16) {
    static_assert(HALF > 0, "at least four values");
    // the permute exchanges the upper half (odd rows of 16) of one register with the lower half (even rows) of the
    // other: afterwards both hold a value and its partner's copy of it, lane by lane
#pragma unroll
    for (int i = 0; i < HALF; ++i) {
      typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
      const unsigned x = __float_as_uint(v[i]), y = __float_as_uint(v[i + HALF]);
      u32x2 r;
      if constexpr (OFF == 32) r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
      else r = __builtin_amdgcn_permlane16_swap(x, y, false, false);
      v[i] = __uint_as_float(r.x) + __uint_as_float(r.y);
    }
  } else if constexpr (HALF > 0) {
    const bool up = (lane & OFF) != 0;
#pragma unroll
    for (int i = 0; i < HALF; ++i) {
      const float keep = up ? v[i + HALF] : v[i];
      const float send = up ? v[i] : v[i + HALF];
      v[i] = keep + lane_xor<OFF>(send);
    }
  } else {
    v[0] += lane_xor<OFF>(v[0]);
  }
  if constexpr (OFF > 1) transpose_sum_step<HALF / 2, OFF / 2>(v, lane);
}
template <int N>
__device__ __forceinline__ void wave_transpose_sum(float (&v)[N]) {
  static_assert(N >= 4 && N <= 64 && (N & (N - 1)) == 0, "a power of two up to the wave size");
  transpose_sum_step<N / 2, 32>(v, lane_id());
}

static constexpr int ROWDOT_MAX_ROWS = 8;   // launches with more rows than this go to the MFMA tiles
static constexpr int RD_R = 4;        // rows per tile
static constexpr int RD_C = 8;        // columns per workgroup pass
static constexpr int RD_WAVES = 4;
static constexpr int RD_PIECE = 512;  // contraction elements one wave instruction covers (64 lanes x 8)

// This wave's share of one column group: C weight rows against R input rows; `w[c]` and `x[r]` are wave-uniform row
// addresses, the lane's bytes off, off + step, ... (16 each, below `end`) of every row are multiplied.  Afterwards
// lane l holds the wave's total of value (r * C + c) = l / (64 / (R * C)) in acc[0].
template <typename T, int R, int C>
__device__ __forceinline__ void rowdot_wave(const char* const (&x)[RD_R], const char* const (&w)[C], unsigned off,
                                            unsigned step, unsigned end, float (&acc)[R * C]) {
#pragma unroll
  for (int i = 0; i < R * C; ++i) acc[i] = 0.0f;
#pragma unroll 1
  for (; off < end; off += step) {
    u32x4 wv[C], xv[R];
#pragma unroll
    for (int c = 0; c < C; ++c) wv[c] = __builtin_nontemporal_load((const u32x4*)(w[c] + off));   // read once
#pragma unroll
    for (int r = 0; r < R; ++r) xv[r] = *(const u32x4*)(x[r] + off);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[r * C + c] = Pair<T>::dot(xv[r][q], wv[c][q], acc[r * C + c]);
  }
  wave_transpose_sum<R * C>(acc);
}

// One column group by the whole workgroup, the waves taking the contraction pieces round-robin.  Leaves the R*C totals
// in part[0][r*C + c] (visible to the whole workgroup on return).
template <typename T, int R, int C, int NW>
__device__ __forceinline__ void rowdot_pass_r(const char* const (&x)[RD_R], const char* const (&w)[C], int K,
                                              float (&part)[NW][RD_R * C]) {
  constexpr int LPV = 64 / (R * C);              // lanes per value
  const int wave = threadIdx.x >> 6, lane = lane_id();
  float acc[R * C];
  rowdot_wave<T, R, C>(x, w, threadIdx.x * 16u, NW * RD_PIECE * 2u, (unsigned)K * 2u, acc);
  __syncthreads();                               // the previous pass has read `part`
  if (lane % LPV == 0) part[wave][lane / LPV] = acc[0];
  __syncthreads();
  if (threadIdx.x < R * C) {
    float v = 0.0f;
#pragma unroll
    for (int w_ = 0; w_ < NW; ++w_) v += part[w_][threadIdx.x];
    part[0][threadIdx.x] = v;                    // only this thread read column threadIdx.x of `part`
  }
  __syncthreads();
}
// A tile of one row (the usual one when there are more experts than rows) costs a quarter of the dot products and of
// the exchanges of a full one; same additions per value either way, hence the same bits.
template <typename T, int C, int NW>
__device__ __forceinline__ void rowdot_pass(const char* const (&x)[RD_R], const char* const (&w)[C], int K, int rows,
                                            float (&part)[NW][RD_R * C]) {
  if (rows == 1) rowdot_pass_r<T, 1, C, NW>(x, w, K, part);
  else rowdot_pass_r<T, RD_R, C, NW>(x, w, K, part);
}

template <typename T, bool GLU>
__global__ __launch_bounds__(RD_WAVES * 64) void s2s_rowdot_kernel(S2SArgs a, int n_groups, int gpw) {
  constexpr int R = RD_R, C = RD_C;
  __shared__ float part[RD_WAVES][R * C];
  const int wave = threadIdx.x >> 6, lane = lane_id();
  int e, row0, rows;
  if (!find_tile<R>(a.off, a.E, blockIdx.y, e, row0, rows)) return;

  // source rows of X and destination rows of Y (uniform over the workgroup)
  const char* x[R];
  int64_t dst[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t n = row0 + (r < rows ? r : rows - 1);
    int64_t src = n, d = n;
    if (!a.x_grouped || !a.y_grouped) {
      const int64_t i = a.idx[n];
      if (!a.x_grouped) src = i / a.fan_out;
      if (!a.y_grouped) d = i;
    }
    x[r] = (const char*)a.X + src * a.sxm * 2;
    dst[r] = d;
  }
  const char* Wb = (const char*)a.W + (int64_t)e * a.swe * 2;
  const T* bias = a.b ? (const T*)a.b + (int64_t)e * a.sbe : nullptr;
  const int F = a.N;                         // GLU: hidden width (the weights have 2F columns)
  const int K = a.K;

  for (int g = blockIdx.x * gpw; g < min(n_groups, (int)(blockIdx.x + 1) * gpw); ++g) {
    // column c of the pass -> weight column
    int col[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (GLU) {
        const int hc = g * (C / 2) + c % (C / 2);
        col[c] = hc < F ? hc + (c >= C / 2 ? F : 0) : 0;
      } else {
        const int n = g * C + c;
        col[c] = n < F ? n : 0;
      }
    }
    const char* wp[C];
#pragma unroll
    for (int c = 0; c < C; ++c) wp[c] = Wb + (int64_t)col[c] * a.swn * 2;
    rowdot_pass<T, C, RD_WAVES>(x, wp, K, rows, part);
    if (!GLU) {
      if (threadIdx.x < R * C) {
        const int r = threadIdx.x / C, c = threadIdx.x % C;
        const int n = g * C + c;
        if (r < rows && n < F) {
          float v = part[0][threadIdx.x];
          if (bias != nullptr) v += to_f32(bias[(int64_t)n * a.sbn]);
          ((T*)a.Y)[dst[r] * a.sym + n] = from_f32<T>(v);
        }
      }
    } else {
      // both halves are rounded to the storage type first and the hidden value is computed from the rounded values
      if (threadIdx.x < R * (C / 2)) {
        const int r = threadIdx.x / (C / 2), c = threadIdx.x % (C / 2);
        const int n = g * (C / 2) + c;
        if (r < rows && n < F) {
          float v1 = part[0][r * C + c], v2 = part[0][r * C + C / 2 + c];
          if (bias != nullptr) {
            v1 += to_f32(bias[(int64_t)n * a.sbn]);
            v2 += to_f32(bias[(int64_t)(F + n) * a.sbn]);
          }
          const T first = from_f32<T>(v1), second = from_f32<T>(v2);
          const bool gf = (a.act & 1) != 0;
          const float lin = to_f32(gf ? second : first), gat = to_f32(gf ? first : second);
          const int64_t row = row0 + r;            // the fused form works on rows in grouped order
          if (a.Y != nullptr) {
            ((T*)a.Y)[row * a.sym + n] = first;
            ((T*)a.Y)[row * a.sym + F + n] = second;
          }
          ((T*)a.H)[row * a.shm + n] = from_f32<T>(glu_h(a.act, gat, lin));
        }
      }
    }
  }
}

// Called with the operand checks of the MFMA path already done (K-contiguous weights, 16-byte aligned rows,
// K a multiple of 8).  Returns false when the shape is not this kernel's.
bool try_s2s_rowdot(const S2SArgs& a, int dtype, hipStream_t st, int& rc) {
  if (a.glu >= 2 || a.L > ROWDOT_MAX_ROWS) return false;
  const int64_t m_tiles = max_tiles(a.L, a.E, RD_R);
  const int n_groups = a.glu == 1 ? (a.N + RD_C / 2 - 1) / (RD_C / 2) : (a.N + RD_C - 1) / RD_C;
  // enough workgroups to give every CU several, few enough that the tile lookup is amortised
  int gpw = 1;
  while (gpw < 8 && m_tiles * ((n_groups + 2 * gpw - 1) / (2 * gpw)) >= 2048) gpw *= 2;
  const dim3 grid((unsigned)((n_groups + gpw - 1) / gpw), (unsigned)m_tiles), block(RD_WAVES * 64);
  if (dtype == SMOE_BF16) {
    if (a.glu) hipLaunchKernelGGL((s2s_rowdot_kernel<bf16_t, true>), grid, block, 0, st, a, n_groups, gpw);
    else hipLaunchKernelGGL((s2s_rowdot_kernel<bf16_t, false>), grid, block, 0, st, a, n_groups, gpw);
  } else {
    if (a.glu) hipLaunchKernelGGL((s2s_rowdot_kernel<f16_t, true>), grid, block, 0, st, a, n_groups, gpw);
    else hipLaunchKernelGGL((s2s_rowdot_kernel<f16_t, false>), grid, block, 0, st, a, n_groups, gpw);
  }
  rc = launch_status("s2s_rowdot_kernel");
  return true;
}

// =====================================================================================================
// The whole gated MLP of a decode step (a handful of (token, slot) rows, forward only) in two launches: layer 1 with
// its GLU, then layer 2 with the gate-weighted combine.  Neither needs the routing triple: every wave holds one
// expert id per lane and groups the rows itself (rows of one expert share a pass over that expert's weights, four
// at a time, in slot order).  Hidden rows travel between the launches in slot order (row t*k + j).
// Same arithmetic, in the same order, as the general path (row-dot scatter2scatter launches + combine), so the
// results are bit-identical to it.
// Reference: GLUMLP.forward, scattermoe/mlp.py:74-95, with flatten_sort_count (parallel_experts.py:14-21) and
// the gate combine of ParallelLinear.forward (parallel_experts.py:38-46) folded in.
//
// What bounds it: with narrow experts the launches are a latency chain, not a stream (one token, 128 experts, top-8,
// d = 2048, F = 768: 50 + 25 MB of weights).  Hence no serial sort ahead of the first weight load, all of a launch's
// weight rows requested at once - layer 2 gives every (tile, share of the contraction) of its eight columns a wave of
// its own instead of walking the experts one after the other - and short code: no private array indexed at run time
// (the compiler moves such an array to LDS and finds its place from the dispatch packet, which lies in host memory:
// 2 to 15 us per workgroup), no division, no column test (d and F are multiples of 8).
// Measured (layer 1 + layer 2, kernel time): that token 17.4 + 25.9 -> 10.5 + 7.3 us; two experts of d = 4096,
// F = 14336 (705 MB) 71 + 39 -> 71 + 36 us = 6.6 TB/s, the rate of a plain read.
// =====================================================================================================
struct DecodeTile { int rows, s0, s1, s2, s3; };     // up to RD_R slots of one expert (unused ones repeat the last)
struct DecodeRows {
  int e;                         // lane i: expert id of slot i (-1 past the last slot or outside [0, E))
  __device__ __forceinline__ void load(const DecodeArgs& a) {
    const unsigned i = lane_id(), t = (i * a.k_inv) >> 16;
    e = -1;
    if (i < (unsigned)(a.T * a.k)) {
      const int64_t id = a.experts[(int64_t)t * a.set + (int64_t)(i - t * a.k) * a.sek];
      if (id >= 0 && id < a.E) e = (int)id;          // rows with an invalid expert id are dropped
    }
  }
  __device__ __forceinline__ int expert(int slot) const { return __builtin_amdgcn_readlane(e, slot); }
  // The tile led by `slot`: it and the next up to RD_R - 1 slots of the same expert.  rows = 0: `slot` leads no tile
  // (invalid id, or the number of slots of its expert before it is no multiple of RD_R).
  __device__ __forceinline__ DecodeTile tile(int slot) const {
    const int es = expert(slot);
    const unsigned long long same = __ballot(e == es), from = ~0ull << slot;
    if (es < 0 || (__popcll(same & ~from) & (RD_R - 1)) != 0) return DecodeTile{0, 0, 0, 0, 0};
    unsigned long long left = same & from;
    DecodeTile t;
    t.rows = min(RD_R, __popcll(left));
    t.s0 = slot;
    left &= left - 1ull;
    t.s1 = left ? __ffsll((long long)left) - 1 : t.s0;
    left &= left - 1ull;
    t.s2 = left ? __ffsll((long long)left) - 1 : t.s1;
    left &= left - 1ull;
    t.s3 = left ? __ffsll((long long)left) - 1 : t.s2;
    return t;
  }
  // bit i: slot i leads a tile
  __device__ __forceinline__ unsigned long long leaders(int L) const {
    int rank = 0;
#pragma unroll 1
    for (int j = 0; j < L; ++j) rank += expert(j) == e && j < lane_id() ? 1 : 0;
    return __ballot(e >= 0 && (rank & (RD_R - 1)) == 0);
  }
};
__device__ __forceinline__ int slot_of(const DecodeTile& t, int r) {
  return r == 0 ? t.s0 : r == 1 ? t.s1 : r == 2 ? t.s2 : t.s3;
}

template <typename T>
__global__ __launch_bounds__(RD_WAVES * 64) void decode_l1_kernel(DecodeArgs a, int n_groups, int gpw) {
  constexpr int R = RD_R, C = RD_C;
  static_assert(R == 4, "DecodeTile holds four slots");
  __shared__ float part[RD_WAVES][R * C];
  DecodeRows ids;
  ids.load(a);
  const DecodeTile t = ids.tile(blockIdx.y);
  if (t.rows == 0) return;
  const int e = ids.expert(blockIdx.y);
  const char* x[R];
#pragma unroll
  for (int r = 0; r < R; ++r) x[r] = (const char*)a.X + (int64_t)(((unsigned)slot_of(t, r) * a.k_inv) >> 16) * a.sxm * 2;
  const int F = a.F, g_end = min(n_groups, (int)(blockIdx.x + 1) * gpw);
  const char* Wb = (const char*)a.W1 + (int64_t)e * a.sw1e * 2;
  const T* bias = a.b1 ? (const T*)a.b1 + (int64_t)e * a.sb1e : nullptr;
#pragma unroll 1
  for (int g = blockIdx.x * gpw; g < g_end; ++g) {
    const char* w[C];
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] = Wb + (int64_t)(g * (C / 2) + c % (C / 2) + (c >= C / 2 ? F : 0)) * a.sw1n * 2;
    rowdot_pass<T, C, RD_WAVES>(x, w, a.d, t.rows, part);
    const int r = threadIdx.x / (C / 2), c = threadIdx.x % (C / 2), n = g * (C / 2) + c;
    if (r < t.rows) {
      float v1 = part[0][r * C + c], v2 = part[0][r * C + C / 2 + c];
      if (bias != nullptr) {
        v1 += to_f32(bias[(int64_t)n * a.sb1n]);
        v2 += to_f32(bias[(int64_t)(F + n) * a.sb1n]);
      }
      const T first = from_f32<T>(v1), second = from_f32<T>(v2);
      const bool gf = (a.act & 1) != 0;
      const float lin = to_f32(gf ? second : first), gat = to_f32(gf ? first : second);
      ((T*)a.H)[(int64_t)slot_of(t, r) * a.shm + n] = from_f32<T>(glu_h(a.act, gat, lin));
    }
  }
}

// One unit of layer 2, by one wave: share `s` of the contraction for tile t; the totals go to part[slot][s][c].
template <typename T, int R, int C>
__device__ __forceinline__ void decode_l2_unit(const char* const (&x)[RD_R], const char* const (&w)[C],
                                               const DecodeTile& t, int s, int F, float (*part)[RD_WAVES][C]) {
  constexpr int LPV = 64 / (R * C);
  const int lane = lane_id();
  float acc[R * C];
  rowdot_wave<T, R, C>(x, w, (unsigned)(s * 64 + lane) * 16u, RD_WAVES * RD_PIECE * 2u, (unsigned)F * 2u, acc);
  const int r = lane / (LPV * C), c = (lane / LPV) % C;
  if (lane % LPV == 0 && r < t.rows) part[slot_of(t, r)][s][c] = acc[0];
}

template <typename T, int NW>
__global__ __launch_bounds__(NW * 64) void decode_l2_kernel(DecodeArgs a, int shares) {
  constexpr int R = RD_R, C = RD_C;
  __shared__ float part[DECODE_MAX_ROWS][RD_WAVES][C];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int L = a.T * a.k;
  const int n0 = blockIdx.x * C;
  DecodeRows ids;
  ids.load(a);
  // Unit u of the workgroup: share s of the contraction of a tile; wave by wave, shares fastest.  Piece p of RD_PIECE
  // elements belongs to share p % RD_WAVES, as in the general path (shares without a piece would add zero).
  unsigned long long lead = ids.leaders(L);
  int s = wave;
#pragma unroll 1
  while (true) {
#pragma unroll 1
    for (; s >= shares; s -= shares) lead &= lead - 1ull;
    if (lead == 0) break;
    const int first = __ffsll((long long)lead) - 1;
    const DecodeTile t = ids.tile(first);
    const char* W = (const char*)a.W2 + ((int64_t)ids.expert(first) * a.sw2e + (int64_t)n0 * a.sw2n) * 2;
    const char *w[C], *x[R];
#pragma unroll
    for (int c = 0; c < C; ++c) w[c] = W + c * a.sw2n * 2;
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = (const char*)a.H + (int64_t)slot_of(t, r) * a.shm * 2;
    if (t.rows == 1) decode_l2_unit<T, 1, C>(x, w, t, s, a.F, part);
    else decode_l2_unit<T, R, C>(x, w, t, s, a.F, part);
    s += NW;
  }
  __syncthreads();
  // layer-2 output of every slot, rounded to the storage type, then the sum over a token's slots: one wave, lane =
  // (slot, column)
  static_assert(DECODE_MAX_ROWS * C == 64, "the last step is one wave");
  if (wave != 0) return;
  const int slot = threadIdx.x / C, c = threadIdx.x % C;
  const int es = __shfl(ids.e, slot, 64);
  float y = 0.0f, gate = 0.0f;
  if (slot < L) {
    const unsigned t = ((unsigned)slot * a.k_inv) >> 16;
    gate = to_f32(((const T*)a.gates)[(int64_t)t * a.sgt + (int64_t)(slot - t * a.k) * a.sgk]);
    if (es >= 0) {
      for (int q = 0; q < shares; ++q) y += part[slot][q][c];
      if (a.b2 != nullptr) y += to_f32(((const T*)a.b2)[(int64_t)es * a.sb2e + (int64_t)(n0 + c) * a.sb2n]);
      y = to_f32(from_f32<T>(y));
    }
  }
  float acc = 0.0f;
  for (int j = 0; j < a.k; ++j) {
    const int from = ((slot * a.k + j) * C + c) & 63;              // lane of slot j of token `slot`
    acc = fmaf(__shfl(gate, from, 64), __shfl(y, from, 64), acc);
  }
  if (slot < a.T) ((T*)a.OUT)[(int64_t)slot * a.som + n0 + c] = from_f32<T>(acc);
}

template <typename T>
static void launch_decode_t(const DecodeArgs& a, hipStream_t st) {
  const int L = a.T * a.k;
  const int n_groups = a.F / (RD_C / 2);
  int gpw = 1;
  while (gpw < 8 && (int64_t)L * ((n_groups + 2 * gpw - 1) / (2 * gpw)) >= 2048) gpw *= 2;
  const dim3 grid1((unsigned)((n_groups + gpw - 1) / gpw), (unsigned)L), grid2((unsigned)(a.d / RD_C));
  hipLaunchKernelGGL(decode_l1_kernel<T>, grid1, dim3(RD_WAVES * 64), 0, st, a, n_groups, gpw);
  // a wave for every unit of the widest case, up to 16
  const int shares = std::min(RD_WAVES, (a.F + RD_PIECE - 1) / RD_PIECE);
  if (L * shares > 8) hipLaunchKernelGGL((decode_l2_kernel<T, 16>), grid2, dim3(16 * 64), 0, st, a, shares);
  else hipLaunchKernelGGL((decode_l2_kernel<T, 8>), grid2, dim3(8 * 64), 0, st, a, shares);
}

int launch_decode_glu_mlp(const DecodeArgs& a, int dtype, hipStream_t st) {
  if (dtype == SMOE_BF16) launch_decode_t<bf16_t>(a, st);
  else launch_decode_t<f16_t>(a, st);
  return launch_status("decode_glu_mlp kernels");
}

}  // namespace smoe
