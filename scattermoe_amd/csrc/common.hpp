// Shared device/host helpers for the gfx950 ScatterMoE kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include "../../include/scattermoe_amd.h"

namespace smoe {

typedef __bf16 bf16_t;
typedef _Float16 f16_t;

// ---- error text, one slot per host thread -------------------------------------------------------
void set_error(const char* fmt, ...);
int launch_status(const char* what);  // hipGetLastError() -> return code (+ error text)

// ---- element conversion --------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ float to_f32(T v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f32(float v) { return (T)v; }

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// ---- gated linear unit math (shared by the stand-alone passes and the fused GEMM epilogues) ----------------
// Every multiplication / addition below is kept as written (no contraction into FMAs, no reassociation), so
// that the fused epilogues and the stand-alone passes give the same bits whatever code surrounds them.
// The reciprocal is the hardware's (v_rcp_f32, 1 ulp) rather than a correctly rounded division: the epilogues of
// the fused launches spend their time in this function (a division is about ten instructions), and every result
// is rounded to a 16-bit type or compared at 1e-4 afterwards.
__device__ __forceinline__ float sigmoidf_(float x) {
#pragma clang fp contract(off) reassociate(off)
  const float e = __expf(-x);
  const float d = 1.0f + e;
  return __builtin_amdgcn_rcpf(d);
}
// act & 1 selects which half of `pre` is the activated (gate) half: 0 = second half (GLUMLP of the reference),
// 1 = first half (the Hugging Face `act(gate) * up` convention).  The activation itself is SiLU.
__device__ __forceinline__ float act_f(int act, float g) {
#pragma clang fp contract(off) reassociate(off)
  (void)act;
  const float s = sigmoidf_(g);
  return g * s;
}
__device__ __forceinline__ float act_df(int act, float g) {
#pragma clang fp contract(off) reassociate(off)
  (void)act;
  const float s = sigmoidf_(g);
  const float a = 1.0f - s;
  const float b = g * a;
  const float c = 1.0f + b;
  return s * c;
}
// hidden value and the two gradients of h = act(gate) * lin
__device__ __forceinline__ float glu_h(int act, float gat, float lin) {
#pragma clang fp contract(off) reassociate(off)
  const float a = act_f(act, gat);
  return a * lin;
}
__device__ __forceinline__ float glu_dlin(int act, float dh, float gat) {
#pragma clang fp contract(off) reassociate(off)
  const float a = act_f(act, gat);
  return dh * a;
}
__device__ __forceinline__ float glu_dgat(int act, float dh, float gat, float lin) {
#pragma clang fp contract(off) reassociate(off)
  const float t = dh * lin;
  const float d = act_df(act, gat);
  return t * d;
}

// both gradients at once (one sigmoid); same operations in the same order as glu_dlin and glu_dgat
__device__ __forceinline__ void glu_grad(int act, float dh, float gat, float lin, float& d_lin, float& d_gat) {
#pragma clang fp contract(off) reassociate(off)
  (void)act;
  const float s = sigmoidf_(gat);
  const float a0 = gat * s;
  d_lin = dh * a0;
  const float t = dh * lin;
  const float a = 1.0f - s;
  const float b = gat * a;
  const float c = 1.0f + b;
  const float d = s * c;
  d_gat = t * d;
}

// gated unit of the gpt-oss experts over one (gate, up) pair and its gradient (clamped inputs pass no gradient)
__device__ __forceinline__ float oss_h(float gate, float up, float alpha, float limit) {
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  return (u + 1.0f) * (g * sigmoidf_(alpha * g));
}
__device__ __forceinline__ void oss_grad(float gate, float up, float dh, float alpha, float limit, float& dgate,
                                         float& dup) {
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  const float s = sigmoidf_(alpha * g);
  const float glu = g * s;
  dup = (up >= -limit && up <= limit) ? dh * glu : 0.0f;
  const float dglu = dh * (u + 1.0f);
  dgate = gate <= limit ? dglu * (s + alpha * g * s * (1.0f - s)) : 0.0f;
}

// ---- expert-aligned tile lookup -------------------------------------------------------------------
// Inclusive sums over the wave's lanes: row shifts and row broadcasts (a lane without a source adds 0).  The lookups below stand at
// the head of every tile, where nothing hides them, and are nothing but latency: a scan through six LDS shuffles takes about 700
// cycles, this one about 60.
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);       // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);       // lane 15 of a row to the next row
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);       // lane 31 to the upper half
  return v;
}
// Rows [lo, hi) of expert e0 + lane (none beyond the last one).
__device__ __forceinline__ void load_expert_rows(const int64_t* __restrict__ off, int E, int e0, int& lo, int& hi) {
  const int e = e0 + lane_id();
  lo = hi = 0;
  if (e < E) {
    hi = (int)off[e];
    lo = e ? (int)off[e - 1] : 0;
  }
}

// Rows are expert-sorted; expert e owns rows [off[e-1], off[e]).  Tiles of height BM never straddle
// two experts: expert e contributes ceil(count_e / BM) tiles and tiles are numbered expert-major.
// Every wave of the block runs this redundantly and gets the same (uniform) answer.
// Returns false when `t` is past the last tile (the grid is sized by the host-known upper bound
// floor(L/BM) + E, so surplus blocks simply exit).
// `skip_small` > 0: an expert's last, partly filled tile is left out when it holds at most `skip_small` rows (another
// launch with lower tiles takes those rows, see find_remainder).
template <int BM>
__device__ __forceinline__ bool find_tile(const int64_t* __restrict__ off, int E, int t,
                                          int& expert, int& row_start, int& rows, int skip_small = 0) {
  int tiles_before = 0, lo, hi;
  load_expert_rows(off, E, 0, lo, hi);
  for (int e0 = 0; e0 < E; e0 += 64) {
    int lo_next = 0, hi_next = 0;                               // of the next 64 experts: on their way meanwhile
    if (e0 + 64 < E) load_expert_rows(off, E, e0 + 64, lo_next, hi_next);
    int nt = (hi - lo + BM - 1) / BM;
    const int rem = (hi - lo) % BM;
    if (rem != 0 && rem <= skip_small) nt -= 1;
    const int incl = wave_scan(nt);
    const int cum = tiles_before + incl;
    const unsigned long long hit = __ballot(cum > t);
    if (hit) {
      const int src = __ffsll((long long)hit) - 1;
      // readlane: the answer stays in scalar registers (a shuffle's would hold vector registers across the main loop)
      const int lo_s = __builtin_amdgcn_readlane(lo, src), hi_s = __builtin_amdgcn_readlane(hi, src);
      const int first = __builtin_amdgcn_readlane(cum - nt, src);
      expert = e0 + src;
      row_start = lo_s + (t - first) * BM;
      rows = min(BM, hi_s - row_start);
      return true;
    }
    tiles_before += __builtin_amdgcn_readlane(incl, 63);
    lo = lo_next, hi = hi_next;
  }
  return false;
}

// Number of tile rows of height BM that the experts have.
template <int BM>
__device__ __forceinline__ int count_tile_rows(const int64_t* __restrict__ off, int E) {
  int n = 0;
  for (int e = lane_id(); e < E; e += 64) n += ((int)(off[e] - (e ? off[e - 1] : 0)) + BM - 1) / BM;
  return __builtin_amdgcn_readlane(wave_scan(n), 63);
}

// Largest of the wave's values, in a scalar register: six row shifts and row broadcasts (lanes without a source keep
// their own value).
__device__ __forceinline__ int wave_max(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false));       // row_shr 1, 2, 4, 8
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xf, 0xf, false));
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));       // lane 15 of a row to the next row
  v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));       // lane 31 to the upper half
  return __builtin_amdgcn_readlane(v, 63);
}

// The same for launches whose workgroups take all output tiles in an order that keeps together what shares operands:
// expert by expert, inside an expert column by column (of `n_tiles`), the expert's tile rows of a column side by side.
// The XCD of a workgroup is `pid` % 8; the order is cut into 8 R chunks of equal length and XCD x takes the chunks
// x, x + 8, ... (in turn from either end).  How many tiles there are is known only here, from `off`: R = 1, or with
// `round` > 0 as many as there are rounds of that many tiles (256 or more).  A grid of chunked_grid() workgroups covers every tile.
// Returns 1: this workgroup's tile; 0: none; -1: the experts that have rows differ in tile rows by more than a quarter of
// the most, so that equal numbers of tiles are not equal work: another order has to be taken (the same answer in every
// workgroup, and for the same loads in any order).  HEIGHTS: tiles cost their rows in blocks of 64, so loads whose blocks
// differ by no more are even too: around a multiple of BM rows most experts end in a tile that others don't have
// (us, stripes -> chunks, 32 experts x 238 rows, one of them 270, 2880 -> 2 x 2880 325 -> 273, 2880 -> 2880 218 -> 151;
// 128 x 238, 16 of them 270, 2048 -> 2 x 768 290 -> 265, 768 -> 2048 159 -> 155).
template <int BM, bool HEIGHTS>
__device__ __forceinline__ int find_tile_chunked(const int64_t* __restrict__ off, int E, int pid, int n_tiles,
                                                 int round, int& expert, int& row_start, int& rows, int& column) {
  // experts e0 .. e0 + 63, one per lane; the first 128 are loaded once, side by side
  int lo0, hi0, lo1 = 0, hi1 = 0;
  load_expert_rows(off, E, 0, lo0, hi0);
  if (E > 64) load_expert_rows(off, E, 64, lo1, hi1);
  auto load = [&](int e0, int& lo, int& hi, int& nt) {
    if (e0 == 0) lo = lo0, hi = hi0;
    else if (e0 == 64) lo = lo1, hi = hi1;
    else load_expert_rows(off, E, e0, lo, hi);
    nt = (hi - lo + BM - 1) / BM;
  };
  int lo, hi, nt;
  load(0, lo, hi, nt);
  // tile rows, and blocks of 64 rows, of an expert that has any
  auto blocks = [](int l_, int h_) { return (h_ - l_ + 63) >> 6; };
  int most = nt, least = nt > 0 ? nt : 0x7fffffff, most_b = blocks(lo, hi), least_b = hi > lo ? most_b : 0x7fffffff;
  for (int e0 = 64; e0 < E; e0 += 64) {
    int l_, h_, n_;
    load(e0, l_, h_, n_);
    most = max(most, n_);
    most_b = max(most_b, blocks(l_, h_));
    if (n_ > 0) least = min(least, n_), least_b = min(least_b, blocks(l_, h_));
  }
  auto differ = [](int most_, int least_) {                   // by more than a quarter of the most
    most_ = wave_max(most_);
    return 4 * (most_ + wave_max(-least_)) > most_;
  };
  if (__ballot(most > 1) && differ(most, least) && (!HEIGHTS || differ(most_b, least_b))) return -1;
  int incl = wave_scan(nt);
  int total = __builtin_amdgcn_readlane(incl, 63);
  for (int e0 = 64; e0 < E; e0 += 64) {
    int l_, h_, n_;
    load(e0, l_, h_, n_);
    total += __builtin_amdgcn_readlane(wave_scan(n_), 63);
  }
  const unsigned tiles = (unsigned)total * n_tiles;
  const unsigned R = round && tiles >= round + round / 2u ? (tiles + round / 2u) / round : 1;
  const unsigned len = __builtin_amdgcn_readfirstlane((tiles + 8 * R - 1) / (8 * R));
  if (len == 0) return 0;
  const unsigned x = pid & 7, i = (unsigned)pid >> 3, c = i / len;
  const unsigned l = (c * 8 + ((c & 1) ? 7 - x : x)) * len + (i - c * len);
  if (c >= R || l >= tiles) return 0;
  int before = 0;                                             // tile rows of the experts before this group
  for (int e0 = 0;;) {
    const unsigned cum = before + incl;
    const unsigned long long hit = __ballot(cum * n_tiles > l);
    if (hit) {
      const int src = __ffsll((long long)hit) - 1;
      const int lo_s = __builtin_amdgcn_readlane(lo, src), hi_s = __builtin_amdgcn_readlane(hi, src);
      const unsigned nt_s = __builtin_amdgcn_readlane(nt, src);
      const unsigned in_expert = l - (__builtin_amdgcn_readlane((int)cum, src) - nt_s) * n_tiles;
      column = __builtin_amdgcn_readfirstlane(in_expert / nt_s);
      expert = e0 + src;
      row_start = lo_s + __builtin_amdgcn_readfirstlane(in_expert - column * nt_s) * BM;
      rows = min(BM, hi_s - row_start);
      return 1;
    }
    before += __builtin_amdgcn_readlane(incl, 63);
    e0 += 64;
    if (e0 >= E) return 0;
    load(e0, lo, hi, nt);
    incl = wave_scan(nt);
  }
}
// Workgroups of such a launch of at most `tiles` tiles: 8 R chunks round up by less than 8 R <= tiles / 32 + 8.
static inline int64_t chunked_grid(int64_t tiles) { return (tiles + tiles / 32 + 16 + 7) / 8 * 8; }

// The rows that find_tile<BM>(..., skip_small) leaves out, as one tile per expert: the last n % BM rows of expert e
// when there are between 1 and `small` of them.
template <int BM>
__device__ __forceinline__ bool find_remainder(const int64_t* __restrict__ off, int E, int e, int small,
                                               int& row_start, int& rows) {
  if (e >= E) return false;
  const int hi = (int)off[e], lo = e ? (int)off[e - 1] : 0;
  const int rem = (hi - lo) % BM;
  if (rem == 0 || rem > small) return false;
  row_start = hi - rem;
  rows = rem;
  return true;
}

static inline int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Upper bound on the number of expert-aligned tiles of height bm over L rows and E experts.
static inline int64_t max_tiles(int64_t L, int E, int bm) {
  int64_t a = L / bm + E;        // sum ceil(c_e/bm) <= floor(L/bm) + E
  int64_t b = L;                 // and never more than one tile per row
  int64_t r = a < b ? a : b;
  return r < 1 ? 1 : r;
}

// ---- kernel launchers implemented in the individual .hip files ---------------------------------------
struct S2SArgs {
  const void* X; int64_t sxm, sxk;
  const void* W; int64_t swe, swk, swn;
  const void* b; int64_t sbe, sbn;
  void* Y; int64_t sym, syn;
  const int64_t* eid; const int64_t* idx; const int64_t* off;
  int L, K, N, E, fan_out;
  int x_grouped, y_grouped;
  // fused gated-linear-unit epilogues (MFMA path only, rows in grouped order):
  //   glu == 1: W has 2N columns; Y (may be NULL) receives the pre-activation (L, 2N), H the hidden (L, N)
  //   glu == 2: Y receives d(pre) (L, 2N) computed from the product (= d hidden) and the saved pre-activation AUX
  //   glu == 3: gpt-oss form, N = 2F columns holding (gate, up) pairs: Y (may be NULL) receives the pre-activation
  //             (L, 2F), H the hidden (L, F)
  //   glu == 4: gpt-oss form, N = F: Y receives d(pre) (L, 2F) from the product (= d hidden) and the saved AUX
  int glu = 0, act = 0;
  const void* aux = nullptr; int64_t saux = 0;
  void* H = nullptr; int64_t shm = 0;
  float alpha = 0.0f, limit = 0.0f;
  // Part of a product split by tile rows (MFMA path only): the launch covers the tile rows
  // [m_begin, m_begin + m_count) of its tile height.
  int m_begin = 0, m_count = 0x7fffffff;
  // Products whose experts end in a partly filled tile (MFMA path only).  1: this launch leaves out every expert's
  // last tile when it holds at most 128 rows; 2: this launch takes exactly those rows, one tile row per expert.
  int tail_mode = 0;
  // The contraction of every tile is cut into `ksplit` parts of `k_part` (the last may be shorter), one workgroup each, which
  // leave their float32 sums in `partial` (tail_mode 2: accumulators, see splitk_floats; whole products: rows, see
  // parts_sum_kernel); a second launch adds the parts up in a fixed order and writes the output rows.
  // `partial` / `partial_floats`: the caller's workspace, may be NULL / 0.
  int ksplit = 1, k_part = 0;
  float* partial = nullptr;
  int64_t partial_floats = 0;
};

struct XtYArgs {
  const void* DY; int64_t sdym, sdyn;
  const void* X; int64_t sxm, sxk;
  void* DW; int64_t sdwe, sdwk, sdwn;
  void* Db; int64_t sdbe, sdbn;
  const int64_t* off;
  int L, K, N, E;
  // X is the (L / fan_out, K) matrix the grouped rows would be gathered from: grouped row r = X[idx[r] / fan_out]
  // (MFMA path only); NULL: X holds the L grouped rows themselves
  const int64_t* idx = nullptr;
  int fan_out = 1;
};

struct GroupArgs {
  const void* A; int64_t sam, sak;
  const void* coeff;
  void* Y; int64_t sym, syk;
  const int64_t* idx;
  int L, K, fan_out;
};

// Whole gated MLP for at most DECODE_MAX_ROWS (token, slot) rows, forward only (csrc/s2s_rowdot.hip)
static constexpr int DECODE_MAX_ROWS = 8;
struct DecodeArgs {
  const void* X; int64_t sxm;                        // (T, d) tokens, columns contiguous
  const int64_t* experts; int64_t set, sek;          // (T, k) expert ids
  const void* gates; int64_t sgt, sgk;               // (T, k) routing weights
  const void* W1; int64_t sw1e, sw1n;                // (E, 2F, d), d contiguous
  const void* b1; int64_t sb1e, sb1n;                // (E, 2F) or NULL
  const void* W2; int64_t sw2e, sw2n;                // (E, d, F), F contiguous
  const void* b2; int64_t sb2e, sb2n;                // (E, d) or NULL
  void* H; int64_t shm;                              // (T*k, F) workspace: hidden rows in slot order
  void* OUT; int64_t som;                            // (T, d)
  int T, k, d, F, E, act;
  unsigned k_inv;                                    // ceil(65536 / k): slot i belongs to token (i * k_inv) >> 16
};
int launch_decode_glu_mlp(const DecodeArgs& a, int dtype, hipStream_t st);

int launch_s2s_generic(const S2SArgs& a, int dtype, hipStream_t st);
int launch_xty_generic(const XtYArgs& a, int dtype, hipStream_t st);
int launch_group(const GroupArgs& a, int dtype, hipStream_t st);
// MFMA paths return 1 if they took the call, 0 if the shape/layout is not theirs, <0 / >1 never.
bool try_s2s_mfma(const S2SArgs& a, int dtype, hipStream_t st, int& rc);
// float32 values of workspace with which a plain bf16 / fp16 product of these sizes can split the contraction of
// its experts' last, sparsely filled tiles (0: the product would not use one)
int64_t s2s_workspace_floats(int64_t L, int64_t K, int64_t N, int E, int dtype);
bool try_s2s_f32(const S2SArgs& a, hipStream_t st, int& rc);     // float32 MFMA paths (csrc/gemm_f32.hip)
bool try_xty_f32(const XtYArgs& a, hipStream_t st, int& rc);
bool try_s2s_rowdot(const S2SArgs& a, int dtype, hipStream_t st, int& rc);   // few-row launches; after try_s2s_mfma's checks
bool try_xty_mfma(const XtYArgs& a, int dtype, hipStream_t st, int& rc);

int launch_combine(const void* Y, int64_t sy, const void* G, int64_t sgt, int64_t sgk, void* O, int64_t so,
                   int64_t Tn, int k, int N, int dtype, hipStream_t st);
int launch_gate_grad(const void* Y, int64_t sy, const void* D, int64_t sd, void* DG, int64_t sgt, int64_t sgk,
                     int64_t Tn, int k, int N, int dtype, hipStream_t st);
int launch_glu_fwd(const void* pre, int64_t sp, void* h, int64_t sh, int64_t rows, int f, int act, int dtype,
                   hipStream_t st);
int launch_glu_bwd(const void* pre, int64_t sp, const void* dh, int64_t sdh, void* dpre, int64_t sdp, int64_t rows,
                   int f, int act, int dtype, hipStream_t st);

int launch_oss_glu_fwd(const void* pre, int64_t sp, void* h, int64_t sh, int64_t rows, int f, float alpha, float limit,
                       int dtype, hipStream_t st);
int launch_oss_glu_bwd(const void* pre, int64_t sp, const void* dh, int64_t sdh, void* dpre, int64_t sdp, int64_t rows,
                       int f, float alpha, float limit, int dtype, hipStream_t st);
int launch_topk_softmax(const void* logits, int64_t slt, int64_t sle, float* w, int64_t swt, int64_t swk,
                        int64_t* idx, int64_t sit, int64_t sik, int64_t Tn, int E, int k, int renorm, int dtype,
                        hipStream_t st);
int launch_route(const void* expert_idxs, int idx_dtype, int64_t L, int E, int64_t* eid_out,
                 int64_t* idx_out, int64_t* off_out, void* ws, hipStream_t st);
size_t route_workspace_bytes(int64_t L, int E);
int launch_route_static(const void* expert_idxs, int idx_dtype, int64_t L, int E, int64_t* eid_out,
                        int64_t* idx_out, int64_t* off_out, hipStream_t st);
int route_static_init();
int launch_offsets_from_sorted(const int64_t* eid, int64_t L, int E, int64_t* off, hipStream_t st);
int launch_group_by_source(const GroupArgs& a, int* inv, int dtype, hipStream_t st);
int launch_invert_index(const int64_t* idx, int64_t L, int* inv, hipStream_t st);   // inv[idx[r]] = r
// gate gradient and the scaled, expert-sorted copy of the output gradient in one pass (csrc/fused.hip);
// SMOE_ERR_UNSUPPORTED when rows are not 16-byte pieces
int launch_gate_grad_group(const void* Y, int64_t sy, const void* D, int64_t sd, const void* G, int64_t sgt, int64_t sgk,
                           const int64_t* idx, int* inv, void* DY, int64_t sdy, void* DG, int64_t sdgt, int64_t sdgk,
                           int64_t Tn, int k, int N, int dtype, hipStream_t st);

}  // namespace smoe
