// bf16 instantiation of the MFMA kernels (gemm_mfma.hpp) and the choice between them and the other paths; the fp16
// instantiation is a source of its own (gemm_mfma_f16.hip) so that the two compile side by side.
#include "gemm_mfma.hpp"

namespace smoe {

int dispatch_s2s_f16(const S2SArgs& a, bool b_tr, hipStream_t st);
int dispatch_xty_bf16(const XtYArgs& a, hipStream_t st);
int dispatch_xty_f16(const XtYArgs& a, hipStream_t st);

int64_t s2s_workspace_floats(int64_t L, int64_t K, int64_t N, int E, int dtype) {
  if ((dtype != SMOE_BF16 && dtype != SMOE_F16) || E <= 0) return 0;
  if (const int parts = whole_parts_for(L, K, N, E); parts > 1) return L * N * parts;
  if (L / E < REMAINDER_MIN_AVG_ROWS) return 0;
  if (2.0 * (double)L * K * N < REMAINDER_MIN_FLOP) return 0;
  const int ks = tail_ksplit_for(K, N, E, 0);
  return ks > 1 ? splitk_floats(N, E, ks) : 0;
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool fits_u32(int64_t bytes) { return bytes >= 0 && bytes < (int64_t)0xfff00000LL; }

bool try_s2s_mfma(const S2SArgs& a, int dtype, hipStream_t st, int& rc) {
  if (dtype == SMOE_F32) return try_s2s_f32(a, st, rc);
  if (dtype != SMOE_BF16 && dtype != SMOE_F16) return false;
  if (a.K < 8 || a.K % 8 != 0) return false;
  if (a.sxk != 1 || a.sxm % 8 != 0 || !aligned16(a.X)) return false;
  if (a.syn != 1) return false;
  if (!aligned16(a.W) || a.swe % 8 != 0) return false;
  bool b_tr;
  if (a.swk == 1 && a.swn % 8 == 0) b_tr = false;
  else if (a.swn == 1 && a.swk % 8 == 0 && a.N % 8 == 0) b_tr = true;
  else return false;
  // lane offsets inside the kernel are 32-bit byte offsets from a scalar base (X, and W[e])
  const int64_t x_rows = a.x_grouped ? 256 : a.L / a.fan_out;        // grouped rows: relative to the tile's first row
  if (fits_u32((x_rows - 1) * a.sxm * 2 + (int64_t)a.K * 2) == false) return false;
  const int64_t w_cols = a.glu == 1 ? 2 * (int64_t)a.N : a.N;
  if (b_tr ? !fits_u32(BK * a.swk * 2 + w_cols * 2) : !fits_u32((w_cols - 1) * a.swn * 2 + (int64_t)a.K * 2))
    return false;
  if (!b_tr && try_s2s_rowdot(a, dtype, st, rc)) return true;
  rc = dtype == SMOE_BF16 ? dispatch_s2s<bf16_t>(a, b_tr, st) : dispatch_s2s_f16(a, b_tr, st);
  return true;
}

bool try_xty_mfma(const XtYArgs& a, int dtype, hipStream_t st, int& rc) {
  if (dtype == SMOE_F32) return a.idx == nullptr && try_xty_f32(a, st, rc);    // the float32 kernels do not gather
  if (dtype != SMOE_BF16 && dtype != SMOE_F16) return false;
  if (a.K % 8 != 0 || a.N % 8 != 0) return false;
  if (a.sdyn != 1 || a.sxk != 1 || a.sdym % 8 != 0 || a.sxm % 8 != 0) return false;
  if (!aligned16(a.DY) || !aligned16(a.X)) return false;
  if (a.sdwk != 1 && a.sdwn != 1) return false;
  if (!fits_u32(BK * a.sdym * 2 + (int64_t)a.N * 2) || !fits_u32(BK * a.sxm * 2 + (int64_t)a.K * 2)) return false;
  // gathered X: lane offsets are 32-bit byte offsets from the start of the token matrix
  if (a.idx != nullptr && !fits_u32(((int64_t)a.L / a.fan_out) * a.sxm * 2 + (int64_t)a.K * 2)) return false;
  // Looking the rows up costs the kernel about 4 % of its time; the gathered copy it saves costs 4 K bytes of HBM
  // traffic per row against 2 K N flops, i.e. a share of the kernel time that shrinks with N.  Measured per training
  // step: N = 1536 (Qwen-like, top-8) 9.12 -> 8.90 ms, N = 5760 (gpt-oss-like) 6.07 -> 6.03 ms, N = 28672 (Mixtral)
  // 31.3 -> 31.5 ms: wide layers keep the separate pass.  Not where X is streamed past a held operand, which looks every row up
  // once per unit (the experts of more than 256 rows do so in every slice of a tile, all the same): random launches of N from
  // 6200 on, even loads / as 1 / rank^0.42, ^0.84, ^1.8, against the copy and 128 x 128 tiles 1.42 / 1.17 / 1.05 / 0.99; where X
  // is held (N contiguous) 1.3 / 1.0 / 0.90 / 0.88 with lookups, 1.27 / 1.02 / 0.94 / 0.93 over the copy.
  if (a.idx != nullptr && a.N > XTY_GATHER_MAX_N && !(xty_held(a) && a.sdwk == 1)) return false;
  rc = dtype == SMOE_BF16 ? dispatch_xty_bf16(a, st) : dispatch_xty_f16(a, st);
  return true;
}

}  // namespace smoe

