// Measurement aid of bench.py, built into a library of its own (libsmoe_bench_probe.so): not part of the MoE path,
// not in the product library or its header.  What the matrix pipe of this GPU sustains on its own.  One wave per
// SIMD on every CU issues independent 16x16x32 bf16 MFMAs, the ones that the products are made of, on operands that stay in registers - no memory traffic,
// no LDS - so the rate is the shader clock the power management grants, and that clock depends on the operand bits
// (all-zero operands run near the nominal clock, operands with random signs and mantissas 15-25 % below it).
// bench.py reports both rates beside the roofline fraction, which is priced against the nominal peak.
#include <hip/hip_runtime.h>

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 probe_bf16x8;
typedef __attribute__((ext_vector_type(4))) float probe_f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned probe_u32x4;

static constexpr int PROBE_WGS = 256, PROBE_THREADS = 256, PROBE_MFMAS = 128, PROBE_ACCS = 32;

__device__ __forceinline__ unsigned probe_hash(unsigned x) {
  x ^= x >> 16; x *= 0x7feb352dU; x ^= x >> 15; x *= 0x846ca68bU; x ^= x >> 16;
  return x;
}

__global__ __launch_bounds__(PROBE_THREADS) void mfma_rate_kernel(float* out, int iters, int random_operands) {
  const int t = threadIdx.x + blockIdx.x * PROBE_THREADS;
  probe_bf16x8 a[8], b[8];
  for (int i = 0; i < 8; ++i) {
    probe_u32x4 ua, ub;
    for (int e = 0; e < 4; ++e) {
      // pairs of bf16 with exponents of values in [0.5, 2), random sign and mantissa - or zeros
      const unsigned ra = (probe_hash(t * 64 + i * 8 + e) & 0x807f807fU) | 0x3f003f00U;
      const unsigned rb = (probe_hash(t * 64 + i * 8 + e + 4) & 0x807f807fU) | 0x3f003f00U;
      ua[e] = random_operands ? ra : 0u;
      ub[e] = random_operands ? rb : 0u;
    }
    a[i] = __builtin_bit_cast(probe_bf16x8, ua);
    b[i] = __builtin_bit_cast(probe_bf16x8, ub);
  }
  // From assembly, in place: given the intrinsic, the compiler copies accumulators between the products.  It does not look into
  // assembly, so the distances to the operands' writing (two wait states) and to the results' reading (19) are kept here.
  probe_f32x4 acc[PROBE_ACCS];
  for (int i = 0; i < 8; ++i) asm volatile("s_nop 1" : "+v"(a[i]), "+v"(b[i]));
  for (int i = 0; i < PROBE_ACCS; ++i) {
    acc[i] = probe_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    asm volatile("s_nop 1" : "+a"(acc[i]));
  }
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int m = 0; m < PROBE_MFMAS; ++m)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[m % PROBE_ACCS]) : "v"(a[(m >> 2) & 7]), "v"(b[(m + (m >> 4)) & 7]));
  }
  for (int i = 0; i < PROBE_ACCS; ++i) asm volatile("s_nop 15\n\ts_nop 3" : "+a"(acc[i]));
  float s = 0.0f;
  for (int i = 0; i < PROBE_ACCS; ++i)
    for (int e = 0; e < 4; ++e) s += acc[i][e];
  out[t] = s;
}

}  // namespace

// out: 65536 floats of device memory (overwritten); *flop_out: flop count of the launch.  0 = launched,
// -1 = NULL pointer, -5 = iters out of range, > 0 = hipError_t of the launch.
extern "C" int smoe_bench_mfma_rate(float* out, int iters, int random_operands, double* flop_out, void* stream) {
  if (!out) return -1;
  if (iters < 1 || iters > (1 << 22)) return -5;
  if (flop_out) *flop_out = (double)PROBE_WGS * (PROBE_THREADS / 64) * (double)iters * PROBE_MFMAS * (2.0 * 16 * 16 * 32);
  hipLaunchKernelGGL(mfma_rate_kernel, dim3(PROBE_WGS), dim3(PROBE_THREADS), 0, (hipStream_t)stream, out, iters,
                     random_operands != 0);
  return (int)hipGetLastError();
}
