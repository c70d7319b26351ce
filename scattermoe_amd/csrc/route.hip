// Routing prep: deterministic stable counting sort of flattened expert ids + inclusive offsets.
// Counterpart of flatten_sort_count (scattermoe/parallel_experts.py:14-21), which runs
// torch.sort + bincount + cumsum.  Keys are tiny (expert ids), so a counting sort with an LDS
// histogram per block and a wavefront match/rank scatter replaces the generic 64-bit radix sort.
//
// Inputs of up to 16384 rows (one workgroup of 4 or 16 waves) run in ONE launch; larger ones in three:
//   hist    : per-chunk LDS histogram                       -> counts[chunk][E]
//   scan    : exclusive scan over (expert-major, chunk)     -> bases[chunk][E], off[E]
//   scatter : stable rank inside the chunk + base           -> eid_out, idx_out
// (us, all three, chunks ranked by 16 waves in one pass instead of 4 waves in two: 31992 rows of 128 experts 26.9 -> 13.6,
// 32768 of 8 18.7 -> 11.1, 262144 of 128 33.9 -> 20.6)
// The result is independent of scheduling: every output position is a pure function of the input.
#include "common.hpp"
#include <mutex>

namespace smoe {

static constexpr int kRouteThreads = 256;
static constexpr int kRouteChunk = 4096;       // elements per block
static constexpr int kRouteMaxE = 2048;        // LDS: (waves+1) * E ints
static constexpr int kRouteFusedMax = 16384;   // rows one workgroup of 1024 threads sorts by itself, without a
                                               // workspace (the three launches: 10 us and more) ...
static constexpr int kRouteFusedMaxE = 512;    // ... for at most this many experts (17 * E ints of LDS)

// An id is compared at its full width: the low half of a 64-bit id that is no expert may look like one.
template <typename I>
__device__ __forceinline__ bool is_expert(I id, int E) { return (uint64_t)(int64_t)id < (uint64_t)E; }

// Lanes of the wave that hold the same key as this lane (keys < 2^nbits), inactive lanes excluded.
__device__ __forceinline__ unsigned long long match_any(int key, int nbits, bool active) {
  unsigned long long m = __ballot(active);
  for (int b = 0; b < nbits; ++b) {
    const bool bit = (key >> b) & 1;
    const unsigned long long v = __ballot(bit);
    m &= bit ? v : ~v;
  }
  return m;
}

__device__ __forceinline__ int bits_for(int E) {
  int nbits = 0;
  while ((1 << nbits) < E) ++nbits;
  return nbits;
}

// A wave's contiguous segment of at most IT * 64 rows, read once: key[u] is the id of row seg_lo + 64 u + lane (-1: no
// row, or an id that is no expert), loc[u] its rank among the wave's rows of that expert.  hist_w (zero on entry) ends
// as the wave's histogram: equal ids of 64 rows are found by match_any and added by one lane, whose returned value is
// the number of such rows before these (a wave's LDS operations complete in order), so neither many lanes on one
// counter nor a second counting pass is needed to place the rows.
template <typename I, int IT>
__device__ __forceinline__ void wave_rank(const I* __restrict__ ids, int64_t seg_lo, int64_t seg_hi, int E, int nbits,
                                          int* __restrict__ hist_w, int (&key)[IT], int (&loc)[IT]) {
  const int lane = lane_id();
  const unsigned long long lt = (1ull << lane) - 1ull;
  I id[IT];                             // all loads ahead of the first comparison: one memory round trip, not IT of them
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const int64_t p = seg_lo + u * 64 + lane;
    id[u] = p < seg_hi ? ids[p] : (I)0;
  }
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    const bool ok = seg_lo + u * 64 + lane < seg_hi && is_expert(id[u], E);
    key[u] = ok ? (int)id[u] : -1;
    loc[u] = 0;
    if (seg_lo + u * 64 < seg_hi) {
      const unsigned long long same = match_any(ok ? key[u] : 0, nbits, ok);
      const int leader = __ffsll((long long)same) - 1;   // -1 only for lanes with ok == false
      int first = 0;
      if (ok && lane == leader) first = atomicAdd(&hist_w[key[u]], __popcll(same));
      first = __shfl(first, leader < 0 ? 0 : leader, 64);
      loc[u] = first + __popcll(same & lt);
    }
  }
}

// hist[w][e], w < W -> number of rows of expert e in the waves before w (from `run` on); returns the end.
// All counters are read before the first is written: 16 LDS round trips one after the other otherwise.
template <int W>
__device__ __forceinline__ int prefix_over_waves(int* __restrict__ hist, int E, int e, int run) {
  int c[W];
#pragma unroll
  for (int w = 0; w < W; ++w) c[w] = hist[w * E + e];
#pragma unroll
  for (int w = 0; w < W; ++w) {
    hist[w * E + e] = run;
    run += c[w];
  }
  return run;
}

// The places behind the last valid row (as many as there are ids that are no expert): an id past the experts and an
// index that is no slot, which every launch that reads the vectors skips.  Unwritten they would hold what the memory
// held before: an address to nowhere, or a slot that has a place already.
__device__ __forceinline__ void fill_dropped(int64_t first, int64_t step, int64_t L, int E, int64_t* __restrict__ eid_out,
                                             int64_t* __restrict__ idx_out) {
  for (int64_t i = first; i < L; i += step) {
    eid_out[i] = (int64_t)E;
    idx_out[i] = -1;
  }
}

// ---- single-launch path: whole input in one block ------------------------------------------------
// Bound by latency (one read of the ids, LDS counters, four barriers) and, written row by row, by one CU's rate of
// scattered 8-byte stores: the sorted rows are put together in LDS and written out in whole lines.
// us, two passes over the ids by 4 waves (up to 4096 rows) or 16, rows written one by one -> now:
// 1554 rows of 8 experts 6.6 -> 3.8, 1600 of 128 8.6 -> 4.6, 6004 of 32 8.4 -> 7.8, 16384 of 128 23.2 -> 19.3.
template <typename I, int THREADS, int IT>
__global__ __launch_bounds__(THREADS) void route_fused_kernel(
    const I* __restrict__ ids, int L, int E, int64_t* __restrict__ eid_out,
    int64_t* __restrict__ idx_out, int64_t* __restrict__ off_out) {
  constexpr int W = THREADS / 64, EMAX = W == 16 ? kRouteFusedMaxE : kRouteMaxE;
  static_assert(THREADS * IT <= 65536 && EMAX <= 65536, "row and expert share a word");
  __shared__ int hist[W * EMAX];        // [W][E] wave histograms, then the wave's first place within the expert
  __shared__ int total[EMAX];           // [E] rows of the expert, then its first place
  __shared__ unsigned sorted[THREADS * IT];
  __shared__ int n_valid;
  const int tid = threadIdx.x, w = tid >> 6;
  for (int i = tid; i < W * E; i += THREADS) hist[i] = 0;
  __syncthreads();
  const int seg = ((L + W - 1) / W + 63) / 64 * 64;      // at most IT * 64 (the launcher's choice)
  const int lo = min(w * seg, L), hi = min(lo + seg, L);
  int key[IT], loc[IT];
  wave_rank<I, IT>(ids, lo, hi, E, bits_for(E), hist + w * E, key, loc);
  __syncthreads();
  for (int e = tid; e < E; e += THREADS) total[e] = prefix_over_waves<W>(hist, E, e, 0);
  __syncthreads();
  // exclusive scan of totals over experts (wave 0, 64 experts per step), inclusive offsets out
  if (w == 0) {
    const int lane = lane_id();
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane;
      const int c = e < E ? total[e] : 0;
      int incl = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        int v = __shfl_up(incl, d, 64);
        if (lane >= d) incl += v;
      }
      if (e < E) {
        total[e] = carry + incl - c;           // exclusive base of expert e
        off_out[e] = (int64_t)(carry + incl);  // inclusive end
      }
      carry += __shfl(incl, 63, 64);
    }
    if (lane == 0) n_valid = carry;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u)
    if (key[u] >= 0)
      sorted[total[key[u]] + hist[w * E + key[u]] + loc[u]] = (unsigned)key[u] << 16 | (unsigned)(lo + u * 64 + lane_id());
  __syncthreads();
  for (int i = tid; i < n_valid; i += THREADS) {
    eid_out[i] = (int64_t)(sorted[i] >> 16);
    idx_out[i] = (int64_t)(sorted[i] & 0xffff);
  }
  fill_dropped(n_valid + tid, THREADS, L, E, eid_out, idx_out);
}

// ---- three-launch path ------------------------------------------------------------------------------
template <typename I, int THREADS>
__global__ __launch_bounds__(THREADS) void route_hist_kernel(
    const I* __restrict__ ids, int64_t L, int E, int* __restrict__ counts /*[nchunk][E]*/) {
  extern __shared__ int lds[];  // [E]
  const int tid = threadIdx.x;
  for (int i = tid; i < E; i += THREADS) lds[i] = 0;
  __syncthreads();
  const int64_t lo = (int64_t)blockIdx.x * kRouteChunk;
  const int64_t hi = min(lo + kRouteChunk, L);
  for (int64_t p = lo + tid; p < hi; p += THREADS) {
    const I id = ids[p];
    if (is_expert(id, E)) atomicAdd(&lds[(int)id], 1);
  }
  __syncthreads();
  for (int i = tid; i < E; i += THREADS) counts[(int64_t)blockIdx.x * E + i] = lds[i];
}

// One block of 16 waves.  counts[c][e] -> exclusive position of chunk c's first row of expert e.
// A wave takes the experts e = wave, wave + 16, ...; its lanes take 64 chunks at a time (wave-wide scan, carry
// between the groups of 64), so the walk over the chunks of an expert is 64 wide instead of serial.
__global__ __launch_bounds__(1024) void route_scan_kernel(int* __restrict__ counts, int nchunk, int64_t L, int E,
                                                         int64_t* __restrict__ eid_out, int64_t* __restrict__ idx_out,
                                                         int64_t* __restrict__ off_out) {
  extern __shared__ int total[];  // [E]
  __shared__ int n_valid;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  // many experts, few chunks: an expert per thread, eight chunks' counters in flight (a wave per expert would walk
  // E / 16 experts one memory round trip after the other)
  const bool by_thread = E >= 64 && nchunk <= 64;
  auto over_chunks = [&](int e, auto use) {
    for (int c0 = 0; c0 < nchunk; c0 += 8) {
      int v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = c0 + u < nchunk ? counts[(int64_t)(c0 + u) * E + e] : 0;
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (c0 + u < nchunk) use(c0 + u, v[u]);
    }
  };
  if (by_thread) {
    for (int e = tid; e < E; e += 1024) {
      int run = 0;
      over_chunks(e, [&](int, int v) { run += v; });
      total[e] = run;
    }
  } else
  for (int e = w; e < E; e += 16) {
    int run = 0;
    for (int c0 = 0; c0 < nchunk; c0 += 64) {
      const int c = c0 + lane;
      const int v = c < nchunk ? counts[(int64_t)c * E + e] : 0;
      int incl = v;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        int u = __shfl_up(incl, d, 64);
        if (lane >= d) incl += u;
      }
      if (c < nchunk) counts[(int64_t)c * E + e] = run + incl - v;
      run += __shfl(incl, 63, 64);
    }
    if (lane == 0) total[e] = run;
  }
  __syncthreads();
  if (tid < 64) {
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + lane;
      const int c = e < E ? total[e] : 0;
      int incl = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        int v = __shfl_up(incl, d, 64);
        if (lane >= d) incl += v;
      }
      if (e < E) {
        total[e] = carry + incl - c;
        off_out[e] = (int64_t)(carry + incl);
      }
      carry += __shfl(incl, 63, 64);
    }
    if (lane == 0) n_valid = carry;
  }
  __syncthreads();
  fill_dropped((int64_t)n_valid + tid, 1024, L, E, eid_out, idx_out);
  if (by_thread) {
    for (int e = tid; e < E; e += 1024) {
      int run = total[e];
      over_chunks(e, [&](int c, int v) {
        counts[(int64_t)c * E + e] = run;
        run += v;
      });
    }
    return;
  }
  for (int64_t i = tid; i < (int64_t)nchunk * E; i += blockDim.x) counts[i] += total[i % E];
}

template <typename I, int THREADS>
__global__ __launch_bounds__(THREADS) void route_scatter_kernel(
    const I* __restrict__ ids, int64_t L, int E, const int* __restrict__ bases /*[nchunk][E]*/,
    int64_t* __restrict__ eid_out, int64_t* __restrict__ idx_out) {
  constexpr int W = THREADS / 64, SEG = kRouteChunk / W, IT = SEG / 64;
  extern __shared__ int lds[];  // [W][E]
  const int tid = threadIdx.x, w = tid >> 6;
  for (int i = tid; i < W * E; i += THREADS) lds[i] = 0;
  __syncthreads();
  const int64_t chunk_lo = (int64_t)blockIdx.x * kRouteChunk;
  const int64_t lo = min(chunk_lo + (int64_t)w * SEG, L), hi = min(lo + SEG, L);
  int key[IT], loc[IT];
  wave_rank<I, IT>(ids, lo, hi, E, bits_for(E), lds + w * E, key, loc);
  __syncthreads();
  for (int e = tid; e < E; e += THREADS) prefix_over_waves<W>(lds, E, e, bases[(int64_t)blockIdx.x * E + e]);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IT; ++u) {
    if (key[u] >= 0) {
      const int pos = lds[w * E + key[u]] + loc[u];
      eid_out[pos] = (int64_t)key[u];
      idx_out[pos] = lo + u * 64 + lane_id();
    }
  }
}

size_t route_workspace_bytes(int64_t L, int E) {
  if (L <= kRouteChunk || (L <= kRouteFusedMax && E <= kRouteFusedMaxE)) return 0;
  return (size_t)cdiv64(L, kRouteChunk) * (size_t)E * sizeof(int);
}

template <typename I>
static int launch_route_t(const I* ids, int64_t L, int E, int64_t* eid_out, int64_t* idx_out,
                          int64_t* off_out, void* ws, hipStream_t st) {
  auto fused = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(1), dim3(threads), 0, st, ids, (int)L, E, eid_out, idx_out, off_out);
    return launch_status("route_fused_kernel");
  };
  // 16 waves need 17 E ints of LDS; with more experts, and for a row per thread, 4 waves
  if (L <= kRouteThreads) return fused(&route_fused_kernel<I, kRouteThreads, 1>, kRouteThreads);
  if (L <= kRouteChunk && E <= kRouteFusedMaxE) return fused(&route_fused_kernel<I, 1024, 4>, 1024);
  if (L <= kRouteChunk) return fused(&route_fused_kernel<I, kRouteThreads, 16>, kRouteThreads);
  // one workgroup of 16 waves: a launch costs more than ranking 1024 rows per wave does
  if (L <= kRouteFusedMax / 2 && E <= kRouteFusedMaxE) return fused(&route_fused_kernel<I, 1024, 8>, 1024);
  if (L <= kRouteFusedMax && E <= kRouteFusedMaxE) return fused(&route_fused_kernel<I, 1024, 16>, 1024);
  const int nchunk = (int)cdiv64(L, kRouteChunk);
  int* counts = (int*)ws;
  hipLaunchKernelGGL((route_hist_kernel<I, 1024>), dim3(nchunk), dim3(1024), (size_t)E * sizeof(int), st, ids, L, E,
                     counts);
  hipLaunchKernelGGL(route_scan_kernel, dim3(1), dim3(1024), (size_t)E * sizeof(int), st, counts, nchunk, L,
                     E, eid_out, idx_out, off_out);
  auto scatter = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(nchunk), dim3(threads), (size_t)(threads / 64) * E * sizeof(int), st, ids, L, E,
                       (const int*)counts, eid_out, idx_out);
  };
  if (E <= kRouteFusedMaxE) scatter(&route_scatter_kernel<I, 1024>, 1024);
  else scatter(&route_scatter_kernel<I, kRouteThreads>, kRouteThreads);
  return launch_status("route_scatter_kernel");
}

// ---- routing without a caller workspace -----------------------------------------------------------------
// The per-chunk histograms of the three-launch path live in a fixed device array instead of caller memory, for
// callers that can neither allocate nor bring a workspace (code under stream capture, serving loops).  Each GPU
// holds its own copy of the array at its own address; `scratch_ptr` resolves and caches that address once per
// device.  The array keeps the previous call's contents; nothing has to start at zero, because the histogram
// launch writes every entry the later launches read.  Calls that overlap on one GPU share the array and race.
static __device__ __align__(256) unsigned char route_scratch[SMOE_ROUTE_STATIC_BYTES];

static constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mutex;

// Device address of this GPU's copy of `route_scratch` (the array's name is only a host-side handle).
static int scratch_ptr(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("smoe_route_static: cannot identify the current device (%s)", hipGetErrorString(e));
    return e != hipSuccess ? (int)e : SMOE_ERR_RANGE;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(route_scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("smoe_route_static: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
      return e != hipSuccess ? (int)e : SMOE_ERR_NULL;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

int route_static_init() {
  void* p = nullptr;
  return scratch_ptr(&p);
}

int launch_route(const void* ids, int idx_dtype, int64_t L, int E, int64_t* eid_out, int64_t* idx_out,
                 int64_t* off_out, void* ws, hipStream_t st);

int launch_route_static(const void* ids, int idx_dtype, int64_t L, int E, int64_t* eid_out, int64_t* idx_out,
                        int64_t* off_out, hipStream_t st) {
  if (E > kRouteMaxE) {          // before the buffer check: too many experts is a range error, not a workspace one
    set_error("smoe_route_static: E=%d exceeds the supported maximum %d", E, kRouteMaxE);
    return SMOE_ERR_RANGE;
  }
  const size_t need = route_workspace_bytes(L, E);
  if (need > (size_t)SMOE_ROUTE_STATIC_BYTES) {
    set_error("smoe_route_static: L=%lld rows over E=%d experts need %zu bytes of histograms, the built-in buffer "
              "holds %d (use smoe_route with a workspace)", (long long)L, E, need, SMOE_ROUTE_STATIC_BYTES);
    return SMOE_ERR_WORKSPACE;
  }
  void* ws = nullptr;
  if (need > 0) {
    if (const int rc = scratch_ptr(&ws)) return rc;
  }
  return launch_route(ids, idx_dtype, L, E, eid_out, idx_out, off_out, ws, st);
}

int launch_route(const void* ids, int idx_dtype, int64_t L, int E, int64_t* eid_out, int64_t* idx_out,
                 int64_t* off_out, void* ws, hipStream_t st) {
  if (E > kRouteMaxE) {
    set_error("smoe_route: E=%d exceeds the supported maximum %d", E, kRouteMaxE);
    return SMOE_ERR_RANGE;
  }
  switch (idx_dtype) {
    case SMOE_I64: return launch_route_t((const int64_t*)ids, L, E, eid_out, idx_out, off_out, ws, st);
    case SMOE_I32: return launch_route_t((const int32_t*)ids, L, E, eid_out, idx_out, off_out, ws, st);
    case SMOE_I16: return launch_route_t((const int16_t*)ids, L, E, eid_out, idx_out, off_out, ws, st);
    case SMOE_U8: return launch_route_t((const uint8_t*)ids, L, E, eid_out, idx_out, off_out, ws, st);
    default: set_error("smoe_route: unknown index dtype %d", idx_dtype); return SMOE_ERR_DTYPE;
  }
}

// off[e] = number of rows with id <= e, from an ascending id vector.  Boundary n (between rows n-1
// and n, with virtual ids -1 before the first row and E after the last) owns the experts in
// [eid[n-1], eid[n]) and writes n to each, so every off[e] is written exactly once.
__global__ __launch_bounds__(256) void offsets_from_sorted_kernel(const int64_t* __restrict__ eid, int64_t L,
                                                                 int E, int64_t* __restrict__ off) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (n > L) return;
  int64_t lo = n > 0 ? eid[n - 1] : 0;
  int64_t cur = n < L ? eid[n] : (int64_t)E;
  if (lo < 0) lo = 0;
  if (cur > E) cur = E;
  for (int64_t e = lo; e < cur; ++e) off[e] = n;
}

int launch_offsets_from_sorted(const int64_t* eid, int64_t L, int E, int64_t* off, hipStream_t st) {
  const int64_t n = L + 1;
  hipLaunchKernelGGL(offsets_from_sorted_kernel, dim3((unsigned)cdiv64(n, 256)), dim3(256), 0, st, eid, L, E, off);
  return launch_status("offsets_from_sorted_kernel");
}

}  // namespace smoe
