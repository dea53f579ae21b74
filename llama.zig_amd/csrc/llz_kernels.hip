// llz_kernels.hip -- MI355X (gfx950) kernels around the fused sampling kernel
// (llz_stats.h):
//   k_penalty     (optional) penalised copy of the rows   sampler.zig:54-75
//   k_math_probe  the device exp/log/expm1/tanh (parity tests)
//   k_argmax      greedy rows (temperature <= 0)          sampler.zig:31-41,50
#include <hip/hip_runtime.h>

#include <algorithm>

#include "llz_internal.h"
#include "llz_rowops.h"

namespace llz {

constexpr int kMaxNT = 256;        // threads of the k_penalty workgroups
constexpr int kMaxPerThread = 16;  // logits per thread in k_penalty

// ---------------------------------------------------------------------------
// k_penalty: penalised copy (sampler.zig:54-75) of the post-processed rows
// (main.zig:653-666), for windows longer than the fused penalty takes.
// Each index is penalised at most once even when it repeats in the window
// (the reference breaks out of the window scan at the first match).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kMaxNT) void k_penalty(const float* __restrict__ logits, int64_t stride,
                                                    int n, const uint32_t* __restrict__ prev,
                                                    int n_prev, int64_t prev_stride, int window,
                                                    float penalty, uint32_t xf, float cap, float inv_scale,
                                                    float* __restrict__ out) {
  const int row = blockIdx.y;
  const int seg0 = blockIdx.x * (kMaxNT * kMaxPerThread);
  const int seg1 = min(n, seg0 + kMaxNT * kMaxPerThread);
  const float* x = logits + (int64_t)row * stride;
  float* y = out + (int64_t)row * n;
  for (int i = seg0 + (int)threadIdx.x; i < seg1; i += kMaxNT) y[i] = logit_post(x[i], xf, cap, inv_scale);
  __syncthreads();
  const uint32_t* pv = prev + (int64_t)row * prev_stride;
  const int w = min(n_prev, window);
  const int start = n_prev - w;
  for (int a = start + (int)threadIdx.x; a < n_prev; a += kMaxNT) {
    const uint32_t tok = pv[a];
    if (tok >= (uint32_t)seg0 && tok < (uint32_t)seg1) {
      bool first = true;
      for (int b = start; b < a; ++b) first = first && (pv[b] != tok);
      if (first) {
        y[tok] = penalise(logit_post(x[tok], xf, cap, inv_scale), penalty);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// k_argmax: sampleArgmax (sampler.zig:31-41) of the post-processed rows, each
// row cut into `chunks` runs of consecutive logits, one workgroup each.
//
// The reference's scan keeps the first strict maximum; a NaN never wins,
// except at index 0, where it is never replaced.  That is the largest key
// under (value, lower index first) with NaN below everything and index 0's
// NaN above it, so chunks combine in any order.  They combine through the
// row's token word itself, with no scratch memory: a workgroup reads the
// word, and while its own best beats the element the word names it swaps its
// index in.  The word needs no initialisation: what an earlier call left
// there is either not an index of the row (any element beats it) or names a
// real element of it, which the row's best beats or equals.  (Token words in
// host memory take one chunk per row: stored, not exchanged over the bus.)
//
// Bound by HBM latency and launch: a workgroup per row with one 4-byte load
// in flight per thread took 19.8 us per call of 32 x 50021, back to back;
// chunks of at least kArgChunk logits over up to kArgGroups workgroups, four
// 16-byte loads in flight per thread, take 9.9 (the kernel alone under the
// profiler, which lengthens both: 21.3 and 10.6).
// ---------------------------------------------------------------------------
constexpr int kArgNT = 256;
constexpr int kArgUnroll = 4;                            // float4 loads in flight per thread
constexpr int kArgStep = kArgNT * 4 * kArgUnroll;        // logits per loop step of a workgroup
constexpr int kArgChunk = kArgStep;                      // logits per chunk at least
constexpr int kArgGroups = 1024;                         // workgroups aimed at (four per CU)

// The order of sampleArgmax as an unsigned key (larger wins).
__device__ __forceinline__ uint64_t amax_key(float v, uint32_t i) {
  const uint32_t b = __float_as_uint(v + 0.0f);  // -0 and +0 are one value
  const uint32_t o = b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
  const uint32_t k = v != v ? (i == 0u ? 0xffffffffu : 0u) : o;
  return ((uint64_t)k << 32) | (uint32_t)~i;
}

__global__ __launch_bounds__(kArgNT) void k_argmax(const float* __restrict__ logits, int64_t stride,
                                                   int n, int chunks, uint32_t per_chunk, uint32_t xf, float cap,
                                                   float inv_scale, uint32_t* __restrict__ tokens,
                                                   uint8_t* __restrict__ consumed, uint32_t* __restrict__ kept_count,
                                                   uint32_t* __restrict__ path) {
  __shared__ uint64_t best[kArgNT / kWave];
  const int row = (int)(blockIdx.x / (unsigned)chunks), c = (int)(blockIdx.x % (unsigned)chunks);
  const float* x = logits + (int64_t)row * stride;
  // chunks divide the row: p0 < n (positions unsigned: a step past a row of
  // nearly 2^31 logits stays above its end)
  const uint32_t p0 = (uint32_t)c * per_chunk, p1 = min((uint32_t)n, p0 + per_chunk);
  uint64_t bk = 0ull;  // below every element's key
  if (p1 - p0 >= 4) {
    // starts past the chunk's last four logits are moved back to them: an
    // element read twice changes no maximum, and no load needs a branch
    for (uint32_t base = p0; base < p1; base += kArgStep) {
      llz_f4u v[kArgUnroll];
      uint32_t pos[kArgUnroll];
#pragma unroll
      for (int u = 0; u < kArgUnroll; ++u) {
        pos[u] = min(base + ((uint32_t)u * kArgNT + threadIdx.x) * 4u, p1 - 4u);
        v[u] = *reinterpret_cast<const llz_f4u*>(x + pos[u]);
      }
#pragma unroll
      for (int u = 0; u < kArgUnroll; ++u)
#pragma unroll
        for (int k = 0; k < 4; ++k) bk = max(bk, amax_key(logit_post(v[u][k], xf, cap, inv_scale), pos[u] + (uint32_t)k));
    }
  } else {
    for (uint32_t i = p0 + threadIdx.x; i < p1; i += kArgNT)
      bk = max(bk, amax_key(logit_post(x[i], xf, cap, inv_scale), i));
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) bk = max(bk, (uint64_t)__shfl_xor((unsigned long long)bk, m, kWave));
  if (lane_id() == 0) best[wave_id()] = bk;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kArgNT / kWave; ++w) bk = max(bk, best[w]);
    const uint32_t mine = ~(uint32_t)bk;
    if (chunks == 1) {
      tokens[row] = mine;
    } else {
      uint32_t cur = __hip_atomic_load(&tokens[row], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // each failed exchange means another chunk's better or worse index
      // came in between: at most one per chunk
      while (cur >= (uint32_t)n || bk > amax_key(logit_post(x[cur], xf, cap, inv_scale), cur)) {
        if (__hip_atomic_compare_exchange_strong(&tokens[row], &cur, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
          break;
      }
    }
    if (c == 0) {
      if (consumed) consumed[row] = 0;
      if (kept_count) kept_count[row] = 0;
      if (path) path[row] = 0;
    }
  }
}

// ---------------------------------------------------------------------------
// k_math_probe: the device exp/log/expm1/tanh on an array (parity tests of
// the math).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_math_probe(const float* __restrict__ in, float* __restrict__ out_exp,
                                                   float* __restrict__ out_log, float* __restrict__ out_expm1,
                                                   float* __restrict__ out_tanh, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    const float x = in[i];
    if (out_exp) out_exp[i] = exp_f32(x);
    if (out_log) out_log[i] = log_f32(x);
    if (out_expm1) out_expm1[i] = expm1_f32(x);
    if (out_tanh) out_tanh[i] = tanh_f32(x);
  }
}

// ---------------------------------------------------------------------------
// k_hw_error: the largest relative error of the hardware exp2 (op 0), log2
// (op 1) or reciprocal (op 2) over a range of float bit patterns, against
// double precision, as error * 2^43 (units of 2^-23, times 2^20) folded into
// *max_err; op 3: the log2's error relative to max(1, |log2 x|).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_hw_error(int op, uint32_t first, uint32_t count,
                                                  uint32_t* __restrict__ max_err) {
  uint32_t worst = 0;
  const uint64_t step = (uint64_t)gridDim.x * 256u;
  for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < count; i += step) {
    const float x = __uint_as_float(first + (uint32_t)i);
    float r;
    double y;
    if (op == 0) {
      r = __builtin_amdgcn_exp2f(x);
      y = exp2((double)x);
    } else if (op == 1 || op == 3) {
      r = __builtin_amdgcn_logf(x);
      y = log2((double)x);
    } else {
      r = __builtin_amdgcn_rcpf(x);
      y = 1.0 / (double)x;
    }
    const double q = fabs((double)r - y) / (op == 3 ? fmax(1.0, fabs(y)) : fabs(y)) * 0x1p43;
    worst = max(worst, q < 4.0e9 ? (uint32_t)q : 0xffffffffu);  // NaN -> saturated
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) worst = max(worst, (uint32_t)__shfl_xor((int)worst, m, kWave));
  if (lane_id() == 0) atomicMax(max_err, worst);
}

// ---------------------------------------------------------------------------
// k_stage: pinned host memory to device memory, 16 bytes per thread.  On the
// compute queue, so that the sampling kernel behind it needs no signal from
// a copy engine.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_stage(uint4* __restrict__ dst, const uint4* __restrict__ src, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_stage(void* dst, const void* pinned, size_t units16, hipStream_t st) {
  if (units16 == 0) return hipSuccess;
  hipLaunchKernelGGL(k_stage, dim3((unsigned)((units16 + 255) / 256)), dim3(256), 0, st, (uint4*)dst,
                     (const uint4*)pinned, (uint32_t)units16);
  return hipGetLastError();
}

__global__ void k_zero_u32(uint32_t* p) { *p = 0u; }

hipError_t launch_hw_error(int op, uint32_t first, uint32_t count, uint32_t* max_err, hipStream_t st) {
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, st, max_err);
  const uint64_t blocks = std::min<uint64_t>(4096, ((uint64_t)count + 255) / 256);
  hipLaunchKernelGGL(k_hw_error, dim3((unsigned)blocks), dim3(256), 0, st, op, first, count, max_err);
  return hipGetLastError();
}

hipError_t launch_math_probe(const float* in, float* out_exp, float* out_log, float* out_expm1, float* out_tanh,
                             int64_t n, hipStream_t st) {
  const int64_t blocks = (n + 255) / 256;
  hipLaunchKernelGGL(k_math_probe, dim3((unsigned)blocks), dim3(256), 0, st, in, out_exp, out_log, out_expm1,
                     out_tanh, n);
  return hipGetLastError();
}

hipError_t launch_penalty(const float* logits, int64_t stride, int rows, int n, const uint32_t* prev,
                          int n_prev, int64_t prev_stride, int window, float penalty, uint32_t xf, float cap,
                          float inv_scale, float* out, hipStream_t st) {
  dim3 grid((n + kMaxNT * kMaxPerThread - 1) / (kMaxNT * kMaxPerThread), rows);
  hipLaunchKernelGGL(k_penalty, grid, dim3(kMaxNT), 0, st, logits, stride, n, prev, n_prev,
                     prev_stride, window, penalty, xf, cap, inv_scale, out);
  return hipGetLastError();
}

// chunks per row: as many as fill kArgGroups workgroups, none below kArgChunk
// logits but the last, and none empty
static uint32_t argmax_per_chunk(int n, int chunks) {
  return (((uint32_t)n + (uint32_t)chunks - 1) / (uint32_t)chunks + 3u) & ~3u;
}

int argmax_chunks(int rows, int n) {
  const uint32_t un = (uint32_t)n;
  const uint32_t most = (un + kArgChunk - 1) / kArgChunk;
  const uint32_t want = std::min(most, (uint32_t)std::max(1, kArgGroups / rows));
  const uint32_t per = argmax_per_chunk(n, (int)want);
  return (int)((un + per - 1) / per);
}

hipError_t launch_argmax(const float* logits, int64_t stride, int rows, int n, int chunks, uint32_t xf, float cap,
                         float inv_scale, uint32_t* tokens, uint8_t* consumed, uint32_t* kept_count,
                         uint32_t* path, hipStream_t st) {
  hipLaunchKernelGGL(k_argmax, dim3((unsigned)rows * (unsigned)chunks), dim3(kArgNT), 0, st, logits, stride, n, chunks,
                     argmax_per_chunk(n, chunks), xf, cap, inv_scale, tokens, consumed, kept_count, path);
  return hipGetLastError();
}


}  // namespace llz
