// llz_rowops.h -- per-row helpers shared by the kernels: workgroup maximum,
// sampleArgmax over a row, vector loads and the reference's term.
#pragma once

#include <hip/hip_runtime.h>

#include "llz_internal.h"
#include "llz_math.h"
#include "llz_norm.h"
#include "llz_wg.h"
#include "llz_xform.h"

namespace llz {

constexpr int kNT = 512;           // threads of the per-row workgroup
constexpr int kV = kLaneV;         // logits per thread per streaming tile
constexpr int kTile = kNT * kV;    // 4096 logits per tile
constexpr int kCap = kCandCap;     // candidate list capacity (power of two)
constexpr float kInf = __builtin_inff();

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ float wave_fmax(float v) {
  const uint32_t r = wave_incl_scan_op(__float_as_uint(v), __float_as_uint(-kInf), [](uint32_t a, uint32_t b) {
    return __float_as_uint(fmaxf(__uint_as_float(a), __uint_as_float(b)));
  });
  return __uint_as_float(lane_readlast(r));
}

template <int NT>
__device__ __forceinline__ float wg_fmax(float v, WgScratch<NT>& sh, int& bank) {
  v = wave_fmax(v);
  if (lane_id() == 0) sh.red[bank][wave_id()] = __float_as_uint(v);
  lds_barrier();
  float r = __uint_as_float(sh.red[bank][0]);
#pragma unroll
  for (int w = 1; w < WgScratch<NT>::W; ++w) r = fmaxf(r, __uint_as_float(sh.red[bank][w]));
  bank ^= 1;
  return r;
}

// (value, index) ordering of sampleArgmax (sampler.zig:31-41): larger value
// wins, equal values keep the lower index, NaN never wins.
__device__ __forceinline__ bool amax_better(float v, uint32_t i, float bv, uint32_t bi) {
  if (v != v) return false;
  if (bv != bv) return true;
  return v > bv || (v == bv && i < bi);
}

// sampleArgmax over one row with the whole workgroup.  A NaN at index 0
// is never replaced by the reference's loop, so the answer is then 0.
template <int NT, class Src>
__device__ uint32_t wg_argmax_row(const Src& x, int n, WgScratch<NT>& sh, int& bank) {
  const int t = (int)threadIdx.x;
  float bv = __builtin_nanf("");
  uint32_t bi = 0xffffffffu;
  for (int i = t; i < n; i += NT) {
    const float v = x.at(i);
    if (amax_better(v, (uint32_t)i, bv, bi)) { bv = v; bi = (uint32_t)i; }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const float ov = __shfl_xor(bv, m, kWave);
    const uint32_t oi = __shfl_xor(bi, m, kWave);
    if (amax_better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
  }
  if (lane_id() == 0) {
    sh.red[bank][wave_id()] = bi;
    sh.red[bank ^ 1][wave_id()] = __float_as_uint(bv);
  }
  lds_barrier();
  float rv = __builtin_nanf("");
  uint32_t ri = 0xffffffffu;
  for (int w = 0; w < WgScratch<NT>::W; ++w) {
    const float v = __uint_as_float(sh.red[bank ^ 1][w]);
    const uint32_t i = sh.red[bank][w];
    if (amax_better(v, i, rv, ri)) { rv = v; ri = i; }
  }
  lds_barrier();  // both banks were used
  const float x0 = x.at(0);
  if (x0 != x0 || ri == 0xffffffffu) ri = 0;
  return ri;
}

// Four logits from position pos of a row of any length and alignment,
// without a branch per lane (so that every load of a wave can be in flight at
// once): a start within the row's last three positions reads the row's last
// four and shifts them; positions >= n are -inf.
__device__ __forceinline__ float4 rd4_any(const float* xr, int pos, int n) {
  float4 v;
  if (n < 4) {
    v.x = pos + 0 < n ? xr[pos + 0] : -kInf;
    v.y = pos + 1 < n ? xr[pos + 1] : -kInf;
    v.z = pos + 2 < n ? xr[pos + 2] : -kInf;
    v.w = pos + 3 < n ? xr[pos + 3] : -kInf;
    return v;
  }
  const int pc = min(pos, n - 4), off = pos - pc;
  const llz_f4u r = __builtin_nontemporal_load(reinterpret_cast<const llz_f4u*>(xr + pc));
  v.x = off == 0 ? r.x : (off == 1 ? r.y : (off == 2 ? r.z : (off == 3 ? r.w : -kInf)));
  v.y = off == 0 ? r.y : (off == 1 ? r.z : (off == 2 ? r.w : -kInf));
  v.z = off == 0 ? r.z : (off == 1 ? r.w : -kInf);
  v.w = off == 0 ? r.w : -kInf;
  return v;
}

// The next row beyond the grid for a workgroup that finished one: a counter
// word tagged with the low 40 bits of the call's epoch (a word left by
// another call, or not yet written, counts as 0 for this one).  Returns grid +
// the count before the claim (>= rows: nothing left).  The first claim of a
// call installs its tag (compare-and-swap); every later one is a single
// fetch-and-add, which the device serves back to back, where a
// compare-and-swap loop lets one claim through per round trip to memory
// (with rows of some 40 us, the workgroups then queued for their claims).
// The count stays below 2^24.  A launch makes exactly `rows` claims (rows -
// grid rows are taken, and each of the grid's workgroups is told once that
// none is left): the last one clears the word, so that a captured launch, whose
// replays carry one epoch, finds it free each time.
[[maybe_unused]] static __device__ __noinline__ int claim_row(unsigned long long* word, unsigned long long epoch, int grid, int rows) {
  constexpr unsigned long long kCnt = (1ull << 24) - 1;
  const unsigned long long tag = (epoch & ((1ull << 40) - 1)) << 24;
  unsigned long long old = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    if ((old & ~kCnt) == tag) {
      const unsigned long long prev = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((int)(prev & kCnt) == rows - 1) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return grid + (int)(prev & kCnt);
    }
    unsigned long long expected = old;
    if (__hip_atomic_compare_exchange_strong(word, &expected, tag | 1ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return grid;
    old = expected;
  }
}

// e_i = exp((v_i - max) / T) as sampler.zig:85 evaluates it.
__device__ __forceinline__ float row_exp(float v, float m, float T, bool t_is_one) {
  float x = v - m;
  if (!t_is_one) x = x / T;  // x / 1.0f == x exactly, so the divide is skipped
  return exp_f32(x);
}

}  // namespace llz
