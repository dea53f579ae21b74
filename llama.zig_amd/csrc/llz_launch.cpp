// llz_launch.cpp -- one kernel launch per llz_sample_rows call: which of the
// sampling kernels (llz_stats_inst.hip) runs, and on what grid.
#include <hip/hip_runtime.h>

#include "llz_internal.h"

namespace llz {

StatsKernel stats_kernel_0(int, int);
StatsKernel stats_kernel_1(int, int);
StatsKernel stats_kernel_2(int, int);
StatsKernel stats_kernel_3(int, int);
StatsKernel stats_kernel_4(int, int);
StatsKernel stats_kernel_5(int, int);
StatsKernel stats_kernel_6(int, int);
StatsKernel stats_kernel_7(int, int);
StatsKernel stats_kernel_8(int, int);
StatsKernel stats_kernel_9(int, int);
StatsKernel stats_kernel_10(int, int);

// Every row's statistics, then its selection.
hipError_t launch_sample(const RowParams& P, const RowPtrs& Q, hipEvent_t ev_begin, hipEvent_t ev_end,
                         hipStream_t st) {
  if (ev_begin && hipEventRecord(ev_begin, st) != hipSuccess) return hipErrorUnknown;
  const bool fastld = (P.flags & kFlagVecSrc) != 0 && (P.n % 4) == 0;
  // the transform mode: soft-capping (the chain's input) takes the
  // estimating single pass, the scale and the penalty alone the exact one
  const int xm = (P.xf_src & kXfCap) ? kXmCap : ((P.xf_src | P.xf_orig) != 0u ? kXmLight : kXmNone);
  const KArgs A{P, Q};
  // more rows than workgroups: the grid's workgroups claim rows (the
  // special-queue overflow area has one block per workgroup of the grid)
  const bool claim = P.grid < P.rows;
  // transformed rows split with chunks of at most 2 float4 per thread (each
  // logit's exact post-processing is then a few per thread)
  const bool split = P.split_s >= 2 && P.rows <= kSplitRows && (xm == kXmNone || P.split_nv <= 2);
  // token-only calls with typical-p (not soft-capped) take the instantiation
  // that carries typical-p's decisions and the list's second collection
  // round; the others keep the shorter code
  const bool ext = (P.flags & kFlagTokenOnly) != 0u && P.typical_p > 0.0f && P.typical_p < 1.0f && xm != kXmCap;
  StatsKernel kern = nullptr;
  if (split)
    kern = xm == kXmNone ? (fastld ? stats_kernel_5(P.split_nv, 0) : stats_kernel_6(P.split_nv, 0))
                         : (fastld ? stats_kernel_7 : stats_kernel_8)(P.split_nv, xm == kXmCap);
  else if (P.flags & kFlagLong)
    kern = stats_kernel_9(fastld, xm);
  else if (xm == kXmCap)
    kern = stats_kernel_4(fastld, claim);
  else if (xm == kXmLight)
    kern = ext ? stats_kernel_3(fastld, claim) : stats_kernel_2(fastld, claim);
  else
    kern = ext ? stats_kernel_1(fastld, claim) : stats_kernel_0(fastld, claim);
  if (!kern) return hipErrorInvalidValue;
  const dim3 grid(split ? P.rows * P.split_s : (claim ? P.grid : P.rows)), block(kStatsNT);
  void* args[] = {const_cast<KArgs*>(&A)};
  if (Q.und) {  // the token-only pass over every row first; kern then takes the rows it marked
    const dim3 tg(P.rows < 3 * P.grid ? P.rows : 3 * P.grid);
    if (hipLaunchKernel((const void*)stats_kernel_10(fastld, xm), tg, block, args, 0, st) != hipSuccess)
      return hipErrorLaunchFailure;
  }
  if (hipLaunchKernel((const void*)kern, grid, block, args, 0, st) != hipSuccess) return hipErrorLaunchFailure;
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (ev_end && hipEventRecord(ev_end, st) != hipSuccess) return hipErrorUnknown;
  return hipSuccess;
}

}  // namespace llz

#ifdef LLZ_PHASE_STAMPS
extern "C" int llz_stamps_0(unsigned long long*, int, int);
extern "C" int llz_stamps_1(unsigned long long*, int, int);
extern "C" int llz_stamps_2(unsigned long long*, int, int);
extern "C" int llz_stamps_3(unsigned long long*, int, int);
extern "C" int llz_stamps_4(unsigned long long*, int, int);
extern "C" int llz_stamps_5(unsigned long long*, int, int);
extern "C" int llz_stamps_6(unsigned long long*, int, int);
extern "C" int llz_stamps_7(unsigned long long*, int, int);
extern "C" int llz_stamps_8(unsigned long long*, int, int);
extern "C" int llz_stamps_9(unsigned long long*, int, int);
extern "C" int llz_stamps_10(unsigned long long*, int, int);

// Measurement builds: the phase timestamps of rows 0 .. rows - 1 (kStampSlots
// per row, 0 where a row did not reach the boundary) into dst.  A row that
// k_tok (the last object) left to k_stats_rows has the latter's.
extern "C" int llz_debug_phase_stamps(unsigned long long* dst, int rows, int clear) {
  if (rows <= 0 || rows > llz::kStampRows || !dst) return -1;
  static int (*const get[])(unsigned long long*, int, int) = {llz_stamps_0, llz_stamps_1, llz_stamps_2, llz_stamps_3,
                                                              llz_stamps_4, llz_stamps_5, llz_stamps_6, llz_stamps_7,
                                                              llz_stamps_8, llz_stamps_9, llz_stamps_10};
  static unsigned long long part[llz::kStampRows * llz::kStampSlots];
  const size_t n = (size_t)rows * llz::kStampSlots;
  if (!clear)
    for (size_t i = 0; i < n; ++i) dst[i] = 0;
  for (auto f : get) {
    const int rc = f(part, rows, clear);
    if (rc != 0) return rc;
    if (clear) continue;
    for (int r = 0; r < rows; ++r) {
      unsigned long long* to = dst + (size_t)r * llz::kStampSlots;
      if (f == llz_stamps_10 && to[0] != 0) continue;
      for (int k = 0; k < llz::kStampSlots; ++k) to[k] |= part[(size_t)r * llz::kStampSlots + k];  // (one other object ran it)
    }
  }
  return 0;
}
#endif
