// llz_stats_inst.hip -- the instantiations of the sampling kernels
// (llz_stats.h), one group per object (LLZ_INST), so that they build in
// parallel:
//   0-4  k_stats / k_stats_rows: plain, plain with typical-p, light, light
//        with typical-p, soft-capped (a: 16-byte aligned rows; b: claimed rows)
//   5, 6 k_split on plain rows: 16-byte aligned, any (a: float4 per thread)
//   7, 8 k_split on transformed rows, the same (a: float4 per thread; b: soft-capped)
//   9    k_long (a: 16-byte aligned rows; b: transform mode)
//   10   k_tok (a: 16-byte aligned rows; b: transform mode, not soft-capped)
#include "llz_long.h"
#include "llz_stats.h"

#ifndef LLZ_INST
#error "LLZ_INST selects the group of kernels"
#endif
#define LLZ_CAT2(a, b) a##b
#define LLZ_CAT(a, b) LLZ_CAT2(a, b)

namespace llz {

StatsKernel LLZ_CAT(stats_kernel_, LLZ_INST)(int a, int b) {
#if LLZ_INST <= 4
  constexpr int XM = LLZ_INST <= 1 ? kXmNone : LLZ_INST <= 3 ? kXmLight : kXmCap;
  constexpr bool EXT = LLZ_INST == 1 || LLZ_INST == 3;
  if (b != 0) return a != 0 ? k_stats_rows<true, XM, EXT> : k_stats_rows<false, XM, EXT>;
  return a != 0 ? k_stats<true, XM, EXT> : k_stats<false, XM, EXT>;
#elif LLZ_INST <= 6
  constexpr bool F = LLZ_INST == 5;
  (void)b;
  return a == 1 ? k_split<1, kXmNone, F> : a == 2 ? k_split<2, kXmNone, F> : a == 4 ? k_split<4, kXmNone, F>
                                       : a == 8 ? k_split<8, kXmNone, F> : nullptr;
#elif LLZ_INST == 10
  if (b == kXmLight) return a != 0 ? k_tok<true, kXmLight> : k_tok<false, kXmLight>;
  return a != 0 ? k_tok<true, kXmNone> : k_tok<false, kXmNone>;
#elif LLZ_INST == 9
  if (b == kXmCap) return a != 0 ? k_long<true, kXmCap> : k_long<false, kXmCap>;
  if (b == kXmLight) return a != 0 ? k_long<true, kXmLight> : k_long<false, kXmLight>;
  return a != 0 ? k_long<true, kXmNone> : k_long<false, kXmNone>;
#else
  constexpr bool F = LLZ_INST == 7;
  if (b != 0) return a == 1 ? k_split<1, kXmCap, F> : k_split<2, kXmCap, F>;
  return a == 1 ? k_split<1, kXmLight, F> : k_split<2, kXmLight, F>;
#endif
}

}  // namespace llz

#ifdef LLZ_PHASE_STAMPS
// Measurement builds: this object's phase timestamps (each object has its
// own copy of the array; a call's rows are all in one, but for k_tok's pass
// over rows that another object then samples).
extern "C" int LLZ_CAT(llz_stamps_, LLZ_INST)(unsigned long long* dst, int rows, int clear) {
  const size_t bytes = (size_t)rows * llz::kStampSlots * sizeof(unsigned long long);
  if (clear) {
    static unsigned long long zeros[llz::kStampRows * llz::kStampSlots];
    return hipMemcpyToSymbol(HIP_SYMBOL(llz::llz_phase_stamps), zeros, sizeof(zeros)) == hipSuccess ? 0 : -3;
  }
  return hipMemcpyFromSymbol(dst, HIP_SYMBOL(llz::llz_phase_stamps), bytes) == hipSuccess ? 0 : -3;
}
#endif
