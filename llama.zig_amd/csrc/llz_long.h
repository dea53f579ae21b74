// llz_long.h -- rows beyond the single pass's residency (129024 logits, up to
// kLongMax): k_long, one workgroup per row.
//
// k_stats keeps a row's estimates in registers and LDS; a longer row does
// not fit, and its streaming normaliser (llz_norm.h) reads the row twice
// after a scan for the maximum, with two barriers per 8192 logits: 256 us for a
// 151936-logit row, also where the call asks for the token alone.  Here the
// row is streamed once, a window of U segment loads in flight per wave:
// per 256-logit segment the running maximum and the sum of the estimates q =
// exp2(v l2e - c_w) (phase L of k_stats), and, on token-only calls, the
// elements that may be candidates.  Those are pushed as they pass: an element
// whose term may reach tok_theta against the row's maximum reaches it
// against any smaller one, so the test against a running maximum (the
// largest the workgroup's waves have published) collects a superset; a full
// buffer is filtered again against the maximum reached.  token_select then decides the
// row as on k_stats's token path (s_est and w_est from the segment sums).
// A row it does not decide, and every row of the other calls, goes on to the
// selection stage with the maximum known.
//
// 64 rows of 151936 logits with top-k, top-p and min-p: 303 us before, 35 us
// now.  Bound by one CU's share of HBM while
// the rows are fewer than the CUs.
//
// Batches of more rows than CUs (token-only calls that the rule in
// llz_api.cpp picks) run the same stream in k_tok first: without the residency
// and the selection stage a workgroup needs 45 KB of LDS and 97 to 105 VGPRs,
// so two share a CU (three where the registers allow) and one row's tail
// (re-reads, sort, decisions: 20 us behind 18 us of loads in k_stats_rows)
// runs under the others' loads.  Rows it does not decide are listed, and
// sampled by a k_stats_rows launch behind it.
// 4096 rows of 128256 with every filter: 705 us in k_stats_rows alone, 494 with
// k_tok (4.2 TB/s; it takes 418 of them in the kernel trace, 5.0 TB/s, and the
// rest is one listed row's exact phases).
#pragma once

#include "llz_fast.h"
#include "llz_select.h"
#include "llz_token.h"

namespace llz {

constexpr int kLongBuf = 512;    // candidate buffer entries per wave

struct LongShared {
  uint64_t tl[2 * kTokCap];                      // collected, then sorted
  uint8_t part[(kNT / kWave) * kTokCap];         // token_sort's partial ranks
  float bv[kNT / kWave][kLongBuf];               // per wave: candidates' logits
  uint32_t bp[kNT / kWave][kLongBuf];            //   and positions
  float mw[kNT / kWave], cw[kNT / kWave], qs[kNT / kWave], qw[kNT / kWave];
  uint32_t cnt[2][kNT / kWave];                  // per wave: buffered candidates above a threshold
  uint32_t tcand, tfail;
};

union LongLds {
  LongShared lng;
  SampleShared select;
};

// One row through the stream and, on token-only calls, token_select; true when
// the row is finished.  m_out: its maximum; nan_out: a NaN logit was seen.
// LEAN (k_tok): a row whose candidates flood a buffer is given up at once (no
// maximum then).  U: segment loads in flight per wave.
template <bool FASTLD, int XM, int U, bool LEAN, class Src>
__device__ __forceinline__ bool tok_stream(const RowParams& P, const RowPtrs& Q, int row, LongShared& F, PenShared& pen_sh,
                                           const Src& X, float& m_out, bool& nan_out) {
  constexpr int W = kNT / kWave, SEG = fastp::SEG;
  constexpr bool XF = XM != kXmNone;
  LLZ_STAMP(row, 0);
  const int t = (int)threadIdx.x, lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const int n = P.n;
  const bool t1 = (P.flags & kFlagTIsOne) != 0u;
  const float T = P.temperature, l2e = P.l2e_t;
  const float* xr = Q.src + (int64_t)row * P.src_stride;
  const float u_row = Q.uniforms[row];
  if constexpr (XF) {
    if (P.xf_src & kXfPen) {  // each id < n penalised once (sampler.zig:62-70)
      const uint32_t id = pen_window_id(P, Q, row);
      bool first = id < (uint32_t)n;
      for (int j = 0; j < P.pen_w; ++j) {
        const uint32_t o = readlane_u32(id, j);
        first = first && !(j < lane && o == id);
      }
      pen_list(pen_sh, first ? id : (id | 0x80000000u));
    }
  }
  if (t == 0) {
    F.tcand = 0u;
    F.tfail = 0u;
  }
  if (t < W) F.mw[t] = -kInf;
  lds_barrier();

  const int G = (n + SEG - 1) / SEG;
  const int nseg = max(0, (G - w + W - 1) / W);  // wave w: segments w, w + W, ...
  const bool tok = (P.flags & kFlagTokenOnly) != 0u && P.tok_theta > 0.0f && l2e > 0.0f && l2e <= 0x1p40f;
  // an element passes while v >= mx - dv: its term may reach tok_theta
  // against the maximum mx seen so far (2^-8 octaves to spare for the
  // roundings here and of the reference's argument)
  const float dv = tok ? (-__builtin_amdgcn_logf(P.tok_theta) + 0x1p-8f) / l2e * (1.0f + 0x1p-20f) : 0.0f;
  // (nothing passes before a finite logit was seen)
  auto uni_max = [](float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); };
  auto thr_of = [&](float x) { return x > -kInf ? x - dv - fabsf(x) * 0x1p-22f : kInf; };
  float mx = -kInf, cw = 0.0f, thr = kInf;
  float qsum = 0.0f, qwsum = 0.0f;  // lane 63: the wave's sum of estimates, and weighted by n - the segment's start
  int nb = 0;                       // the wave's buffered candidates
  bool ovf = false;
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
  auto load = [&](int k) -> float4 {
    const int pos = (w + W * k) * SEG + lane * 4;
    if constexpr (FASTLD) {
      const float4 v = ld_nt4(xr + (k < nseg && pos < n ? pos : 0));
      return k < nseg && pos < n ? v : make_float4(-kInf, -kInf, -kInf, -kInf);
    } else {
      return rd4_any(xr, k < nseg ? pos : n, n);
    }
  };
  // drop the buffered elements below the threshold reached
  auto compact = [&]() {
    int o = 0;
    for (int b = 0; b < nb; b += kWave) {
      const int i = b + lane;
      const float v = i < nb ? F.bv[w][i] : -kInf;
      const uint32_t p = i < nb ? F.bp[w][i] : 0u;
      const bool keep = i < nb && v >= thr;
      const uint64_t km = bal64(keep);
      __builtin_amdgcn_wave_barrier();
      if (keep) {
        const int s = o + (int)__popcll(km & lt);  // s <= i: never past what is still to be read
        F.bv[w][s] = v;
        F.bp[w][s] = p;
      }
      o += (int)__popcll(km);
      __builtin_amdgcn_wave_barrier();
    }
    nb = o;
  };
  float4 cur[U], nxt[U];
#pragma unroll
  for (int u = 0; u < U; ++u) cur[u] = load(u);
  for (int k0 = 0; k0 < nseg; k0 += U) {
    if (LEAN && __builtin_amdgcn_readfirstlane((int)*(volatile uint32_t*)&F.tfail) != 0) break;
#pragma unroll
    for (int u = 0; u < U; ++u) nxt[u] = load(k0 + U + u);
    if constexpr (XF) {
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = X.fix4((w + W * (k0 + u)) * SEG + lane * 4, cur[u], k0 + u < nseg ? n : 0);
    }
    float ml = -kInf;
#pragma unroll
    for (int u = 0; u < U; ++u)  // fmaxf skips NaN (sampler.zig:80-81)
      ml = fmaxf(ml, fmaxf(fmaxf(cur[u].x, cur[u].y), fmaxf(cur[u].z, cur[u].w)));
    ml = wave_max_f32(ml);
    mx = fmaxf(mx, ml);
    // a finite offset whatever the maximum: an infinite one would make the
    // estimates of -inf logits and absent positions NaN (a maximum whose
    // product overflows fails the |awi| test below)
    if (k0 == 0) cw = fabsf(mx * l2e) <= 3.0e38f ? mx * l2e : 0.0f;
    // the threshold against the largest maximum any wave has published (no
    // barrier: an older one only lets more pass)
    if (lane == 0) F.mw[w] = mx;
    float ms = F.mw[lane & (W - 1)];
    ms = fmaxf(ms, __shfl_xor(ms, 1, kWave));
    ms = fmaxf(ms, __shfl_xor(ms, 2, kWave));
    ms = fmaxf(ms, __shfl_xor(ms, 4, kWave));
    thr = thr_of(fmaxf(mx, uni_max(ms)));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int seg0 = (w + W * (k0 + u)) * SEG;
      const float4 v = cur[u];
      const float q0 = __builtin_amdgcn_exp2f(fmaf(v.x, l2e, -cw)), q1 = __builtin_amdgcn_exp2f(fmaf(v.y, l2e, -cw));
      const float q2 = __builtin_amdgcn_exp2f(fmaf(v.z, l2e, -cw)), q3 = __builtin_amdgcn_exp2f(fmaf(v.w, l2e, -cw));
      const float a = wave_fold_f32((q0 + q1) + (q2 + q3));
      qsum += a;
      qwsum += a * (float)(n - min(seg0, n));
      if (tok && !ovf) {  // (a row whose candidates flood the buffer is not decided here)
        const bool hit = fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)) >= thr;
        if (bal64(hit) != 0ull) {
          const float vs[4] = {v.x, v.y, v.z, v.w};
          uint64_t im[4];
          int nh = 0;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            im[c] = bal64(vs[c] >= thr);
            nh += (int)__popcll(im[c]);
          }
          if (nb + nh > kLongBuf) {
            compact();
            ovf = nb + nh > kLongBuf;
            if (ovf) {
              nb = 0;
              if (LEAN && lane == 0) F.tfail = 1u;
            }
          }
          if (!ovf) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              if ((im[c] >> lane) & 1ull) {
                const int s = nb + (int)__popcll(im[c] & lt);
                F.bv[w][s] = vs[c];
                F.bp[w][s] = (uint32_t)(seg0 + lane * 4 + c);
              }
              nb += (int)__popcll(im[c]);
            }
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) cur[u] = nxt[u];
  }
  if (lane == kWave - 1) {
    F.qs[w] = qsum;
    F.qw[w] = qwsum;
  }
  if (lane == 0) {
    F.mw[w] = mx;
    F.cw[w] = cw;
    if (ovf) F.tfail = 1u;
  }
  lds_barrier();
  LLZ_STAMP(row, 1);
  float m = -kInf, s_est = 0.0f, w_est = 0.0f;
  bool bad = false, nanrow = false;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    m = fmaxf(m, F.mw[i]);
    // only a NaN logit makes an estimate NaN (l2e > 0, the offset finite), and
    // q >= 0 otherwise, so no inf - inf
    nanrow = nanrow || F.qs[i] != F.qs[i];
  }
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const float awi = fmaf(m, -l2e, F.cw[i]);
    const float ri = __builtin_amdgcn_exp2f(awi);
    bad = bad || (G > i && !(fabsf(awi) <= 64.0f));
    s_est += G > i ? F.qs[i] * ri : 0.0f;
    w_est += G > i ? F.qw[i] * ri : 0.0f;
  }
  m_out = m;
  nan_out = nanrow;
  // (a NaN logit or an infinite maximum makes the reference's sum NaN: the
  // selection stage handles that row)
  if (tok && !bad && !nanrow && fabsf(m) <= 3.0e38f && F.tfail == 0u) {
    float theta = P.tok_theta;
    thr = thr_of(m);
    // the buffered candidates at or above x, over the waves (one barrier: the
    // counts alternate between two rows)
    int bank = 0;
    auto count_at = [&](float x) -> int {
      int c = 0;
      for (int b = 0; b < nb; b += kWave) c += (int)__popcll(bal64(b + lane < nb && F.bv[w][b + lane] >= x));
      if (lane == 0) F.cnt[bank][w] = (uint32_t)c;
      lds_barrier();
      int s = 0;
#pragma unroll
      for (int i = 0; i < W; ++i) s += (int)F.cnt[bank][i];
      bank ^= 1;
      return s;
    };
    // More candidates than the list holds: under a top-k of at most kTokCap /
    // 4 a higher threshold on the logits is searched whose elements fit and
    // hold more than top-k of the row.  Every element left out has v < x, so
    // its term is at most e(x) (1 + 2^-21) (the argument is monotone in v and
    // exp within an ulp), which takes tok_theta's place.
    const uint32_t kk = P.top_k;
    if (kk >= 1u && kk <= (uint32_t)(kTokCap / 4) && kk < (uint32_t)n && count_at(thr) > kTokCap) {
      float lo = thr, hi = m;
      for (int it = 0; it < 16; ++it) {
        const float mid = lo + 0.5f * (hi - lo);
        const int c = count_at(mid);
        if (c > kTokCap) {
          lo = mid;
        } else if (c <= (int)kk) {
          hi = mid;
        } else {
          thr = mid;
          theta = fmaxf(theta, exact_term(mid, m, T, t1) * (1.0f + 0x1p-21f));
          break;
        }
      }
    }
    for (int b = 0; b < nb; b += kWave) {
      const int i = b + lane;
      const float v = i < nb ? F.bv[w][i] : -kInf;
      const bool live = i < nb && v >= thr;
      if (bal64(live) == 0ull) continue;
      const float e = live ? exact_term(v, m, T, t1) : 0.0f;  // sampler.zig:85
      const bool cand = live && e >= theta;
      const uint64_t cb = bal64(cand);
      if (cb != 0ull) {
        uint32_t b0 = 0u;
        if (lane == 0) b0 = atomicAdd(&F.tcand, (uint32_t)__popcll(cb));
        const uint32_t s = readlane_u32(b0, 0) + (uint32_t)__popcll(cb & lt);
        if (cand && s < (uint32_t)kTokCap) F.tl[s] = ((uint64_t)(~__float_as_uint(e)) << 32) | F.bp[w][i];
      }
    }
    lds_barrier();
    LLZ_STAMP(row, 33);
    const int tc = (int)F.tcand;
    if (tc <= kTokCap) {
      token_sort(F.tl, F.tl + kTokCap, F.part, tc);
      LLZ_STAMP(row, 34);
      if (w == 0) {
        // typical-p: decided where it drops nothing or nothing is kept
        // before it (no interval of the entropy here)
        if (P.typical_p > 0.0f && P.typical_p < 1.0f)
          token_select<true>(kernel_args_ptr(), row, F.tl + kTokCap, tc, s_est, w_est, 0.0, -1.0, u_row, theta, &F.tfail);
        else
          token_select<false>(kernel_args_ptr(), row, F.tl + kTokCap, tc, s_est, w_est, 0.0, -1.0, u_row, theta, &F.tfail);
      }
      lds_barrier();
      if (F.tfail == 0u) {
        LLZ_STAMP(row, 15);
        return true;
      }
    }
  }
  lds_barrier();  // every wave is done with F
  return false;
}

// A row's readers: the chain's, and sampleArgmax's (sampler.zig:89).
template <int XM>
using ChainSrc = typename std::conditional<XM == kXmCap, RowSrc,
                                           typename std::conditional<XM != kXmNone, LightSrc, PlainSrc>::type>::type;

template <bool FASTLD, int XM>
__device__ __forceinline__ void long_row(const KArgs& A, int row, LongLds& U, PenShared& pen_sh, int wslot) {
  constexpr bool XF = XM != kXmNone;
  const RowParams& P = A.P;
  const RowPtrs& Q = A.Q;
  using OSrc = typename std::conditional<XF, RowSrc, PlainSrc>::type;
  const ChainSrc<XM> X = make_src<ChainSrc<XM>>(P, Q, row, &pen_sh);
  OSrc O;
  if constexpr (XF) {
    O = row_orig(P, Q, row);
  } else {
    O = PlainSrc{Q.orig + (int64_t)row * P.orig_stride};
  }
  float m;
  bool nanrow;
  if (tok_stream<FASTLD, XM, 8, false>(P, Q, row, U.lng, pen_sh, X, m, nanrow)) return;
  const bool nan_sum = nanrow || !(fabsf(m) < kInf);
  select_row(P, Q, U.select, m, nan_sum ? __builtin_nanf("") : 0.0f, 0u, !nan_sum, Q.uniforms[row], false, 0ull, 0u, X, O,
             XF ? &pen_sh : nullptr, kernel_args_ptr(), row, wslot, P.cand_theta);
  LLZ_STAMP(row, 15);
}

// One workgroup per row, or (claim) one per CU taking further rows as
// k_stats_rows does.
template <bool FASTLD, int XM>
__global__ __launch_bounds__(kNT) void k_long(KArgs A) {
  __shared__ LongLds U;
  __shared__ PenShared pen_sh;
  __shared__ int next_row;
  for (int row = (int)blockIdx.x;;) {
    const __attribute__((address_space(4))) KArgs* Ap =
        (const __attribute__((address_space(4))) KArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    long_row<FASTLD, XM>(*(const KArgs*)Ap, row, U, pen_sh, (int)blockIdx.x);
    if (A.P.grid >= A.P.rows) return;
    if (threadIdx.x == 0) next_row = claim_row(A.Q.claim, A.P.epoch, A.P.grid, A.P.rows);
    __syncthreads();
    row = next_row;
    if (row >= A.P.rows) return;
  }
}

// The token-only pass over many rows (see the head of the file): up to three
// workgroups per CU, each claiming row after row; undecided rows go to the
// list Q.und.
template <bool FASTLD, int XM>
__global__ __launch_bounds__(kNT, 4) void k_tok(KArgs A) {
  __shared__ LongShared F;
  __shared__ PenShared pen_sh;
  __shared__ int next_row;
  for (int row = (int)blockIdx.x;;) {
    const __attribute__((address_space(4))) KArgs* Ap =
        (const __attribute__((address_space(4))) KArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(Ap));
    const RowParams& P = ((const KArgs*)Ap)->P;
    const RowPtrs& Q = ((const KArgs*)Ap)->Q;
    const ChainSrc<XM> X = make_src<ChainSrc<XM>>(P, Q, row, &pen_sh);
    float m;
    bool nanrow;
    const bool done = tok_stream<FASTLD, XM, 4, true>(P, Q, row, F, pen_sh, X, m, nanrow);
    if (threadIdx.x == 0) {
      if (!done) {
        const int i = claim_row(Q.nund, P.epoch, 0, 0x7fffffff);  // (a count: k_stats_rows clears it)
        if (i < P.rows) Q.und[i] = (uint32_t)row;
      }
      next_row = claim_row(A.Q.claim, A.P.epoch, (int)gridDim.x, A.P.rows);
    }
    __syncthreads();
    row = next_row;
    if (row >= A.P.rows) return;
    __syncthreads();  // next_row read by every thread before it is written again
  }
}

}  // namespace llz
