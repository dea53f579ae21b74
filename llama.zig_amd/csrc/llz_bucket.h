// llz_bucket.h -- top-k / top-p / min-p, the total and the draw
// (sampler.zig:106-126, 156-168) for a row whose kept prefix is longer than
// the candidate list, without sorting the row.
//
// The chain reads the row in the order (p desc, id asc).  Top-k, top-p and
// min-p keep a prefix of that order; the total is the sequential f32 sum of
// the prefix; the draw subtracts the prefix's terms from u * total until the
// value reaches 0.  Keys k = ~bits(p) ascend in that order, so the order is
// (k asc, id asc), and buckets of consecutive key ranges hold consecutive
// runs of it.
//
// While a sequential f32 sum stays in one binade [2^j, 2^(j+1)) its grid is
// u = 2^(j-23) and every term adds RN(p / u) units, whatever the order of the
// terms (llz_exact.h), unless a term is a tie.  The same holds for the
// draw's subtractions while the value stays above 2^j.  So a bucket whose
// running value is predicted to stay inside one binade (PLAIN) contributes
// one integer sum, accumulated in any order; only the buckets where the
// value may cross a binade boundary, where the top-p cut or the kept prefix's
// end may fall, where the draw may stop, or that hold a tie (EXACT) need
// their elements in order: they are gathered, sorted in LDS, and taken term
// by term.  The walks check every prediction (the value must leave a PLAIN
// bucket on its grid); a row whose check fails, or whose EXACT buckets hold
// too many elements, returns false and takes the sorting path.
//
// Passes over the row (one workgroup):
//   A  the exact p of every element (the reference's operations), its key
//      written to the fallback buffer; a coarse histogram of the keys
//      (count and mass) locates the region the chain can reach;
//   A' a fine histogram of that region from the stored keys;
//   B  (per walk) the PLAIN buckets' integer sums on their grids and the
//      EXACT buckets' elements; B2 gathers buckets a tie made EXACT.
#pragma once

#include "llz_accum.h"
#include "llz_rowops.h"

namespace llz {

constexpr int kNB = 4096;          // fine buckets
constexpr int kBList = 4096;       // gathered (EXACT) elements per walk at most
constexpr int kCoarseShift = 17;   // coarse histogram: 2^17 keys per bucket
constexpr int kBucketMinN = 8192;  // shorter rows keep the sorting path
// Relative margin of the predictions: the exact running value differs from
// the histogram's real-valued prefix by the sequential rounding (about
// sqrt(count / 12) units of the running value's grid on random data: 9e-6
// relative after configuration 4's 217k terms, so 2^-16 declined 3% of its
// rows), the truncation of lower-binade terms in the bucket masses and their
// f32 rounding (each about 2^-24).
constexpr double kBucketDelta = 0x1p-13;
constexpr int kCountShift = 44;  // histogram word: count << 44 | sum of scaled significands
// Bucket arrays are padded by one entry per 64 buckets: wave 0's scan of the
// list's places gives each lane 64 consecutive buckets, which unpadded would
// sit in one LDS bank.
constexpr int kNBP = kNB + kNB / 64;
__device__ __forceinline__ int bix(int b) { return b + (b >> 6); }

constexpr int kJgBias = 128;  // binades -120 .. 126
enum : uint8_t { kBNone = 0, kBEmpty = 1, kBPlain = 2, kBExact = 3, kBExactTie = 4 };

struct BucketShared {  // arrays indexed through bix()
  uint32_t cnt[kNBP];   // elements per bucket
  float mass[kNBP];     // their p summed (predictions only)
  union {
    struct {
      uint32_t sum[kNBP];  // PLAIN: integer sum of RN(p / u) on grid jg
      uint32_t off[kNBP];  // EXACT: first position in the sorted list
    };
    uint64_t hist[kNBP];   // histogram passes: count << 44 | the significands of p scaled to the bucket's top binade
  };
  uint16_t cj[kNBP];    // class (bits 0-2); PLAIN: the binade of the running value, + kJgBias (bits 3-10)
  uint8_t tie[kNBP];    // PLAIN: a term is a tie on its grid
  uint64_t list[kBList];  // EXACT buckets' elements, (key << 32 | id), sorted
  uint32_t nlist;
  uint32_t ctl[8];
  __device__ __forceinline__ uint32_t cls(int b) const { return cj[bix(b)] & 7u; }
  __device__ __forceinline__ int jg(int b) const { return (int)(cj[bix(b)] >> 3) - kJgBias; }
  __device__ __forceinline__ void set_cls(int b, uint32_t c) { cj[bix(b)] = (uint16_t)((cj[bix(b)] & ~7u) | c); }
  uint32_t nties, ties[8];  // buckets a tie made EXACT
  uint16_t run_b[64];       // bucket_order: the list's runs
  uint32_t wc[8];  // bucket_scan: per wave, its buckets' count and mass
  double wm[8];
};

struct BucketResult {
  uint32_t K;       // kept prefix length
  float total;      // sampler.zig:156-159
  uint32_t token;
  uint32_t consumed;
  uint32_t why;     // the bucket path declined: 1 + step (diagnostic, status bits 8-15)
};

typedef uint32_t llz_u4u __attribute__((ext_vector_type(4), aligned(4)));

// One pass of a workgroup over n elements, V per thread and tile, with the
// loads of the next kDepth tiles in flight: a pass whose work per tile is
// short is bound by the bytes it has in flight (8 words per thread took 97-118
// us over a row's 256000 stored keys, 54-80 with four tiles).  load(pos,
// out) must not read out of bounds for any pos; body(pos, values) must not
// hold a barrier.
template <int NT, int V, int D, typename T, typename Load, typename Body>
__device__ __forceinline__ void pipelined_tiles(int n, Load load, Body body) {
  constexpr int TILE = NT * V;
  const int p0 = (int)threadIdx.x * V;
  T buf[D][V];
#pragma unroll
  for (int d = 0; d < D; ++d) load(d * TILE + p0, buf[d]);
  for (int base = 0; base < n; base += D * TILE) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int pos = base + d * TILE + p0;
      T cur[V];
#pragma unroll
      for (int k = 0; k < V; ++k) cur[k] = buf[d][k];
      if (base + (D + d) * TILE < n) load(pos + D * TILE, buf[d]);
      if (base + d * TILE < n) body(pos, cur);
    }
  }
}

// A pass over a row's stored keys (n >= 8), absent positions as 0xffffffff,
// which no bucket range holds.
template <int NT, typename Body>
__device__ __forceinline__ void key_pass(const uint32_t* Kp, int n, Body body) {
  const __attribute__((address_space(1))) uint32_t* g = (const __attribute__((address_space(1))) uint32_t*)Kp;
  pipelined_tiles<NT, 8, 4, uint32_t>(
      n,
      [&](int pos, uint32_t (&k)[8]) {
        const int pc = min(pos, n - 8);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const llz_u4u q = *(const __attribute__((address_space(1))) llz_u4u*)(g + pc + 4 * h);
          k[4 * h + 0] = q.x; k[4 * h + 1] = q.y; k[4 * h + 2] = q.z; k[4 * h + 3] = q.w;
        }
      },
      [&](int pos, uint32_t (&k)[8]) {
        if (pos > n - 8) {  // the row's end: read again, element by element
#pragma unroll
          for (int i = 0; i < 8; ++i) k[i] = pos + i < n ? g[pos + i] : 0xffffffffu;
        }
        body(pos, k);
      });
}

// RN(e / S) for 2^-90 <= e <= 1 and 2^-20 <= S <= 2^20 from y = RN(1 / S), by
// Markstein's method (llz_math.h): the first correction makes the quotient
// faithful, and the second, from a faithful quotient and the correctly
// rounded reciprocal, rounds correctly; remainders are exact in an fma, and
// no operation underflows in this range.  Six operations, where the IEEE
// division takes about twelve.
__device__ __forceinline__ float div_by(float e, float S, float y) {
  const float q0 = e * y;
  const float q1 = fmaf(fmaf(-S, q0, e), y, q0);
  return fmaf(fmaf(-S, q1, e), y, q1);
}

__device__ __forceinline__ float key_p(uint32_t key) { return __uint_as_float(~key); }

// Biased exponent of p = key_p(key) (1 for subnormals) and its 24-bit
// significand: p = sig * 2^(E - 150).
__device__ __forceinline__ uint32_t key_E(uint32_t key) {
  const uint32_t e = (~key >> 23) & 0xffu;
  return e == 0u ? 1u : e;
}
__device__ __forceinline__ uint32_t key_sig(uint32_t key) {
  const uint32_t b = ~key;
  return (b & 0x7fffffu) | (((b >> 23) & 0xffu) != 0u ? 0x800000u : 0u);
}

// One element's histogram word for a bucket whose largest p has biased
// exponent Etop: its count and its significand scaled to 2^(Etop - 150)
// (terms of lower binades lose their low bits: relative error < 2^-23 each).
__device__ __forceinline__ uint64_t hist_word(uint32_t key, uint32_t Etop) {
  const uint32_t d = Etop - key_E(key);  // >= 0: p <= the bucket's largest
  const uint64_t v = d < 24u ? (uint64_t)(key_sig(key) >> d) : 0ull;
  return (1ull << kCountShift) | v;
}

// Count and mass of a bucket from its histogram word (Etop as above).
__device__ __forceinline__ void hist_unpack(uint64_t h, uint32_t Etop, uint32_t& cnt, float& mass) {
  cnt = (uint32_t)(h >> kCountShift);
  const double sig = (double)(h & ((1ull << kCountShift) - 1ull));
  mass = (float)(sig * exp2((double)((int)Etop - 150)));
}

// Binade of a positive double (its unbiased exponent; -1023 for 0).
__device__ __forceinline__ int dbl_binade(double x) {
  return (int)((uint64_t)__double_as_longlong(x) >> 52 & 0x7ffu) - 1023;
}

// A wave's sequential chain over len terms (sampler.zig:112-117 / :162-166):
// ADD stops at the first value > thr (thr >= 0), SUB at the first value <= 0.
// Returns the value after the stopping term (or after the last), with
// `before` the value before the stopping term.
template <bool SUB, typename TermFn>
__device__ float wave_seq_stop(float s, int len, float thr, int& stop, float& before, TermFn term) {
  stop = -1;
  const int lane = lane_id();
  for (int base = 0; base < len; base += kWave) {
    const int p = base + lane;
    const float x0 = p < len ? term(p) : -0.0f;
    const int cnt = min(kWave, len - base);
    const bool present = lane < cnt && !(as_bits(x0) >> 31);
    const float acc = wave_chain_lanes<SUB>(s, x0, cnt);
    const bool hit = present && (SUB ? (acc <= 0.0f) : (thr >= 0.0f && acc > thr));
    const uint64_t hits = bal64(hit);
    if (hits != 0ull) {
      const int L = __ffsll((long long)hits) - 1;
      stop = base + L;
      before = L > 0 ? readlane_f32(acc, L - 1) : s;
      return readlane_f32(acc, L);
    }
    s = readlane_f32(acc, cnt - 1);
  }
  before = s;
  return s;
}

// Every thread: exclusive prefixes of the buckets' counts and masses, kNB / NT
// consecutive buckets a thread; calls cls_of(b, excl_count, excl_mass) for
// each of them in order.  (One wave with 64 buckets a lane took 14-24 us.)
template <int NT, typename ClsFn>
__device__ __forceinline__ void bucket_scan(BucketShared& bs, ClsFn cls_of) {
  constexpr int PL = kNB / NT;
  const int t = (int)threadIdx.x, lane = lane_id(), w = wave_id();
  uint32_t c = 0;
  double ms = 0.0;
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    c += bs.cnt[bix(t * PL + i)];
    ms += (double)bs.mass[bix(t * PL + i)];
  }
  uint32_t ci = c;
  double mi = ms;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t oc = __shfl_up(ci, d, kWave);
    const double om = __shfl_up(mi, d, kWave);
    if (lane >= d) {
      ci += oc;
      mi += om;
    }
  }
  if (lane == kWave - 1) {
    bs.wc[w] = ci;
    bs.wm[w] = mi;
  }
  __syncthreads();
  uint32_t ec = ci - c;
  double em = mi - ms;
  for (int i = 0; i < w; ++i) {
    ec += bs.wc[i];
    em += bs.wm[i];
  }
#pragma unroll
  for (int i = 0; i < PL; ++i) {
    const int b = t * PL + i;
    cls_of(b, ec, em);
    ec += bs.cnt[bix(b)];
    em += (double)bs.mass[bix(b)];
  }
  __syncthreads();
}

// Bucket of a key in the fine range [kmin, kcut): (key - kmin) >> shift.
struct BucketRange {
  uint32_t kmin, kcut;
  int shift;
  __device__ __forceinline__ bool in(uint32_t key) const { return key >= kmin && key < kcut; }
  __device__ __forceinline__ int of(uint32_t key) const { return (int)min((key - kmin) >> shift, (uint32_t)kNB - 1u); }
};

// Pass B over [blo, bhi) = the whole range when every EXACT bucket's elements
// fit the list (`gather`): the PLAIN buckets' integer sums of RN(p / u) on
// their grids, with tie flags, and the EXACT buckets' elements put in their
// places of the list (bs.off, each bucket's run in any order).  Then a bucket
// holding a tie becomes EXACT: with `gather`, ExactTie, still to be gathered.
template <int NT>
__device__ void bucket_sums(const uint32_t* Kp, int n, const BucketRange& br, BucketShared& bs, bool gather) {
  const int t = (int)threadIdx.x;
  for (int b = t; b < kNB; b += NT) {
    bs.sum[bix(b)] = 0u;
    bs.tie[bix(b)] = 0u;
  }
  __syncthreads();
  // per element one LDS read (its bucket's class and grid, all eight in
  // flight) and one atomic without a result; the few EXACT elements, whose
  // atomics return their place, follow one per lane and step
  key_pass<NT>(Kp, n, [&](int pos, uint32_t (&k)[8]) {
    uint32_t bb[8], cj[8], ex = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool in = br.in(k[i]);
      bb[i] = (uint32_t)bix(in ? br.of(k[i]) : 0);
      cj[i] = in ? bs.cj[bb[i]] : 0u;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t cl = cj[i] & 7u;
      bool tie;
      const uint32_t r = grid_round(key_p(k[i]), (int)(cj[i] >> 3) - kJgBias, tie);
      // a PLAIN bucket's mass lies within one binade, 2^23 units of its grid:
      // its sum cannot wrap
      if (cl == kBPlain) {
        atomicAdd(&bs.sum[bb[i]], r);
        if (tie) bs.tie[bb[i]] = 1u;
      }
      ex |= (cl == kBExact ? 1u : 0u) << i;
    }
    if (!gather) ex = 0u;
    while (ex != 0u) {
      const int i = __ffs((int)ex) - 1;
      ex &= ex - 1u;
      uint32_t key = 0u, b = 0u;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        key = q == i ? k[q] : key;
        b = q == i ? bb[q] : b;
      }
      bs.list[atomicAdd(&bs.off[b], 1u)] = ((uint64_t)key << 32) | (uint32_t)(pos + i);
    }
  });
  __syncthreads();
  for (int b = t; b < kNB; b += NT) {
    const uint32_t cl = bs.cls(b);
    if (gather && cl == kBExact) bs.off[bix(b)] -= bs.cnt[bix(b)];  // back to the run's start
    if (cl == kBPlain && bs.tie[bix(b)]) bs.set_cls(b, gather ? kBExactTie : kBExact);
  }
  __syncthreads();
}

// Wave 0: the EXACT buckets from `blo` on whose elements fit the list
// together: each bucket's place in the list, and the end of that range (kNB
// when every remaining one fits), for every thread.
template <int NT>
__device__ int bucket_places(BucketShared& bs, int blo) {
  if (wave_id() == 0) {
    // EXACT counts from blo in bucket order, 64 buckets a lane
    constexpr int PL = kNB / kWave;
    const int lane = lane_id();
    uint32_t c = 0;
    for (int i = 0; i < PL; ++i) {
      const int b = lane * PL + i;
      c += (b >= blo && bs.cls(b) == kBExact) ? bs.cnt[bix(b)] : 0u;
    }
    uint32_t ci = c;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t o = __shfl_up(ci, d, kWave);
      if (lane >= d) ci += o;
    }
    uint32_t run = ci - c;
    int bhi = kNB;
    for (int i = 0; i < PL; ++i) {
      const int b = lane * PL + i;
      const bool ex = b >= blo && bs.cls(b) == kBExact;
      if (ex && run + bs.cnt[bix(b)] > (uint32_t)kBList && b < bhi) bhi = b;
      bs.off[bix(b)] = run;
      run += ex ? bs.cnt[bix(b)] : 0u;
    }
    bhi = (int)wave_min_u32((uint32_t)bhi);
    const uint32_t total = readlane_u32(ci, kWave - 1);
    if (lane == 0) {
      bs.ctl[6] = (uint32_t)bhi;
      bs.ctl[7] = total;  // the list's length when bhi == kNB
      bs.nlist = 0u;
    }
  }
  __syncthreads();
  return (int)bs.ctl[6];
}

// The elements of the buckets of class CLS in [blo, bhi), put in their places.
template <int NT>
__device__ void bucket_gather(const uint32_t* Kp, int n, const BucketRange& br, BucketShared& bs, int blo, int bhi,
                              uint32_t cls) {
  const int t = (int)threadIdx.x;
  key_pass<NT>(Kp, n, [&](int pos, uint32_t (&k)[8]) {
    uint32_t ex = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool in = br.in(k[i]);
      const int b = in ? br.of(k[i]) : 0;
      ex |= (in && b >= blo && b < bhi && bs.cls(b) == cls ? 1u : 0u) << i;
    }
    while (ex != 0u) {
      const int i = __ffs((int)ex) - 1;
      ex &= ex - 1u;
      uint32_t key = 0u;
#pragma unroll
      for (int q = 0; q < 8; ++q) key = q == i ? k[q] : key;
      bs.list[atomicAdd(&bs.off[bix(br.of(key))], 1u)] = ((uint64_t)key << 32) | (uint32_t)(pos + i);
    }
  });
  __syncthreads();
  for (int b = blo + t; b < bhi; b += NT)
    if (bs.cls(b) == cls) bs.off[bix(b)] -= bs.cnt[bix(b)];
  __syncthreads();
}

// The same for at most kTieMax buckets b[0, nb) whose keys are told by their
// ranges alone, without a look at a class per element.
constexpr int kTieMax = 8;
template <int NT>
__device__ void bucket_gather_few(const uint32_t* Kp, int n, const BucketRange& br, BucketShared& bs, const uint32_t* b,
                                  int nb) {
  uint32_t lo[kTieMax], wd[kTieMax];
#pragma unroll
  for (int q = 0; q < kTieMax; ++q) {
    const uint32_t bq = q < nb ? b[q] : 0u;
    lo[q] = br.kmin + (bq << br.shift);
    // (the last bucket holds every key up to the range's end)
    wd[q] = q < nb ? (bq == (uint32_t)kNB - 1u ? br.kcut - lo[q] : min(1u << br.shift, br.kcut - lo[q])) : 0u;
  }
  key_pass<NT>(Kp, n, [&](int pos, uint32_t (&k)[8]) {
    uint32_t ex = 0u;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      bool hit = false;
#pragma unroll
      for (int q = 0; q < kTieMax; ++q) hit = hit || k[i] - lo[q] < wd[q];
      ex |= (hit ? 1u : 0u) << i;
    }
    while (ex != 0u) {
      const int i = __ffs((int)ex) - 1;
      ex &= ex - 1u;
      uint32_t key = 0u;
#pragma unroll
      for (int q = 0; q < 8; ++q) key = q == i ? k[q] : key;
      bs.list[atomicAdd(&bs.off[bix(br.of(key))], 1u)] = ((uint64_t)key << 32) | (uint32_t)(pos + i);
    }
  });
  __syncthreads();
  if (threadIdx.x < (unsigned)nb) bs.off[bix((int)b[threadIdx.x])] -= bs.cnt[bix((int)b[threadIdx.x])];
  __syncthreads();
}

// Orders each bucket's run of the list[0, nl) (runs of some 100 to 300
// elements on near-flat rows).  Each of the up to kOrdRuns runs is cut into 64
// equal steps of its keys; an element's place is first that of its step (a
// count per step, a scan per run), then, among the step's few elements, that
// of its key.  scr: 64 kOrdRuns words.  (The bitonic network over the list
// took some 70 us, counting each run's smaller keys 97 us; this 8.)  More runs
// than that are counted.
constexpr int kOrdRuns = 64;
template <int NT>
__device__ void bucket_order(const BucketRange& br, BucketShared& bs, int nl, uint32_t* scr) {
  constexpr int PT = kBList / NT;
  const int t = (int)threadIdx.x, lane = lane_id(), w = wave_id();
  uint64_t k[PT];
  uint32_t at[PT];
  // number the runs in the list (bs.tie: a bucket's ties are known by now)
  if (t == 0) bs.nties = 0u;
  for (int i = t; i < 64 * kOrdRuns; i += NT) scr[i] = 0u;
  lds_barrier();
  for (int b = t; b < kNB; b += NT) {
    const uint32_t c = bs.cnt[bix(b)], o = bs.off[bix(b)];
    if (bs.cls(b) == kBExact && c > 0u && o + c <= (uint32_t)nl) {
      const uint32_t q = atomicAdd(&bs.nties, 1u);
      bs.tie[bix(b)] = (uint8_t)min(q, 255u);
      if (q < (uint32_t)kOrdRuns) bs.run_b[q] = (uint16_t)b;
    }
  }
  lds_barrier();
  const int nr = (int)bs.nties;
  if (nr > kOrdRuns) {
#pragma unroll
    for (int q = 0; q < PT; ++q) {
      const int i = q * NT + t;
      k[q] = i < nl ? bs.list[i] : ~0ull;
      at[q] = 0u;
      if (i < nl) {
        const int b = br.of((uint32_t)(k[q] >> 32));
        const uint32_t s = bs.off[bix(b)], e = s + bs.cnt[bix(b)];
        uint32_t r = 0u;
        for (uint32_t j = s; j < e; ++j) r += bs.list[j] < k[q] ? 1u : 0u;
        at[q] = s + r;
      }
    }
    lds_barrier();
#pragma unroll
    for (int q = 0; q < PT; ++q)
      if (q * NT + t < nl) bs.list[at[q]] = k[q];
    lds_barrier();
    return;
  }
  const int sh = max(0, br.shift - 6);
  auto step_of = [&](uint64_t key) {
    const uint32_t kk = (uint32_t)(key >> 32), b = (uint32_t)br.of(kk);
    return ((uint32_t)bs.tie[bix((int)b)] << 6) | min((kk - br.kmin - (b << br.shift)) >> sh, 63u);
  };
  uint32_t st[PT];
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const int i = q * NT + t;
    k[q] = i < nl ? bs.list[i] : ~0ull;
    st[q] = i < nl ? step_of(k[q]) : 0u;
    at[q] = i < nl ? atomicAdd(&scr[st[q]], 1u) : 0u;
  }
  lds_barrier();
  // per run: its steps' starts, with their counts above (places fit 13 bits)
  static_assert(kBList < (1 << 13), "a place and a count share a word");
  for (int r = w; r < nr; r += NT / kWave) {
    const uint32_t c = scr[64 * r + lane];
    const uint32_t in = wave_incl_scan_op(c, 0u, [](uint32_t x, uint32_t y) { return x + y; });
    scr[64 * r + lane] = (bs.off[bix((int)bs.run_b[r])] + in - c) | (c << 16);
  }
  lds_barrier();
#pragma unroll
  for (int q = 0; q < PT; ++q)
    if (q * NT + t < nl) bs.list[(scr[st[q]] & 0xffffu) + at[q]] = k[q];
  lds_barrier();
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    if (q * NT + t < nl) {
      const uint32_t x = scr[st[q]], s = x & 0xffffu, c = x >> 16;
      uint32_t r = 0u;
      for (uint32_t j = s; j < s + c; ++j) r += bs.list[j] < k[q] ? 1u : 0u;
      at[q] = s + r;
    }
  }
  lds_barrier();
#pragma unroll
  for (int q = 0; q < PT; ++q)
    if (q * NT + t < nl) bs.list[at[q]] = k[q];
  lds_barrier();
}

// Why a walk stops (kWalkOk: the chain ended; kWalkMore: it reached the end
// of the batch's bucket range; the others decline the row).
enum : uint32_t { kWalkOk = 0, kWalkLeftBinade = 1, kWalkCutInPlain = 2, kWalkEndInPlain = 3, kWalkUnpredicted = 4,
                  kWalkPastRange = 5, kWalkMore = 6 };

// One walk over buckets [b_from, b_to) in key order by wave 0 (SUB: the
// draw), continuing from the running value v at position pos.  Positions
// [0, lim) take part; ADD stops at the first value > thr (thr < 0: never),
// SUB at the first value <= 0.  On kWalkOk: stop and the stopping element's
// position (pos), id and the value before it; or pos = lim.
template <bool SUB>
__device__ uint32_t bucket_walk(const BucketShared& bs, float& v, float& before, uint32_t& pos, uint32_t lim,
                                float thr, bool& stop, uint32_t& id_out, int b_from, int b_to) {
  const int lane = lane_id();
  stop = false;
  before = v;
  for (int b0 = b_from & ~(kWave - 1); b0 < b_to; b0 += kWave) {
    const int b = b0 + lane;  // < kNB
    const uint32_t cl = bs.cls(b);
    const int jb = bs.jg(b);
    const uint32_t sm = bs.sum[bix(b)], ct = bs.cnt[bix(b)], of = bs.off[bix(b)];
    int i = b0 < b_from ? b_from - b0 : 0;
    const int iend = min(kWave, b_to - b0);
    while (i < iend) {
      if (pos >= lim) return kWalkOk;
      const Grid g = grid_of(v);
      const bool live = lane >= i && lane < iend;
      const bool easy = live && (cl == kBEmpty || (cl == kBPlain && jb == g.j));
      const uint64_t hard = bal64(live && !easy);
      const int e = hard != 0ull ? __ffsll((long long)hard) - 1 : iend;
      const bool run = lane >= i && lane < e;
      const uint32_t add = wave_sum_sat(run && cl == kBPlain ? sm : 0u, kSat);
      const uint32_t pc = wave_sum_sat(run ? ct : 0u, 0x7fffffffu);
      if (e > i) {
        if (SUB) {
          if (add != 0u) {
            if (add >= g.N || g.N - add <= kGridBase) return kWalkLeftBinade;
            v = grid_value(g.N - add, g.j);
          }
        } else {
          if (add != 0u) {
            if (g.N + add >= kGridTop || g.N < kGridBase) return kWalkLeftBinade;
            v = grid_value(g.N + add, g.j);
          }
          if (thr >= 0.0f && v > thr) return kWalkCutInPlain;
        }
        pos += pc;
        if (pos > lim) return kWalkEndInPlain;
      }
      if (e >= iend) break;
      if (pos >= lim) return kWalkOk;
      if (readlane_u32(cl, e) != kBExact) return kWalkUnpredicted;  // NONE, or PLAIN on another grid
      const uint32_t o = readlane_u32(of, e);
      const uint32_t c = readlane_u32(ct, e);
      const int len = (int)min(c, lim - pos);
      int st;
      float bf;
      v = wave_seq_stop<SUB>(v, len, thr, st, bf, [&](int d) { return key_p((uint32_t)(bs.list[o + d] >> 32)); });
      if (st >= 0) {
        stop = true;
        before = bf;
        pos += (uint32_t)st;
        id_out = (uint32_t)bs.list[o + st];
        return kWalkOk;
      }
      pos += (uint32_t)len;
      i = e + 1;
    }
  }
  if (pos >= lim) return kWalkOk;
  return b_to < kNB ? kWalkMore : kWalkPastRange;
}

// A whole walk: PLAIN sums, then batches of EXACT buckets, each walked by
// wave 0 from where the last stopped.  Returns 0 or the decline reason; the
// results are broadcast through bs.ctl.
template <bool SUB, int NT>
__device__ uint32_t bucket_chain(const uint32_t* Kp, int n, const BucketRange& br, BucketShared& bs, float v0,
                                 uint32_t lim, float thr, float& v_out, float& before_out, uint32_t& pos_out,
                                 bool& stop_out, uint32_t& id_out, int row, uint32_t* scr) {
  // one pass when every EXACT bucket fits the list; the buckets a tie made
  // EXACT, if any, take another, behind the others in the list
  bool all = bucket_places<NT>(bs, 0) == kNB;
  uint32_t nl = bs.ctl[7];
  bucket_sums<NT>(Kp, n, br, bs, all);
  LLZ_STAMP(row, 29);
  if (all) {
    if (threadIdx.x == 0) {
      bs.nlist = nl;
      bs.nties = 0u;
    }
    __syncthreads();
    for (int b = (int)threadIdx.x; b < kNB; b += NT) {
      if (bs.cls(b) == kBExactTie) {
        bs.off[bix(b)] = atomicAdd(&bs.nlist, bs.cnt[bix(b)]);
        const uint32_t q = atomicAdd(&bs.nties, 1u);
        if (q < (uint32_t)kTieMax) bs.ties[q] = (uint32_t)b;
      }
    }
    __syncthreads();
    const uint32_t nt = bs.nlist;
    const int ntie = (int)bs.nties;
    all = nt <= (uint32_t)kBList;
    if (all && ntie > 0) {
      if (ntie <= kTieMax)
        bucket_gather_few<NT>(Kp, n, br, bs, bs.ties, ntie);
      else
        bucket_gather<NT>(Kp, n, br, bs, 0, kNB, kBExactTie);
    }
    nl = nt;
    for (int b = (int)threadIdx.x; b < kNB; b += NT)
      if (bs.cls(b) == kBExactTie) bs.set_cls(b, kBExact);
    __syncthreads();
    LLZ_STAMP(row, 59);
    if (all) bucket_order<NT>(br, bs, (int)nl, scr);
  }
  float v = v0, before = v0;
  uint32_t pos = 0, id = 0xffffffffu, why = kWalkMore;
  bool stop = false;
  for (int blo = 0; why == kWalkMore;) {
    // (in batches: the EXACT buckets from blo on that fit the list together)
    int bhi = kNB;
    if (!all) {
      bhi = bucket_places<NT>(bs, blo);
      if (bhi == blo) return 16u;  // one bucket holds more than the list
      bucket_gather<NT>(Kp, n, br, bs, blo, bhi, kBExact);
      // the list's length: the places' end
      uint32_t end = 0u;
      for (int b = blo + (int)threadIdx.x; b < bhi; b += NT)
        if (bs.cls(b) == kBExact) end = max(end, bs.off[bix(b)] + bs.cnt[bix(b)]);
      atomicMax(&bs.nlist, end);
      __syncthreads();
      bucket_order<NT>(br, bs, (int)bs.nlist, scr);
    }
    if (blo == 0) LLZ_STAMP(row, 30);
    if (wave_id() == 0) {
      why = bucket_walk<SUB>(bs, v, before, pos, lim, thr, stop, id, blo, bhi);
      if (lane_id() == 0) {
        bs.ctl[0] = why;
        bs.ctl[1] = __float_as_uint(v);
        bs.ctl[2] = __float_as_uint(before);
        bs.ctl[3] = pos;
        bs.ctl[4] = stop ? 1u : 0u;
        bs.ctl[5] = id;
      }
    }
    __syncthreads();
    why = bs.ctl[0];
    v = __uint_as_float(bs.ctl[1]);
    before = __uint_as_float(bs.ctl[2]);
    pos = bs.ctl[3];
    stop = bs.ctl[4] != 0u;
    id = bs.ctl[5];
    __syncthreads();  // every thread has read ctl before a next batch writes it
    if (blo == 0) LLZ_STAMP(row, 31);
    blo = bhi;
  }
  v_out = v;
  before_out = before;
  pos_out = pos;
  stop_out = stop;
  id_out = id;
  return why;
}

}  // namespace llz
