// Exact top-k selection over a row held in the registers of NT threads (one
// wave for NT = 64, else a workgroup), by counting.
//
// The row's n <= NT * PER order keys (score_order_key) are striped in pieces
// of four: thread t's key[4 r + j] is element (r * NT + t) * 4 + j (whole
// lines per load instruction); elements past n hold key 0, which is below
// every real key.  The selection is the top k under one total order: key
// descending, index ascending on equal keys.
//
// A digit histogram costs an LDS atomic per key and pass, most of them on the
// few bins that scores crowd into.  Here the k-th largest key is found by
// counting the keys at or above a trial key: two VALU operations per key and
// no LDS traffic but one word per wave.  The search keeps a bracket [lo, hi]
// with count(>= lo) >= k > count(> hi).  The first trial comes from a sample
// (the first wave's first keys, searched in that wave alone), the second lies
// past the k-th key by the sample's spacing, and from then on the trial
// interpolates between the bracket's counts in key space; where that shrank
// the bracket by less than half it takes the middle key.  Five or six counts
// find the key of ordinary scores.  After kRowCounts of them (scores that are
// mostly equal to others, or far from a line in key space) the bracket's ends
// are moved to its own smallest and largest key, and again whenever a trial
// falls between two values, so each value is told apart by one count; every
// trial from the twenty-first on takes the middle key, so at most 53 counts are
// ever needed.  2048 rows of 16384, k = 1638, us: normal scores 46, integers
// from -8 to 8 51, rounded to bf16 49 (with trials alone, some 30 counts, 99 and
// 85).  The selection's membership masks are then taken by wave ballots, and
// each thread lists its PER consecutive elements from them, so the output is in
// index order whatever the striping.
#pragma once
#include "wave_select.h"

namespace bytes_amd {

// LDS of one row's selection: membership masks, and words for sums over the
// waves in two halves used in turn.
template <int NT, int PER>
struct RowLds {
  static constexpr int NW = NT / 64;
  uint64_t masks[2 * NW * PER];
  uint32_t red[2][2 * NW];
  uint32_t guess[2];
};

// Barrier of the row's threads.
template <int NT>
__device__ __forceinline__ void row_sync() {
  if constexpr (NT == 64) wave_lds_sync();
  else __syncthreads();
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t x) {   // every lane's total (uniform)
  return (uint32_t)__builtin_amdgcn_readlane((int)wave_prefix_sum(x), 63);
}

// Sum of the waves' totals; `turn` alternates between calls.
template <int NT, class L>
__device__ __forceinline__ uint32_t row_sum(uint32_t s, L& lds, int& turn) {
  if constexpr (NT == 64) return s;
  constexpr int NW = NT / 64;
  turn ^= 1;
  if ((threadIdx.x & 63) == 0) lds.red[turn][threadIdx.x >> 6] = s;
  __syncthreads();
  uint32_t t = 0u;
#pragma unroll
  for (int w = 0; w < NW; ++w) t += lds.red[turn][w];
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
}

// Keys at or above t among the wave's N per lane.  (Counting some or all of
// them on the scalar unit, as population counts of the compare's lane mask, is
// 5% slower.)
template <int N>
__device__ __forceinline__ uint32_t wave_count_ge(const uint32_t* key, uint32_t t) {
  uint32_t c = 0u;
#pragma unroll
  for (int q = 0; q < N; ++q) c += key[q] >= t ? 1u : 0u;
  return wave_sum_u32(c);
}

// The order key of a score that is not NaN (a NaN's key, of either sign,
// falls outside [kKeyNegInf, kKeyPosInf]).
constexpr uint32_t kKeyNegInf = 0x007FFFFFu, kKeyPosInf = 0xFF800000u;
__device__ __forceinline__ uint32_t order_key_ordinary(float x) {
  const uint32_t u = __float_as_uint(x + 0.f);   // -0 becomes +0
  return u ^ ((uint32_t)((int)u >> 31) | 0x80000000u);
}

struct RowBracket {
  uint32_t lo, hi, cl, ch;             // cl = count(>= lo) >= k > ch = count(> hi)
  bool slow;                           // the last interpolation shrank the bracket by less than half
};

constexpr int kRowCounts = 7;          // interpolated counts before the bracket is snapped to its keys

// Moves the bracket's ends to the smallest and the largest key between them.
template <int NT, int PER, class L>
__device__ __forceinline__ void row_snap(const uint32_t (&key)[PER], RowBracket& b, L& lds, int& turn) {
  uint32_t up = 0xFFFFFFFFu, down = 0xFFFFFFFFu; // distances; keys outside wrap past those inside
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    up = min(up, key[q] - b.lo);
    down = min(down, b.hi - key[q]);
  }
  down = ~down;                                  // complemented: one minimum and one maximum
  wave_minmax_u32(up, down);
  if constexpr (NT > 64) {
    constexpr int NW = NT / 64;
    turn ^= 1;
    if ((threadIdx.x & 63) == 0) {
      lds.red[turn][threadIdx.x >> 6] = up;
      lds.red[turn][NW + (threadIdx.x >> 6)] = down;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      up = min(up, lds.red[turn][w]);
      down = max(down, lds.red[turn][NW + w]);
    }
  }
  b.lo += (uint32_t)__builtin_amdgcn_readfirstlane((int)up);
  b.hi -= (uint32_t)__builtin_amdgcn_readfirstlane((int)~down);
}

// A trial key in (lo, hi] (lo < hi): where a line through the bracket's counts
// reaches k, in key space (which is linear in the score within a binade); the
// middle key where the last such line did badly.  Every value here is the same
// on every lane; the arithmetic needs no accuracy.
__device__ __forceinline__ uint32_t row_trial(const RowBracket& b, uint32_t k, bool middle) {
  const float f = ((float)(b.cl - k) + 0.5f) * __builtin_amdgcn_rcpf((float)(b.cl - b.ch));
  const uint32_t w = b.hi - b.lo;
  const uint32_t d = middle || b.slow ? (w >> 1) + 1u : (uint32_t)(f * (float)w);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)(b.lo + min(max(d, 1u), w)));
}

// One count's consequence; true once the k-th key is known (b.lo).
__device__ __forceinline__ bool row_update(RowBracket& b, uint32_t t, uint32_t c, uint32_t k) {
  const uint32_t old = b.cl - b.ch;
  if (c >= k) {
    b.lo = t;
    b.cl = c;
  } else {
    b.hi = t - 1u;
    b.ch = c;
  }
  b.slow = !b.slow && (b.cl - b.ch) * 2u > old;
  return b.cl == k || b.lo >= b.hi;
}

// The selection: keys >= T where `all`; else keys > T and the `need`
// lowest-indexed keys equal to T.
struct RowSel {
  uint32_t T, need;
  bool all;
};

// First trial, and how far one rank is from the next in key space, from a
// sample of one wave's keys: the sample's value of the k-th rank.
template <int N>
__device__ __forceinline__ void row_sample(const uint32_t* key, int n, uint32_t k, uint32_t& t, float& gap) {
  uint32_t mn = 0xFFFFFFFFu, mx = 0u, ns = 0u;
#pragma unroll
  for (int q = 0; q < N; ++q) {
    mx = max(mx, key[q]);
    mn = min(mn, key[q] - 1u);                   // an element past n (key 0) is no minimum
    ns += key[q] ? 1u : 0u;
  }
  wave_minmax_u32(mn, mx);
  ns = wave_sum_u32(ns);
  const float part = (float)ns * __builtin_amdgcn_rcpf((float)n);   // of the row's keys
  const uint32_t ks = max((uint32_t)((float)k * part), 1u);
  RowBracket b;
  b.lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(mn + 1u));
  b.hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)mx);
  b.cl = ns;
  b.ch = 0u;
  b.slow = false;
  // narrow until the bracket holds about one standard error of the rank
  const uint32_t cap = 2u + (uint32_t)__builtin_amdgcn_sqrtf((float)ks);
  for (int i = 0; i < 10 && b.lo < b.hi && b.cl - b.ch > cap && b.cl != ks; ++i) {
    const uint32_t u = row_trial(b, ks, false);
    row_update(b, u, wave_count_ge<N>(key, u), ks);
  }
  t = b.lo < b.hi && b.cl != ks ? row_trial(b, ks, false) : b.lo;
  gap = (float)(b.hi - b.lo) * part * __builtin_amdgcn_rcpf((float)(b.cl - b.ch));
}

// k-th largest of the row's keys.  Every thread calls it; n >= k >= 1.
template <int NT, int PER, class L>
__device__ __forceinline__ RowSel row_search(const uint32_t (&key)[PER], int n, uint32_t k, L& lds) {
  constexpr int NS = PER < 16 ? PER : 16;        // sampled keys per lane
  int turn = 0;
  uint32_t t;
  float gap;
  if constexpr (NT == 64) {
    row_sample<NS>(key, n, k, t, gap);
  } else {
    if (threadIdx.x < 64) {
      row_sample<NS>(key, n, k, t, gap);
      if (threadIdx.x == 0) {
        lds.guess[0] = t;
        lds.guess[1] = __float_as_uint(gap);
      }
    }
    __syncthreads();
    t = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.guess[0]);
    gap = __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)lds.guess[1]));
  }
  RowBracket b{1u, 0xFFFFFFFFu, (uint32_t)n, 0u, false};
  if ((uint32_t)n > k) {
    gap *= 1.5f;
    int i = 0;
    bool done = false;
    for (; i < kRowCounts; ++i) {
      done = row_update(b, t, row_sum<NT>(wave_count_ge<PER>(key, t), lds, turn), k);
      if (done) break;
      if (i < 4 && (b.lo == 1u || b.hi == 0xFFFFFFFFu)) {
        // one side only so far: past the k-th key by the sample's spacing
        const bool up = b.hi == 0xFFFFFFFFu;
        const float step = ((float)(up ? b.cl - k : k - b.ch) + 2.f) * gap;
        const uint32_t w = b.hi - b.lo, d = max((uint32_t)fminf(step, (float)(w >> 1)), 1u);
        t = (uint32_t)__builtin_amdgcn_readfirstlane((int)(up ? b.lo + d : b.hi - d + 1u));
        gap *= 4.f;
        b.slow = false;
      } else {
        t = row_trial(b, k, false);
      }
    }
    if (__builtin_expect(!done, 0)) {
      for (uint32_t in = 0u;; ++i) {
        if (in == 0u || b.cl - b.ch == in) {
          row_snap<NT, PER>(key, b, lds, turn);
          if (b.lo >= b.hi) break;
        }
        in = b.cl - b.ch;
        t = row_trial(b, k, i >= 20);
        if (row_update(b, t, row_sum<NT>(wave_count_ge<PER>(key, t), lds, turn), k)) break;
      }
    }
  }
  RowSel s;
  s.T = b.lo;
  s.all = b.cl == k;
  s.need = k - b.ch;
  return s;
}

// This thread's keys of a row of n floats (padding: key 0), all loads in
// flight together.  load(r) returns elements (r * NT + t) * 4 .. +3 as floats
// (anything past n); NaN keys are mended where any key shows one.
template <int NT, int PER, class LOAD>
__device__ __forceinline__ void row_load(uint32_t (&key)[PER], int n, LOAD load) {
  const int t = threadIdx.x & (NT - 1);
  f32x4 raw[PER / 4];
#pragma unroll
  for (int r = 0; r < PER / 4; ++r) raw[r] = load(r);
  float nan = 0.f;                               // IEEE maximum: NaN as soon as one value is
#pragma unroll
  for (int r = 0; r < PER / 4; ++r)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      key[4 * r + e] = order_key_ordinary(raw[r][e]);
      nan = __builtin_elementwise_maximum(nan, raw[r][e]);
    }
  if (__ballot(nan != nan))
#pragma unroll
    for (int q = 0; q < PER; ++q)
      if (key[q] - kKeyNegInf > kKeyPosInf - kKeyNegInf) key[q] = 0xFFFFFFFFu;
  // pieces past the row's end
  const int left = n - 4 * t;
#pragma unroll
  for (int r = 0; r < PER / 4; ++r)
    if ((r + 1) * NT * 4 > n)                    // wave-uniform
#pragma unroll
      for (int e = 0; e < 4; ++e) key[4 * r + e] = r * NT * 4 + e < left ? key[4 * r + e] : 0u;
}

// Eight bits spread to every fourth bit of 32.
__device__ __forceinline__ uint32_t spread4(uint32_t x) {
  x = (x | (x << 12)) & 0x000F000Fu;
  x = (x | (x << 6)) & 0x03030303u;
  return (x | (x << 3)) & 0x11111111u;
}

// This thread's PER consecutive elements (from PER * t) out of a wave-striped
// mask set: bits of mask 4 r + j of wave w are its lanes' element j of piece r.
template <int NT, int PER>
__device__ __forceinline__ void row_own_bits(const uint64_t* masks, uint32_t (&bits)[(PER + 31) / 32]) {
  constexpr int F = PER / 4;                     // lanes whose pieces make up PER elements
  const int t = threadIdx.x & (NT - 1);
  const int piece = t * F, r = piece / NT, l = piece - r * NT;   // lanes l .. l+F-1 of piece r
  const uint64_t* m = masks + (l >> 6) * PER + 4 * r;
  const int sh = l & 63;
#pragma unroll
  for (int h = 0; h < (PER + 31) / 32; ++h) bits[h] = 0u;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t f = (uint32_t)(m[j] >> sh) & (F >= 32 ? 0xFFFFFFFFu : (1u << F) - 1u);
#pragma unroll
    for (int h = 0; h < (PER + 31) / 32; ++h) bits[h] |= spread4((f >> (8 * h)) & 0xFFu) << j;
  }
}

// The selection in ascending index order, through emit(slot, index).
template <int NT, int PER, class L, class EMIT>
__device__ __forceinline__ void row_emit(const uint32_t (&key)[PER], const RowSel& s, L& lds, EMIT emit) {
  constexpr int NW = NT / 64, NB = (PER + 31) / 32;
  static_assert(PER % 4 == 0 && PER <= 64, "a lane holds one mask");
  const int t = threadIdx.x & (NT - 1), lane = t & 63, w = t >> 6;
  uint64_t* masks = lds.masks;
  auto put = [&](uint64_t* dst, auto pred) {     // lane i keeps the ballot of key[i]
    uint32_t lo = 0u, hi = 0u;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const uint64_t m = __ballot(pred(key[q]));
      asm("s_nop 1\n\tv_writelane_b32 %0, %2, %4\n\tv_writelane_b32 %1, %3, %4"
          : "+v"(lo), "+v"(hi)
          : "s"((uint32_t)m), "s"((uint32_t)(m >> 32)), "n"(q));
    }
    if (lane < PER) dst[w * PER + lane] = ((uint64_t)hi << 32) | lo;
  };
  const uint32_t T = s.T;
  if (s.all) put(masks, [T](uint32_t k) { return k >= T; });
  else {
    put(masks, [T](uint32_t k) { return k > T; });
    put(masks + NW * PER, [T](uint32_t k) { return k == T; });
  }
  row_sync<NT>();
  uint32_t bits[NB], eq[NB];
  row_own_bits<NT, PER>(masks, bits);
  uint32_t ng = 0u, ne = 0u;
#pragma unroll
  for (int h = 0; h < NB; ++h) ng += __popc(bits[h]);
  if (!s.all) {
    row_own_bits<NT, PER>(masks + NW * PER, eq);
#pragma unroll
    for (int h = 0; h < NB; ++h) ne += __popc(eq[h]);
  }
  // exclusive scans over the threads: selected keys above T, and keys equal to T
  uint32_t pg = wave_prefix_sum(ng), pe = s.all ? 0u : wave_prefix_sum(ne);
  if constexpr (NW > 1) {
    if (lane == 63) {
      lds.red[0][w] = pg;
      lds.red[0][NW + w] = pe;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      pg += v < w ? lds.red[0][v] : 0u;
      pe += v < w ? lds.red[0][NW + v] : 0u;
    }
  }
  uint32_t pos = pg - ng;
  if (!s.all) {
    // of the keys equal to T before and in this thread, the first `need` are taken
    uint32_t rank = pe - ne;
    pos += min(rank, s.need);
#pragma unroll
    for (int h = 0; h < NB; ++h)
      while (eq[h]) {
        const uint32_t low = eq[h] & (0u - eq[h]);
        if (rank++ < s.need) bits[h] |= low;
        eq[h] ^= low;
      }
  }
#pragma unroll
  for (int h = 0; h < NB; ++h) {
    uint32_t m = bits[h];
    while (m) {
      emit(pos++, t * PER + 32 * h + __builtin_ctz(m));
      m &= m - 1u;
    }
  }
}

}  // namespace bytes_amd
