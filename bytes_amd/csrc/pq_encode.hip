// PQ encode: idx[n, j] = argmin_c sum_e (x[n, 8j+e] - cb[j][c][e])^2, the sum
// in fp32 in e order with separate multiply and add, first index on ties
// (ProductQuantizer.quantize, src/quantization.py:203-211).
//
// Evaluating that sum for every codeword costs 24 VALU operations each.  The
// kernel ranks the codewords on MFMA instead and evaluates the sum only where
// it decides: with t_c = |c|^2/2 - x.c (half the squared distance, less
// |x|^2/2), one v_mfma_f32_32x32x16_f16 gives t for 32 codewords x 32 vectors
// (k-slots 0-7 hold the codeword against -x, slots 8-9 |c|^2/2 in two fp16
// parts).  A lane receives runs of four consecutive codewords; the run with
// the smallest t is kept together with the second smallest run.  If the two
// are further apart than every error of t (and of the fp32 sum) can bridge,
// the answer lies in the first run and its four sums are evaluated exactly,
// two on each of the vector's two lanes.  Otherwise the whole wave evaluates
// all K sums of that vector, four codewords a lane.  The answer is that of
// the full evaluation for every input: a vector or codebook outside the range
// the error bound covers (not finite, far from the codebook's magnitude)
// takes the full evaluation too.
//
// A wave keeps one subspace's codewords in registers (32 VGPRs) and walks
// blocks of 32 vectors; a workgroup's 16 waves cover the M subspaces (several
// teams of M waves where M <= 8), so the lines of x are read once per CU.
// The exact sums read the codebook from LDS.  Bound by VALU: per 32 vectors
// 160 operations for the minima (1.25 per codeword), 70 for the exact sums and
// 50 to prepare the operand.  Runs of eight would save 48 of the first and
// cost 62 more of the second.  4 x 32768 bf16 vectors of 128, K = 256: 2413 us
// with one thread per (vector, subspace) over all K sums (its lanes' codeword
// reads were 8 KB apart in LDS, 16 to a bank), 53 us ranked.  What the ranking
// leaves undecided costs most: of N(0, 1) vectors 0.3% with 16-bit vectors and
// codebook, 3% with one of them in fp32 (83 to 87 us) and 5% with both, k-means'
// types (109 us, 2300 before), and every vector where each codeword occurs twice
// or the codebook is zero (822 us with an fp16 codebook, 604 with an fp32 one;
// 2368 and 2262 before).
#include <string.h>

#include "common.h"

namespace bytes_amd {

constexpr int kEncK = 256;        // codewords per subspace
constexpr int kEncM = 16;         // subspaces
constexpr int kEncWaves = 16;
constexpr int kEncRows = 32;      // vectors per MFMA

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct EncArgs {
  const void* x;
  int64_t x_rs, rows;             // row stride in elements; rows per head
  const void* cb;
  int64_t cb_sh;
  uint8_t* idx;
  int M, K, teams;
};

template <int DT>                 // 0 bf16, 1 fp16, 2 fp32
struct Enc8 {
  u32x4 v[DT == 2 ? 2 : 1];
  __device__ __forceinline__ float at(int e) const {
    if constexpr (DT == 2) return __uint_as_float(v[e >> 2][e & 3]);
    const uint32_t w = v[0][e >> 1];
    if constexpr (DT == 0) return __uint_as_float((e & 1) ? (w & 0xFFFF0000u) : (w << 16));
    return (float)__builtin_bit_cast(_Float16, (uint16_t)((e & 1) ? (w >> 16) : w));
  }
};

typedef u32x4 __attribute__((aligned(2))) u32x4_any;

// Eight elements at element offset o of p (any element alignment: the loads
// are 16 bytes wide either way).
template <int DT>
__device__ __forceinline__ Enc8<DT> enc_load(const void* p, int64_t o) {
  Enc8<DT> r;
  const char* b = static_cast<const char*>(p) + o * (DT == 2 ? 4 : 2);
  r.v[0] = *reinterpret_cast<const u32x4_any*>(b);
  if constexpr (DT == 2) r.v[1] = *reinterpret_cast<const u32x4_any*>(b + 16);
  return r;
}

// x - c[e].  An fp16 codeword element is widened by the subtraction itself
// (v_fma_mix_f32: -c * 1 + x, rounded once, as the subtraction is).
template <int CT>
__device__ __forceinline__ float enc_sub(float x, const Enc8<CT>& c, int e) {
  if constexpr (CT == 1) {
    float d;
    if (e & 1)
      asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(d) : "v"(c.v[0][e >> 1]), "v"(x));
    else
      asm("v_fma_mix_f32 %0, -%1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(c.v[0][e >> 1]), "v"(x));
    return d;
  } else {
    return x - c.at(e);
  }
}

// The defining sum.
template <int CT>
__device__ __forceinline__ float enc_dist(const float (&x)[8], const Enc8<CT>& c) {
  float dist;
  {
#pragma clang fp contract(off)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = enc_sub<CT>(x[e], c, e);
      dist = e == 0 ? d * d : dist + d * d;
    }
  }
  return dist;
}

__device__ __forceinline__ float min_ieee(float a, float b) { return __builtin_elementwise_minimum(a, b); }

// XT: dtype of x; CT: dtype of the codebook (1 fp16, 2 fp32); NB: blocks of 32
// codewords ranked (32 NB >= K; no branch between the MFMAs, so one block's
// minimum overlaps the next one's MFMA).
template <int XT, int CT, int NB>
__global__ __launch_bounds__(kEncWaves * 64) void pq_encode_kernel(EncArgs a) {
  __shared__ __attribute__((aligned(16))) u32x4 cbs[kEncM * kEncK * (CT == 2 ? 2 : 1)];
  constexpr int CV = CT == 2 ? 2 : 1;            // 16-byte words per codeword
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int head = blockIdx.y;
  const int M = a.M, K = a.K;
  for (int e = threadIdx.x; e < M * K; e += kEncWaves * 64) {
    const Enc8<CT> c = enc_load<CT>(a.cb, (int64_t)head * a.cb_sh + (int64_t)e * 8);
#pragma unroll
    for (int i = 0; i < CV; ++i) cbs[e * CV + i] = c.v[i];
  }
  __syncthreads();
  const int team = __builtin_amdgcn_readfirstlane(w / M), j = __builtin_amdgcn_readfirstlane(w - (w / M) * M);
  if (team >= a.teams) return;                   // no barrier follows
  const u32x4* cj = cbs + j * K * CV;
  auto codeword = [&](int c) {
    Enc8<CT> r;
#pragma unroll
    for (int i = 0; i < CV; ++i) r.v[i] = cj[c * CV + i];
    return r;
  };

  // Power-of-two scale that brings the subspace's largest |c| into [32, 64):
  // fp16 then loses nothing to its lower end, and every bound below is in
  // these units.  Magnitudes outside [2^-30, 2^30] (where fp32 squares could
  // underflow or overflow) and codewords that are not finite: ok is false and
  // every vector takes the full evaluation.
  float amax = 0.f;
  bool fin = true;
  for (int c = lane; c < K; c += 64) {
    const Enc8<CT> v = codeword(c);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float m = fabsf(v.at(e));
      fin = fin && m < __builtin_inff();
      amax = fmaxf(amax, m);
    }
  }
  amax = wave_max_f32(amax);
  const bool ok = __ballot(!fin) == 0 && amax >= 0x1p-30f && amax <= 0x1p30f;
  const int ex = (int)((__float_as_uint(amax) >> 23) & 0xFFu) - 127;
  const float s = ok ? __uint_as_float((uint32_t)(127 + 5 - ex) << 23) : 0.f;

  // A operands: rows are codewords 32 b + lane % 32; lanes 0-31 hold the
  // codeword, lanes 32-63 |c|^2/2 = 16 * hi + 2^-7 * lo (rows past K: larger
  // than any t a vector in range can have).  dc, dn: at least the largest
  // difference of a stored codeword element, and of a stored |c|^2/2, from its
  // value (a scaled fp16 element is stored exactly above 2^-14).
  f16x8 A[NB];
  float dc = CT == 1 ? 0x1p-14f : 0.f, dn = 0.f, nmax = 0.f;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int c = 32 * b + (lane & 31);
    const Enc8<CT> v = codeword(min(c, K - 1));
    const bool in = c < K;
    float n = 0.f;
    f16x8 h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float f = v.at(e) * s;
      n = __builtin_fmaf(f, f, n);
      _Float16 q = (_Float16)f;
      if constexpr (CT == 2) {
        if (fabsf((float)q) < 0x1p-14f) q = (_Float16)0.f;
        dc = fmaxf(dc, in ? fabsf(f - (float)q) : 0.f);
      }
      h[e] = q;
    }
    n *= 0.5f;
    const _Float16 n0 = (_Float16)(n * 0.0625f);
    const float r = n - 16.f * (float)n0;
    const _Float16 n1 = (_Float16)(r * 128.f);
    dn = fmaxf(dn, in ? fabsf(r - (float)n1 * 0.0078125f) : 0.f);
    nmax = fmaxf(nmax, in ? n : 0.f);
    const _Float16 z = (_Float16)0.f;
    if (!in) h = f16x8{z, z, z, z, z, z, z, z};
    A[b] = lane < 32 ? h : f16x8{in ? n0 : (_Float16)65504.f, in ? n1 : z, z, z, z, z, z, z};
  }
  if constexpr (CT == 2) dc = wave_max_f32(dc);
  dn = wave_max_f32(dn) + 0x1p-20f * wave_max_f32(nmax);   // and the rounding of the fp32 sum n
  nmax = wave_max_f32(nmax);

  const int half = lane >> 5;
  const int64_t nblk = (a.rows + kEncRows - 1) / kEncRows;
  const int64_t hrow = (int64_t)head * a.rows;
  const int64_t step = (int64_t)gridDim.x * a.teams;
  int64_t blk = (int64_t)blockIdx.x * a.teams + team;   // wave-uniform
  if (blk >= nblk) return;
  auto fetch = [&](int64_t bk) {                 // rows past the last one repeat it
    const int64_t r0 = bk * kEncRows, left = a.rows - 1 - r0;
    const int r = min(lane & 31, left < 31 ? (int)left : 31);
    const char* base = static_cast<const char*>(a.x) + ((hrow + r0) * a.x_rs + j * 8) * (XT == 2 ? 4 : 2);
    return enc_load<XT>(base, r * a.x_rs);
  };
  Enc8<XT> nxt = fetch(blk);
  for (; blk < nblk; blk += step) {
    const Enc8<XT> cur = nxt;
    nxt = fetch(blk + step < nblk ? blk + step : blk);
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = cur.at(e);
    // B operand: -x (scaled), and the weights of the |c|^2/2 parts.  X: sum of
    // |x|; R: at least the sum of what fp16 left of x.  A bf16 or fp16 element
    // fits fp16 exactly above 2^-14 (and at most that is lost below), so only
    // fp32 elements need the difference itself.
    float X = 0.f, R = XT == 2 ? 0.f : 8.f * 0x1p-14f;
    u32x4 bw;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float f0 = -x[e] * s, f1 = -x[e + 1] * s;
      X += fabsf(f0);
      X += fabsf(f1);
      if constexpr (XT == 2) {
        _Float16 q0 = (_Float16)f0, q1 = (_Float16)f1;
        if (fabsf((float)q0) < 0x1p-14f) q0 = (_Float16)0.f;
        if (fabsf((float)q1) < 0x1p-14f) q1 = (_Float16)0.f;
        R += fabsf(f0 - (float)q0);
        R += fabsf(f1 - (float)q1);
        bw[e / 2] = (uint32_t)__builtin_bit_cast(uint16_t, q0) | ((uint32_t)__builtin_bit_cast(uint16_t, q1) << 16);
      } else {
        bw[e / 2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f0, f1));
      }
    }
    constexpr uint32_t kWeights = 0x20004C00u;   // fp16 {16, 2^-7}
    if (half) bw = u32x4{kWeights, 0u, 0u, 0u};
    const f16x8 B = __builtin_bit_cast(f16x8, bw);
    // smallest and second smallest run, the run's number (this lane's half in
    // bit 5) in the low six bits of its t
    float g1 = __builtin_inff(), g2 = __builtin_inff();
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    // one block's minimum is taken while the next block's MFMA runs
    f32x16 t = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[0], B, z, 0, 0, 0);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      f32x16 u;
      if (b + 1 < NB) u = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[b + 1], B, z, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float m = min_ieee(min_ieee(t[4 * q], t[4 * q + 1]), min_ieee(t[4 * q + 2], t[4 * q + 3]));
        const float p = __uint_as_float((__float_as_uint(m) & ~63u) | (uint32_t)(4 * b + q));
        g2 = __builtin_amdgcn_fmed3f(g1, g2, p);
        g1 = min_ieee(g1, p);
      }
      if (b + 1 < NB) t = u;
    }
    g1 = __uint_as_float(__float_as_uint(g1) | (uint32_t)(half << 5));
    // the vector's other lane (lane ^ 32) holds the other half's runs
    const auto o1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(g1), __float_as_uint(g1), false, false);
    const auto o2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(g2), __float_as_uint(g2), false, false);
    const float a1 = __uint_as_float(o1[0]), b1 = __uint_as_float(o1[1]);
    const float m1 = min_ieee(a1, b1);
    const float m2 = min_ieee(__builtin_elementwise_maximum(a1, b1),
                              min_ieee(__uint_as_float(o2[0]), __uint_as_float(o2[1])));
    // Error of one t: with T >= the sum of its terms' magnitudes, 2^-18 T for
    // the MFMA's fp32 sums and 2^-17 T for the bits given to the run number;
    // what fp16 left of x against |c| < 64; what it left of c against |x|.
    // The fp32 sums rank codewords as their distances do up to 22 * 2^-24 of
    // the distance, which is at most 2 (X^2 + 2 nmax).
    const float T = __builtin_fmaf(64.f, X, nmax);
    const float err = __builtin_fmaf(0x1p-16f, T, __builtin_fmaf(64.f, R, __builtin_fmaf(dc, X, dn)));
    const float thr = __builtin_fmaf(2.f, err, 0x1p-18f * __builtin_fmaf(X, X, 2.f * nmax));
    const bool sure = ok && X <= 4096.f && m2 - m1 > thr;
    // the run's four codewords, two on each lane
    const uint32_t run = __float_as_uint(m1) & 63u;
    const int c0 = (int)(8u * (run & 31u) + 4u * (run >> 5)) + 2 * half;
    const float d0 = enc_dist<CT>(x, codeword(min(c0, K - 1)));
    const float d1 = enc_dist<CT>(x, codeword(min(c0 + 1, K - 1)));
    const bool second = d1 < d0 && c0 + 1 < K;
    const float db = second ? d1 : (c0 < K ? d0 : __builtin_inff());
    const int cbest = c0 + (second ? 1 : 0);
    const auto od = __builtin_amdgcn_permlane32_swap(__float_as_uint(db), __float_as_uint(db), false, false);
    const auto oc = __builtin_amdgcn_permlane32_swap((uint32_t)cbest, (uint32_t)cbest, false, false);
    int res = __uint_as_float(od[1]) < __uint_as_float(od[0]) ? (int)oc[1] : (int)oc[0];
    const int64_t row = blk * kEncRows + lane;   // lanes 0-31
    const bool live = lane < 32 && row < a.rows;
    uint64_t todo = __ballot(live && !sure);
    while (todo) {                               // wave-uniform: one undecided vector at a time
      const int v = __builtin_ctzll(todo);
      todo &= todo - 1;
      float xv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) xv[e] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x[e]), v));
      // this lane's best of codewords lane, lane + 64, ...: only a sum below
      // +inf (and not NaN) is ever taken, index 0 where none is
      uint32_t best = 0x7F800000u, bc = 0u;
      for (int c = lane; c < K; c += 64) {
        const float d = enc_dist<CT>(xv, codeword(c));
        if (d < __uint_as_float(best)) {
          best = __float_as_uint(d);             // sums are >= 0: their bits order as they do
          bc = (uint32_t)c;
        }
      }
      uint32_t dmin = best;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) dmin = min(dmin, (uint32_t)__shfl_xor((int)dmin, off, 64));
      uint32_t cmin = best == dmin ? bc : 0xFFFFFFFFu;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) cmin = min(cmin, (uint32_t)__shfl_xor((int)cmin, off, 64));
      if (lane == v) res = (int)cmin;
    }
    if (live) a.idx[(hrow + row) * M + j] = (uint8_t)res;
  }
}

}  // namespace bytes_amd

using namespace bytes_amd;

extern "C" int bytes_pq_encode(const void* x, int x_dtype, int heads, int64_t rows_per_head, int64_t x_row_stride,
                               int D, const void* cb, int cb_f32, int64_t cb_sh, int K, void* idx, void* stream) {
  if (!x || !cb || !idx || heads <= 0 || rows_per_head < 0 || D <= 0 || D % 8 != 0 || D / 8 > kEncM || K <= 0 ||
      K > kEncK)
    return (int)hipErrorInvalidValue;
  if (x_dtype < 0 || x_dtype > 2 || heads > 65535) return (int)hipErrorInvalidValue;
  if (rows_per_head == 0) return 0;
  EncArgs a;
  a.x = x;
  a.x_rs = x_row_stride;
  a.rows = rows_per_head;
  a.cb = cb;
  a.cb_sh = cb_sh;
  a.idx = static_cast<uint8_t*>(idx);
  a.M = D / 8;
  a.K = K;
  a.teams = kEncWaves / a.M;
  // one workgroup per CU, split over the heads: each stages its head's
  // codebook once and walks its share of the vectors
  const int64_t need = ((rows_per_head + kEncRows - 1) / kEncRows + a.teams - 1) / a.teams;
  int64_t wgs = device_cu_count() / heads;
  wgs = wgs < 1 ? 1 : wgs;
  wgs = wgs < need ? wgs : need;
  const dim3 grid((unsigned)wgs, (unsigned)heads), block(kEncWaves * 64);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define ENC(XT)                                                                               \
  if (K <= 64) {                                                                              \
    if (cb_f32) hipLaunchKernelGGL((pq_encode_kernel<XT, 2, 2>), grid, block, 0, st, a);      \
    else hipLaunchKernelGGL((pq_encode_kernel<XT, 1, 2>), grid, block, 0, st, a);             \
  } else {                                                                                    \
    if (cb_f32) hipLaunchKernelGGL((pq_encode_kernel<XT, 2, 8>), grid, block, 0, st, a);      \
    else hipLaunchKernelGGL((pq_encode_kernel<XT, 1, 8>), grid, block, 0, st, a);             \
  }
  if (x_dtype == 0) {
    ENC(0)
  } else if (x_dtype == 1) {
    ENC(1)
  } else {
    ENC(2)
  }
#undef ENC
  return (int)hipGetLastError();
}
