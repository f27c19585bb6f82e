// One step of the streaming top-k over key chunks (benchmarks/
// sparse_attention.py:286-309) in one launch: the causal mask and forced
// recent window of the chunk's scores (:294-300), the top-k over the row's
// running list and the chunk (:301-307), and the next running list
// (:308-309), or after the last chunk the row's final indices ordered by score
// with the sentinel rule (:288-293).  The row is read once into registers and
// selected by counting (row_select.h); the mask is applied to the keys there,
// so the masked scores are never written, and only the selected entries are
// read again (from L2) to be moved, all loads of the move in flight together
// (moved from the listing loop, one load after another, a step took 52 us).
// The last step sorts in registers (row_sort.h).  Bound by VALU issue and the
// latency of the counts (eight workgroups to a CU).  3584 rows, chunks of 2048
// keys, kb = 819: mask, top-k and merge launches took 24 + 27 + 19 us a step
// (the last, with its sort and fill, 24 + 98 + 19 + 12); fused 29 us for the
// first chunk, 36 for those with a running list, 59 for the last.
#include "row_select.h"
#include "row_sort.h"

namespace bytes_amd {

struct StepArgs {
  const float* cand;         // row r: [running list | chunk] at cand + r * cand_rs + off
  int64_t cand_rs;
  int off, nrun, n;          // running-list entries, chunk keys
  const int32_t* ridx;       // key indices of the running list
  int64_t ridx_rs;
  int kc0;                   // the chunk's first key
  const int64_t* pos;        // [Qc] query positions; row r is query row r % Qc
  int Qc, local_w, S, kb, ksel;
  float* out_v;              // next running list: scores (kb per row) ...
  int64_t out_v_rs;
  int32_t* out_i;            // ... and key indices
  int64_t out_i_rs;
  int64_t* out_f;            // last step: [rows, kb] final indices
};

// SW: waves that sort on the last step (256 selected entries each), 0: not the
// last step.
template <int NT, int PER, int SW>
__global__ __launch_bounds__(NT, 4) void select_step_kernel(StepArgs a) {
  __shared__ __attribute__((aligned(16))) RowLds<NT, PER> lds;
  __shared__ uint64_t sb[SW ? 256 * SW : 1];
  __shared__ uint16_t list[SW ? 256 * SW : NT * PER];   // selected elements, ascending
  const int t = threadIdx.x;
  const int64_t row = blockIdx.x;
  // the row from its last 16-byte boundary: element e of it is candidate
  // e - lead, candidates from nrun on are keys kc0, kc0 + 1, ...
  const int lead = a.off & 3, first = lead + a.nrun, end = first + a.n;
  const float* x = a.cand + row * a.cand_rs + (a.off - lead);
  const int64_t p = a.pos[row % a.Qc];
  // chunk elements past `em` come after the query; those from `ew` up to it are
  // forced in
  const int64_t pe = p - a.kc0 + first;
  const int em = (int)(pe < first - 1 ? first - 1 : pe < end - 1 ? pe : end - 1);
  int ew = end;
  if (a.local_w > 0) {
    const int64_t w0 = p - a.local_w + 1, lo = (w0 > 0 ? w0 : 0) - a.kc0 + first;
    ew = (int)(lo < first ? first : lo < end ? lo : end);
  }
  const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), (short)0, end * 4, 0x00020000);
  uint32_t key[PER];
  row_load<NT, PER>(key, end, [&](int r) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (r * NT + t) * 16, 0, 0));
  });
#pragma unroll
  for (int e = 0; e < 3; ++e)
    if (t == 0 && e < lead) key[e] = 0u;
  if (em < end - 1 || ew < end) {                // row-uniform
    const int e0 = 4 * t;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int e = e0 + (q >> 2) * NT * 4 + (q & 3);
      const bool forced = e >= ew && e <= em, after = e > em && e < end;
      key[q] = forced ? kKeyPosInf : after ? kKeyNegInf : key[q];
    }
  }
  const RowSel s = row_search<NT, PER>(key, a.nrun + a.n, (uint32_t)a.ksel, lds);
  auto value = [&](int e) {                      // element e's score as the mask leaves it
    return e >= ew && e <= em ? __builtin_inff() : e > em ? kNegInf : x[e];
  };
  const int32_t* ri = a.ridx + row * a.ridx_rs;
  auto index = [&](int e) { return e < first ? ri[e - lead] : a.kc0 + (e - first); };
  if constexpr (SW == 0) {
    float* ov = a.out_v + row * a.out_v_rs;
    int32_t* oi = a.out_i + row * a.out_i_rs;
    row_emit<NT, PER>(key, s, lds, [&](uint32_t at, int e) { list[at] = (uint16_t)e; });
    __syncthreads();
#pragma unroll 4
    for (int i = t; i < a.ksel; i += NT) {
      const int e = list[i];
      const float v = value(e);
      const int k = index(e);
      ov[i] = v;
      oi[i] = k;
    }
    for (int i = a.ksel + t; i < a.kb; i += NT) {   // fillers
      ov[i] = kNegInf;
      oi[i] = a.S;
    }
  } else {
    int64_t* of = a.out_f + row * a.kb;
    row_emit<NT, PER>(key, s, lds, [&](uint32_t at, int e) { list[at] = (uint16_t)e; });
    __syncthreads();
#pragma unroll 4
    for (int i = t; i < a.ksel; i += NT) {
      const int e = list[i];
      sb[i] = row_sort_pair(score_order_key(value(e)), e);
    }
    double y[4];
    row_sort_desc<SW>(sb, a.ksel, y);
    const int lane = t & 63, w = t >> 6;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 256 * w + 64 * r + lane;
      if (w < SW && i < a.ksel) {
        const int v = index(row_sort_element(y[r]));
        of[i] = v < a.S && v <= p ? v : a.S;
      }
    }
    for (int i = a.ksel + t; i < a.kb; i += NT) of[i] = a.S;
  }
}

// Longest row (with up to three elements before it) and longest sorted
// selection of the kernel.
constexpr int kStepRow = 16384;

}  // namespace bytes_amd

using namespace bytes_amd;

extern "C" int bytes_select_step(const void* cand, int64_t cand_rs, int off, int nrun, int n, const void* ridx,
                                 int64_t ridx_rs, int kc0, const void* pos, int Qc, int local_w, int S, int kb,
                                 int64_t rows, void* out_vals, int64_t out_vals_rs, int out_off, void* out_idx,
                                 int64_t out_idx_rs, void* final_idx, void* stream) {
  if (!cand || !pos || rows <= 0 || n <= 0 || nrun < 0 || off < 0 || kc0 < 0 || Qc <= 0 || local_w < 0 || S <= 0 ||
      kb <= 0 || (nrun > 0 && !ridx) || (int64_t)off + nrun + n > cand_rs)
    return (int)hipErrorInvalidValue;
  const bool last = final_idx != nullptr;
  if (!last && (!out_vals || !out_idx || out_off < 0 || out_vals_rs < (int64_t)out_off + kb || out_idx_rs < kb))
    return (int)hipErrorInvalidValue;
  // 16-byte loads from the row's last boundary
  if (reinterpret_cast<uintptr_t>(cand) % 16 != 0 || cand_rs % 4 != 0) return (int)hipErrorInvalidValue;
  const int64_t total = (int64_t)(off & 3) + nrun + n;
  const int ksel = (int64_t)kb < (int64_t)nrun + n ? kb : nrun + n;
  if (total > kStepRow || (last && ksel > kRowSortMax)) return (int)hipErrorNotSupported;
  if (rows > 0x7FFFFFFFL) return (int)hipErrorInvalidConfiguration;
  StepArgs a;
  a.cand = static_cast<const float*>(cand);
  a.cand_rs = cand_rs;
  a.off = off; a.nrun = nrun; a.n = n;
  a.ridx = static_cast<const int32_t*>(ridx);
  a.ridx_rs = ridx_rs;
  a.kc0 = kc0;
  a.pos = static_cast<const int64_t*>(pos);
  a.Qc = Qc; a.local_w = local_w; a.S = S; a.kb = kb; a.ksel = ksel;
  a.out_v = last ? nullptr : static_cast<float*>(out_vals) + out_off;
  a.out_v_rs = out_vals_rs;
  a.out_i = static_cast<int32_t*>(out_idx);
  a.out_i_rs = out_idx_rs;
  a.out_f = static_cast<int64_t*>(final_idx);
  hipStream_t st = static_cast<hipStream_t>(stream);
#define STEP1(NT, PER, SW) \
  hipLaunchKernelGGL((select_step_kernel<NT, PER, SW>), dim3((unsigned)rows), dim3(NT), 0, st, a)
#define STEP(NT, PER)                  \
  if (!last) STEP1(NT, PER, 0);        \
  else if (ksel <= 1024) STEP1(NT, PER, 4); \
  else STEP1(512, (NT == 512 ? PER : PER / 2), 8);
  if (total <= 2048) {
    STEP(256, 8)
  } else if (total <= 4096) {
    STEP(256, 16)
  } else if (total <= 8192) {
    STEP(256, 32)
  } else {
    STEP(512, 32)
  }
#undef STEP
#undef STEP1
  return (int)hipGetLastError();
}
