// Native call path of the Python operators.
//
// Each function here does what its operator's Python wrapper does for
// arguments that need no conversion or copy: check them, allocate the output,
// find the workspace and call the C ABI on the current stream.  Anything else
// (a wrong shape or dtype, rows off their 16-byte boundary, a tensor subclass
// or a functorch wrapper, a workspace that is missing or too small, a size its
// query refuses) returns None before anything is allocated or launched, and the
// wrapper goes on in Python, where the copies, the workspace and the error
// messages are.  (So does an output that a dispatch mode gave no memory, before
// anything is launched.)  No state is kept here: workspaces are looked up in the
// package's own table on every call.  The GIL is released while the library
// launches, as ctypes does.
//
// Why: a decode step of a few microseconds was bound by its wrapper's Python
// (eager calls in a row, us a call: dense decode B1 8K 21, KIVI B4 16K 29, PQ
// B1 32K 26, Quest B1 32K 38, of which the launches themselves take 4 to 6; 8,
// 13, 10 and 18 from here).
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <initializer_list>

#include "../../../include/bytes_amd.h"

namespace {

using at::Tensor;

PyObject* g_ws = nullptr;              // {(device index, family): workspace tensor}

struct Refuse {};                      // the Python wrapper takes the call

inline void need(bool ok) {
  if (!ok) throw Refuse{};
}

// A plain CUDA tensor: no subclass, no functorch / functional / Python-key
// wrapper, no lazy negation or conjugation.
const Tensor& plain(const Tensor& t) {
  using K = c10::DispatchKey;
  static const c10::DispatchKeySet bad({K::Python, K::PythonTLSSnapshot, K::FuncTorchBatched, K::FuncTorchGradWrapper,
                                        K::Batched, K::Functionalize, K::Negative, K::Conjugate, K::ZeroTensor});
  need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(bad) && t.has_storage());
  return t;
}

const Tensor& tensor(PyObject* o) {
  need(THPVariable_CheckExact(o));
  return plain(THPVariable_Unpack(o));
}

long integer(PyObject* o) {
  need(PyLong_CheckExact(o));
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Refuse{};
  }
  need(v >= -0x7FFFFFFFL && v <= 0x7FFFFFFFL);
  return v;
}

double number(PyObject* o) {
  if (PyFloat_CheckExact(o)) return PyFloat_AS_DOUBLE(o);
  return (double)integer(o);
}

void same_device(const Tensor& a, std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts) need(t->device() == a.device());
}

bool shape(const Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s); }

uintptr_t addr(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()); }

// Unit stride on the last dim and every row on an `align`-byte boundary.
void rows(const Tensor& t, int align = 16) {
  need(t.stride(-1) == 1 && addr(t) % align == 0);
  const int64_t es = t.element_size();
  for (int64_t d = 0; d + 1 < t.dim(); ++d) need(t.size(d) <= 1 || t.stride(d) * es % align == 0);
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The family's workspace of the tensor's device, at least n bytes (held by the
// caller: another thread may replace the table's entry while the GIL is out).
Tensor workspace(const Tensor& t, const char* family, size_t n) {
  PyObject* key = Py_BuildValue("(is)", (int)t.device().index(), family);
  need(key != nullptr);
  PyObject* o = PyDict_GetItem(g_ws, key);       // borrowed; the table keeps every buffer it ever held
  Py_DECREF(key);
  need(o != nullptr);
  Tensor w = tensor(o);
  need((size_t)w.numel() >= n);
  return w;
}

// A new tensor on like's device.  Under a dispatch mode it may be one without
// memory, which the Python wrapper reports.
Tensor empty(const Tensor& like, at::IntArrayRef s, at::ScalarType dt) {
  Tensor t = at::empty(s, at::TensorOptions().dtype(dt).device(like.device()));
  plain(t);
  return t;
}
Tensor empty(const Tensor& like, std::initializer_list<int64_t> s, at::ScalarType dt) {
  return empty(like, at::IntArrayRef(s), dt);
}

struct Failed {
  int rc;
  const char* name;
};

// Calls the library without the GIL.  The arguments are evaluated before it is
// released (a tensor's data pointer may throw), and the library's C functions
// do not throw.
template <class... P, class... A>
void launch(const char* name, int (*f)(P...), A... args) {
  int rc;
  Py_BEGIN_ALLOW_THREADS rc = f(args...);
  Py_END_ALLOW_THREADS if (rc) throw Failed{rc, name};
}

const void* data(const Tensor& t) { return t.const_data_ptr(); }
int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return 0;
    case at::kHalf: return 1;
    case at::kFloat: return 2;
    default: throw Refuse{};
  }
}
constexpr at::ScalarType kF8 = at::kFloat8_e4m3fn;
bool head_dim(int64_t D) { return D == 64 || D == 128; }

struct QK {                            // q [B, Hq, 1, D] against keys [B, Hk, S, D]
  int64_t B, Hq, Hk, S, D;
};
QK qk(const Tensor& q, const Tensor& k, int64_t k_dim = -1) {
  need(q.dim() == 4 && k.dim() == 4 && q.scalar_type() == at::kBFloat16 && q.size(2) == 1);
  QK s{q.size(0), q.size(1), k.size(1), k.size(2), q.size(3)};
  need(k.size(0) == s.B && (k_dim < 0 ? k.size(3) : k_dim) == s.D && s.Hk > 0 && s.Hq % s.Hk == 0 && head_dim(s.D) &&
       s.S > 0 && s.S <= 0x7FFFFFFF && s.B > 0 && s.Hq > 0);
  same_device(q, {&k});
  rows(q);
  return s;
}

// ---- operators ----

Tensor dense(const Tensor& q, const Tensor& k, const Tensor& v, double scale, long chunk, bool fp8) {
  const QK s = qk(q, k);
  const auto dt = fp8 ? kF8 : at::kBFloat16;
  need(k.scalar_type() == dt && v.scalar_type() == dt && v.sizes() == k.sizes());
  same_device(q, {&v});
  rows(k);
  rows(v);
  size_t n = 0;
  need(bytes_decode_attn_bf16_workspace_size(s.B, s.Hq, s.Hk, s.S, s.D, chunk, &n) == 0);
  const Tensor w = workspace(q, "splitk", n);
  Tensor out = empty(q, {s.B, s.Hq, 1, s.D}, at::kBFloat16);
  void* st = stream_of(q);
  launch(fp8 ? "bytes_decode_attn_fp8" : "bytes_decode_attn_bf16", fp8 ? bytes_decode_attn_fp8 : bytes_decode_attn_bf16,
         data(q), data(k), data(v), out.mutable_data_ptr(), s.B, s.Hq, s.Hk, s.S, s.D, q.stride(0), q.stride(1),
         k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), out.stride(0), out.stride(1),
         (float)scale, (int)chunk, w.mutable_data_ptr(), (size_t)w.numel(), st);
  return out;
}

Tensor kivi(const Tensor& q, const Tensor& kq, const Tensor& ks, const Tensor& km, const Tensor& kr, const Tensor& vq,
            const Tensor& vs, const Tensor& vm, const Tensor& vr, long bits, double scale, bool own_scale, long chunk) {
  need(q.dim() == 4 && kr.dim() == 4 && vr.sizes() == kr.sizes() && kq.dim() == 4 && (bits == 2 || bits == 4));
  need(q.scalar_type() == at::kBFloat16 && kr.scalar_type() == at::kBFloat16 && vr.scalar_type() == at::kBFloat16);
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3), Hk = kr.size(1), R = kr.size(2);
  const int64_t fpi = 32 / bits, Sq = kq.size(3) * fpi;
  need(q.size(2) == 1 && Hk > 0 && Hq % Hk == 0 && head_dim(D) && kr.size(0) == B && kr.size(3) == D && Sq > 0 &&
       Sq % 32 == 0 && Sq + R <= 0x7FFFFFFF);
  need(shape(kq, {B, Hk, D, Sq / fpi}) && shape(ks, {B, Hk, D, Sq / 32}) && shape(km, {B, Hk, D, Sq / 32}) &&
       shape(vq, {B, Hk, Sq, D / fpi}) && shape(vs, {B, Hk, Sq, D / 32}) && shape(vm, {B, Hk, Sq, D / 32}));
  need(kq.scalar_type() == at::kInt && vq.scalar_type() == at::kInt);
  for (const Tensor* t : {&kq, &ks, &km, &vq, &vs, &vm}) need(t->is_contiguous());
  for (const Tensor* t : {&ks, &km, &vs, &vm}) need(t->scalar_type() == at::kHalf);
  same_device(q, {&kq, &ks, &km, &kr, &vq, &vs, &vm, &vr});
  rows(q);
  rows(kr);
  rows(vr);
  size_t n = 0;
  need(bytes_kivi_decode_workspace_size(B, Hq, Hk, Sq, R, D, bits, chunk, &n) == 0);
  const Tensor w = workspace(q, "splitk", n);
  Tensor out = empty(q, {B, Hq, 1, D}, at::kBFloat16);
  const float sc = (float)(own_scale ? scale : 1.0 / std::sqrt((double)D));
  void* st = stream_of(q);
  launch("bytes_kivi_decode_attn", bytes_kivi_decode_attn, data(q), data(kq), data(ks), data(km),
         R ? data(kr) : nullptr, data(vq), data(vs), data(vm), R ? data(vr) : nullptr, out.mutable_data_ptr(), B, Hq,
         Hk, Sq, R, D, bits, q.stride(0), q.stride(1), kr.stride(0), kr.stride(1), kr.stride(2), vr.stride(0),
         vr.stride(1), vr.stride(2), out.stride(0), out.stride(1), sc, (int)chunk, w.mutable_data_ptr(),
         (size_t)w.numel(), st);
  return out;
}

PyObject* kivi_pack(const Tensor& x, long group, long bits) {
  need((bits == 2 || bits == 4) && x.dim() >= 1 && x.is_contiguous() && x.numel() > 0 && group > 0);
  const int64_t T = x.size(-1), fpi = 32 / bits;
  need(T % group == 0 && group % fpi == 0 && T <= 0x7FFFFFFF);
  const int dt = dtype_code(x);
  auto lead = x.sizes().vec();
  lead.back() = T / fpi;
  Tensor code = empty(x, lead, at::kInt);
  lead.back() = T / group;
  Tensor scale = empty(x, lead, at::kHalf), mn = empty(x, lead, at::kHalf);
  void* st = stream_of(x);
  launch("bytes_kivi_quantize_pack", bytes_kivi_quantize_pack, data(x), dt, x.numel() / T, T, T, group, bits,
         code.mutable_data_ptr(), scale.mutable_data_ptr(), mn.mutable_data_ptr(), st);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(code), THPVariable_Wrap(scale), THPVariable_Wrap(mn));
}

struct Codebook {
  int64_t M, K, sh;
};
Codebook codebook(const Tensor& cb, int64_t Hk) {          // fp16, shared or per KV head
  need((cb.dim() == 3 || (cb.dim() == 4 && cb.size(0) == Hk)) && cb.scalar_type() == at::kHalf && cb.is_contiguous());
  const int64_t M = cb.size(-3), K = cb.size(-2);
  need(cb.size(-1) == 8 && K > 0 && K <= 256 && K % 4 == 0);
  return {M, K, cb.dim() == 4 ? M * K * 8 : 0};
}
void codes(const Tensor& c, int64_t M) {
  need(c.dim() == 4 && c.scalar_type() == at::kByte && c.size(3) == M && c.stride(3) == 1 && c.stride(2) == M &&
       addr(c) % 16 == 0);
}

Tensor pq_fused(const Tensor& q, const Tensor& kcb, const Tensor& ki, const Tensor& vi, const Tensor& vcb, double scale,
                long chunk) {
  need(q.dim() == 4 && ki.dim() == 4 && q.scalar_type() == at::kBFloat16 && q.size(2) == 1);
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3), Hk = ki.size(1), S = ki.size(2), M = ki.size(3);
  need(ki.size(0) == B && M * 8 == D && Hk > 0 && Hq % Hk == 0 && S > 0 && S <= 0x7FFFFFFF && head_dim(D));
  codes(ki, M);
  codes(vi, M);
  need(shape(vi, {B, Hk, S, M}));
  const Codebook k = codebook(kcb, Hk), v = codebook(vcb, Hk);
  need(k.M == M && v.M == M && k.K == v.K);
  same_device(q, {&kcb, &ki, &vi, &vcb});
  rows(q);
  size_t n = 0;
  need(bytes_pq_decode_workspace_size(B, Hq, Hk, S, D, chunk, &n) == 0);
  const Tensor w = workspace(q, "splitk", n);
  Tensor out = empty(q, {B, Hq, 1, D}, at::kHalf);         // the value codebook's dtype
  void* st = stream_of(q);
  launch("bytes_pq_decode_attn", bytes_pq_decode_attn, 3, nullptr, data(q), data(kcb), data(ki), data(vi), data(vcb),
         nullptr, out.mutable_data_ptr(), 1, B, Hq, Hk, S, D, k.K, 0, 0, q.stride(0), q.stride(1), k.sh, ki.stride(0),
         ki.stride(1), ki.stride(2), vi.stride(0), vi.stride(1), vi.stride(2), v.sh, 0, 0, 0, out.stride(0),
         out.stride(1), (float)scale, (int)chunk, w.mutable_data_ptr(), (size_t)w.numel(), st);
  return out;
}

// LUT + outlier scores, dense values; paged where bt and cl are given (both or neither).
Tensor pq_asym(const Tensor& lut, const Tensor& ki, const Tensor& ko, const Tensor& qo, const Tensor& v,
               const Tensor* bt, const Tensor* cl, long block_size, long chunk) {
  need(lut.dim() == 4 && ki.dim() == 4 && ko.dim() == 4 && qo.dim() == 3 && lut.scalar_type() == at::kFloat);
  const int64_t B = lut.size(0), Hq = lut.size(1), M = lut.size(2), K = lut.size(3);
  const int64_t lead = ki.size(0), Hk = ki.size(1), bs = ki.size(2), C = ko.size(3), D = M * 8;
  need(Hk > 0 && Hq % Hk == 0 && B > 0 && bs > 0 && lead > 0 && head_dim(D) && K > 0 && K <= 256 && K % 4 == 0);
  need(lut.stride(3) == 1 && lut.stride(2) == K && addr(lut) % 16 == 0);
  codes(ki, M);
  need(shape(ko, {lead, Hk, bs, C}) && shape(qo, {B, Hq, C}) && C > 0 && C <= 16 && ko.stride(3) == 1 &&
       qo.stride(2) == 1);
  const bool f8 = v.scalar_type() == kF8;
  need((f8 || v.scalar_type() == at::kBFloat16) && shape(v, {lead, Hk, bs, D}));
  rows(v);
  same_device(lut, {&ki, &ko, &qo, &v});
  int64_t S = bs;
  if (bt) {
    need(bs == block_size && bt->dim() == 2 && bt->size(0) == B && bt->scalar_type() == at::kInt &&
         bt->stride(1) == 1 && shape(*cl, {B}) && cl->scalar_type() == at::kInt && cl->is_contiguous());
    same_device(lut, {bt, cl});
    S = bt->size(1) * bs;
  } else {
    need(lead == B);
  }
  need(S > 0 && S <= 0x7FFFFFFF);
  size_t n = 0;
  need(bytes_pq_decode_workspace_size(B, Hq, Hk, S, D, chunk, &n) == 0);
  const Tensor w = workspace(lut, "splitk", n);
  const int kd = dtype_code(ko), qd = dtype_code(qo);
  Tensor out = empty(lut, {B, Hq, 1, D}, at::kBFloat16);
  void* st = stream_of(lut);
  launch("bytes_pq_lut_decode_attn", bytes_pq_lut_decode_attn, data(lut), lut.stride(0), lut.stride(1), data(ki),
         ki.stride(0), ki.stride(1), ki.stride(2), nullptr, 0, 0, 0, nullptr, 0, data(v), f8, v.stride(0), v.stride(1),
         v.stride(2), data(ko), kd, ko.stride(0), ko.stride(1), ko.stride(2), data(qo), qd, qo.stride(0), qo.stride(1),
         (int)C, bt ? bt->const_data_ptr<int>() : nullptr, bt ? bt->stride(0) : 0,
         cl ? cl->const_data_ptr<int>() : nullptr, bt ? (int)bs : 0, bt ? (int)lead : 0, out.mutable_data_ptr(), 0,
         out.stride(0), out.stride(1), B, Hq, Hk, S, D, K, 1.0f, (int)chunk, w.mutable_data_ptr(), (size_t)w.numel(),
         st);
  return out;
}

Tensor pq_encode(const Tensor& x, const Tensor& cb) {
  const int xd = dtype_code(x);
  const bool f32 = cb.scalar_type() == at::kFloat;
  need((f32 || cb.scalar_type() == at::kHalf) && (cb.dim() == 3 || cb.dim() == 4) && cb.is_contiguous() &&
       x.is_contiguous() && x.dim() >= 2 && x.numel() > 0);
  same_device(x, {&cb});
  const int64_t D = x.size(-1), M = cb.size(-3), K = cb.size(-2), heads = cb.dim() == 4 ? cb.size(0) : 1;
  need(cb.size(-1) == 8 && M * 8 == D && M <= 16 && K > 0 && K <= 256 && (cb.dim() == 3 || x.size(0) == heads));
  auto s = x.sizes().vec();
  s.back() = M;
  const int64_t n = x.numel() / D;
  Tensor idx = empty(x, s, at::kByte);
  void* st = stream_of(x);
  launch("bytes_pq_encode", bytes_pq_encode, data(x), xd, heads, n / heads, D, D, data(cb), f32,
         cb.dim() == 4 ? M * K * 8 : 0, K, idx.mutable_data_ptr(), st);
  return idx;
}

// A score launch whose arguments have been checked.
struct Score {
  QK s;
  int mode;
  int64_t m0 = 0, m1 = 0, m2 = 0;
};

// Keys k (bf16, fp8, or packed codes with scale / zero) for the score kernel.
Score score_of(const Tensor& q, const Tensor& k, const Tensor* sc, const Tensor* zr, long bits, bool group_sum) {
  Score r;
  if (sc) {
    need(zr && (bits == 4 || bits == 2) && k.dim() == 4 && k.scalar_type() == at::kByte && k.size(3) * 8 % bits == 0);
    r.s = qk(q, k, k.size(3) * 8 / bits);
    for (const Tensor* t : {sc, zr}) {
      need(t->scalar_type() == at::kBFloat16 && shape(*t, {r.s.B, r.s.Hk, r.s.S, r.s.D / 32}));
      rows(*t, (int)(r.s.D / 32 * 2));
    }
    need(sc->strides() == zr->strides());
    same_device(q, {sc, zr});
    r.mode = bits == 4 ? 2 : 3;
    r.m0 = sc->stride(0), r.m1 = sc->stride(1), r.m2 = sc->stride(2);
  } else {
    need(k.scalar_type() == at::kBFloat16 || k.scalar_type() == kF8);
    r.s = qk(q, k);
    r.mode = k.scalar_type() == kF8;
  }
  rows(k);
  need(!group_sum || r.s.Hq / r.s.Hk <= 16);
  return r;
}

// Scores into out [B, H, S]; hist: a top-k workspace whose histogram region
// also counts them.
void score_into(const Score& r, const Tensor& q, const Tensor& k, const Tensor* sc, const Tensor* zr, double scaling,
                bool group_sum, const Tensor& out, void* hist) {
  const QK& s = r.s;
  need(out.scalar_type() == at::kFloat && shape(out, {s.B, group_sum ? s.Hk : s.Hq, s.S}) && out.stride(2) == 1);
  void* st = stream_of(q);
  launch("bytes_sparse_score", bytes_sparse_score, data(q), data(k), r.mode, sc ? data(*sc) : nullptr,
         sc ? data(*zr) : nullptr, out.mutable_data_ptr(), s.B, s.Hq, s.Hk, s.S, s.D, group_sum, q.stride(0),
         q.stride(1), k.stride(0), k.stride(1), k.stride(2), r.m0, r.m1, r.m2, out.stride(0), out.stride(1),
         (float)scaling, hist, st);
}

void score_rows(const Tensor& q, const Tensor& k, double scaling, const Tensor& out) {
  score_into(score_of(q, k, nullptr, nullptr, 0, false), q, k, nullptr, nullptr, scaling, false, out, nullptr);
}

Tensor topk_workspace(const Tensor& t, int64_t rows_, int64_t n, int64_t k) {
  size_t bytes = 0;
  need(bytes_topk_workspace_size(rows_, (int)n, (int)k, &bytes) == 0);
  return workspace(t, "topk", bytes);
}

// Contiguous fp32 scores [.., n].  counted: the workspace whose histogram region
// the score kernel has counted them into.
Tensor topk_of(const Tensor& s, long k, bool sorted, const Tensor* counted) {
  need(s.scalar_type() == at::kFloat && s.dim() >= 1 && s.is_contiguous() && s.numel() > 0);
  const int64_t n = s.size(-1), r = s.numel() / n;
  need(k >= 1 && k <= n && n <= 0x7FFFFFFF);
  const Tensor w = counted ? *counted : topk_workspace(s, r, n, k);
  auto shp = s.sizes().vec();
  shp.back() = k;
  Tensor out = empty(s, shp, at::kInt);
  void* st = stream_of(s);
  launch("bytes_topk", bytes_topk, data(s), r, (int)n, n, (int)k, sorted, counted != nullptr, out.mutable_data_ptr(), k,
         w.mutable_data_ptr(), (size_t)w.numel(), st);
  return out;
}

struct Kv {
  QK s;
  bool f8;
};
Kv kv(const Tensor& q, const Tensor& k, const Tensor& v) {
  const QK s = qk(q, k);
  const bool f8 = k.scalar_type() == kF8;
  need((f8 || k.scalar_type() == at::kBFloat16) && v.scalar_type() == k.scalar_type() && v.sizes() == k.sizes());
  same_device(q, {&v});
  rows(k);
  rows(v);
  return {s, f8};
}

Tensor gather_workspace(const Tensor& q, const QK& s, int64_t kb, bool per_head, long chunk) {
  need(kb > 0 && kb <= 0x7FFFFFFF);
  size_t n = 0;
  need(bytes_gather_attn_workspace_size(s.B, s.Hq, s.Hk, (int)kb, s.D, per_head, (int)chunk, &n) == 0);
  return workspace(q, "splitk", n);
}

// limit -1: every row.
Tensor gather(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& idx, double scaling, long chunk,
              long page, long limit) {
  const Kv x = kv(q, k, v);
  const QK& s = x.s;
  if (limit == -1) limit = s.S;
  need(idx.dim() == 3 && idx.size(0) == s.B && (idx.size(1) == s.Hq || idx.size(1) == s.Hk) && idx.size(2) > 0 &&
       idx.scalar_type() == at::kInt && idx.stride(2) == 1 && page >= 1);
  need(limit >= 0 && limit <= s.S);
  same_device(q, {&idx});
  const bool per_head = idx.size(1) == s.Hq;
  const int64_t kb = idx.size(2) * page;
  const Tensor w = gather_workspace(q, s, kb, per_head, chunk);
  Tensor out = empty(q, {s.B, s.Hq, 1, s.D}, at::kBFloat16);
  void* st = stream_of(q);
  launch("bytes_gather_attn", bytes_gather_attn, data(q), data(k), data(v), x.f8, data(idx), out.mutable_data_ptr(),
         s.B, s.Hq, s.Hk, s.S, s.D, (int)kb, per_head, page == 1 ? 0 : (int)page, (int)limit, q.stride(0), q.stride(1),
         k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), idx.stride(0), idx.stride(1),
         out.stride(0), out.stride(1), (float)scaling, (int)chunk, w.mutable_data_ptr(), (size_t)w.numel(), st);
  return out;
}

// What every launch of a composite needs is looked at before its first one and
// before anything is allocated.
Tensor sparse_decode(const Tensor& q, const Tensor& ks, const Tensor* sc, const Tensor* zr, const Tensor& k,
                     const Tensor& v, double frac, double scaling, long bits) {
  need(bits == 16 ? ks.scalar_type() == at::kBFloat16
                  : bits == 8 ? ks.scalar_type() == kF8 : (bits == 4 || bits == 2) && sc);
  if (bits >= 8) sc = zr = nullptr;
  const Kv x = kv(q, k, v);
  const QK& s = x.s;
  need(ks.dim() == 4 && ks.size(2) == s.S && ks.size(1) == s.Hk);
  const double want = std::nearbyint(frac * (double)s.S);  // round half to even, as Python's round
  need(want <= (double)s.S);
  const int64_t kb = want < 1 ? 1 : (int64_t)want;
  const Score sco = score_of(q, ks, sc, zr, bits, false);
  topk_workspace(q, s.B * s.Hq, s.S, kb);
  gather_workspace(q, s, kb, true, 0);
  Tensor scores = empty(q, {s.B, s.Hq, s.S}, at::kFloat);
  score_into(sco, q, ks, sc, zr, scaling, false, scores, nullptr);
  return gather(q, k, v, topk_of(scores, kb, false, nullptr), scaling, 0, 1, -1);
}

PyObject* token_topk(const Tensor& q, const Tensor& k, const Tensor& v, long kb, double scaling, const Tensor& ks,
                     const Tensor* sc, const Tensor* zr, long bits) {
  const Kv x = kv(q, k, v);
  const QK& s = x.s;
  need(s.Hq > s.Hk);                             // idx [B, Hk, kb] is then one list per KV head
  need(ks.dim() == 4 && ks.size(2) == s.S && ks.size(1) == s.Hk && (sc || ks.sizes() == k.sizes()));
  need((ks.scalar_type() == at::kByte) == (sc != nullptr) && kb >= 1 && kb <= s.S);
  const Score sco = score_of(q, ks, sc, zr, bits, true);
  const bool hist = s.B * s.Hk <= 1024;          // rows of the workspace's histogram region
  const Tensor w = topk_workspace(q, s.B * s.Hk, s.S, kb);
  gather_workspace(q, s, kb, false, 0);
  Tensor scores = empty(q, {s.B, s.Hk, s.S}, at::kFloat);
  score_into(sco, q, ks, sc, zr, scaling, true, scores, hist ? w.mutable_data_ptr() : nullptr);
  Tensor idx = topk_of(scores, kb, false, hist ? &w : nullptr);
  Tensor out = gather(q, k, v, idx, scaling, 0, 1, -1);
  return Py_BuildValue("(NN)", THPVariable_Wrap(out), THPVariable_Wrap(idx));
}

Tensor quest(const Tensor& q, const Tensor& k, const Tensor& v, long kb, double scaling, long page, const Tensor& kmin,
             const Tensor& kmax, long pos, long local_w) {
  const Kv x = kv(q, k, v);
  const QK& s = x.s;
  need(kmin.dim() == 4 && kmin.sizes() == kmax.sizes() && kmin.scalar_type() == at::kBFloat16 &&
       kmax.scalar_type() == at::kBFloat16 && kmin.is_contiguous() && kmax.is_contiguous());
  const int64_t np = kmin.size(2);
  need(kmin.size(0) == s.B && kmin.size(1) == s.Hk && kmin.size(3) == s.D && np > 0 && np <= 4096 && page >= 1);
  need(pos >= 0 && pos + 1 <= s.S && kb > 0);
  same_device(q, {&kmin, &kmax});
  const int64_t pages = (kb + page - 1) / page, npick = pages < np ? pages : np;
  const Tensor w = gather_workspace(q, s, npick * page, true, 0);
  Tensor bound = empty(q, {s.B, s.Hq, np}, at::kFloat);
  Tensor out = empty(q, {s.B, s.Hq, 1, s.D}, at::kBFloat16);
  void* st = stream_of(q);
  launch("bytes_quest_page_scores", bytes_quest_page_scores, data(q), data(kmin), data(kmax), bound.mutable_data_ptr(),
         s.B, s.Hq, s.Hk, (int)np, s.D, (int)page, (int)pos, (int)local_w, q.stride(0), q.stride(1), bound.stride(0),
         bound.stride(1), (float)scaling, st);
  launch("bytes_quest_gather_attn", bytes_quest_gather_attn, data(q), data(k), data(v), x.f8, data(bound),
         bound.stride(0), bound.stride(1), (int)np, (int)npick, out.mutable_data_ptr(), s.B, s.Hq, s.Hk, s.S, s.D,
         (int)page, (int)pos + 1, q.stride(0), q.stride(1), k.stride(0), k.stride(1), k.stride(2), v.stride(0),
         v.stride(1), v.stride(2), out.stride(0), out.stride(1), (float)scaling, 0, w.mutable_data_ptr(),
         (size_t)w.numel(), st);
  return out;
}

// ---- bindings ----

template <class F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (const Refuse&) {
    Py_RETURN_NONE;
  } catch (const Failed& e) {
    const char* m = bytes_error_string(e.rc);
    PyErr_Format(PyExc_RuntimeError, "bytes_amd.%s: %s (hipError %d)", e.name, m ? m : "error", e.rc);
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());   // as torch's own functions report it
  }
  return nullptr;
}

long row_limit(PyObject* o) {
  const long v = integer(o);
  need(v >= 0);
  return v;
}

const Tensor* optional(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }

#define BIND(NAME, N, EXPR)                                                                     \
  PyObject* py_##NAME(PyObject*, PyObject* const* a, Py_ssize_t n) {                            \
    return guarded([&]() -> PyObject* {                                                         \
      need(n == N);                                                                             \
      return EXPR;                                                                              \
    });                                                                                         \
  }
#define WRAP(X) THPVariable_Wrap(X)

BIND(dense, 6, WRAP(dense(tensor(a[0]), tensor(a[1]), tensor(a[2]), number(a[3]), integer(a[4]), a[5] == Py_True)))
BIND(kivi, 13, (need(integer(a[10]) == 32),
                WRAP(kivi(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), tensor(a[5]),
                          tensor(a[6]), tensor(a[7]), tensor(a[8]), integer(a[9]), a[11] == Py_None ? 0.0 : number(a[11]),
                          a[11] != Py_None, integer(a[12])))))
BIND(kivi_pack, 3, kivi_pack(tensor(a[0]), integer(a[1]), integer(a[2])))
BIND(pq_fused, 7, WRAP(pq_fused(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), number(a[5]),
                                integer(a[6]))))
BIND(pq_asym, 6, WRAP(pq_asym(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), nullptr, nullptr, 0,
                              integer(a[5]))))
BIND(pq_paged, 9, WRAP(pq_asym(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4]), &tensor(a[5]),
                               &tensor(a[6]), integer(a[7]), integer(a[8]))))
BIND(pq_encode, 2, WRAP(pq_encode(tensor(a[0]), tensor(a[1]))))
BIND(score_into, 4, (score_rows(tensor(a[0]), tensor(a[1]), number(a[2]), tensor(a[3])), Py_NewRef(a[3])))
BIND(topk, 3, WRAP(topk_of(tensor(a[0]), integer(a[1]), a[2] == Py_True, nullptr)))
BIND(gather, 8, WRAP(gather(tensor(a[0]), tensor(a[1]), tensor(a[2]), tensor(a[3]), number(a[4]), integer(a[5]),
                            integer(a[6]), a[7] == Py_None ? -1 : row_limit(a[7]))))
BIND(sparse_decode, 9, WRAP(sparse_decode(tensor(a[0]), tensor(a[1]), optional(a[2]), optional(a[3]), tensor(a[4]),
                                          tensor(a[5]), number(a[6]), number(a[7]), integer(a[8]))))
BIND(token_topk, 9, token_topk(tensor(a[0]), tensor(a[1]), tensor(a[2]), integer(a[3]), number(a[4]), tensor(a[5]),
                               optional(a[6]), optional(a[7]), a[8] == Py_None ? 0 : integer(a[8])))
BIND(quest, 10, WRAP(quest(tensor(a[0]), tensor(a[1]), tensor(a[2]), integer(a[3]), number(a[4]), integer(a[5]),
                           tensor(a[6]), tensor(a[7]), integer(a[8]), integer(a[9]))))

PyObject* py_set_workspaces(PyObject*, PyObject* d) {
  if (!PyDict_Check(d)) {
    PyErr_SetString(PyExc_TypeError, "expected the workspace table");
    return nullptr;
  }
  Py_INCREF(d);
  Py_XSETREF(g_ws, d);
  Py_RETURN_NONE;
}

#define METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(dense),     METHOD(kivi),   METHOD(kivi_pack), METHOD(pq_fused),
                         METHOD(pq_asym),   METHOD(pq_paged), METHOD(pq_encode), METHOD(score_into), METHOD(topk),
                         METHOD(gather),    METHOD(sparse_decode), METHOD(token_topk), METHOD(quest),
                         {"set_workspaces", py_set_workspaces, METH_O, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Native call path of the operators.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
