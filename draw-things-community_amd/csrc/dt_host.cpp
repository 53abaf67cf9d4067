// The Python operators' way to the C ABI: argument blocks filled from torch tensors without an interpreter step for every
// pointer and stride.  Host code only.
//
// What bounds it: calls of a few rows take the GPU 8 .. 19 us, and a chain of short launches (a UNet block) waits for the
// host, which spent most of a call on one interpreter step after the other (us of the host a call, through Python / from here: 1 x 3072 ->
// 6 x 3072 q8p 23.1 / 8.5, 231 x 1000 -> 1001 13.9 / 4.7, attention with norms and rotation 27.7 / 8.9, a UNet block of thirteen operators 249 /
// 109); what is left is the launch, 4 us, and torch's allocator.
//
// Every function returns None for whatever it does not recognise at once -- subclasses of Tensor, views that need a copy,
// wrong shapes or types -- before it has enqueued anything: the caller then goes the way through Python, which copies or
// names what is wrong.  Nothing is kept from one call for the next.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "../../include/dt_hip.h"

namespace {

constexpr int64_t kRowsMax = 64;  // rows up to which the library streams the weights and takes no scratch

struct Fallback {};  // not a call for this file
struct Raised {};    // a Python exception is set

PyObject* g_qx = nullptr;    // the classes QxTensor, HeadEpilogue and DensePost
PyObject* g_epi = nullptr;
PyObject* g_post = nullptr;
#define NAMES(X) X(data) X(qbits) X(nib) X(shape) X(gamma) X(rot) X(rot_pos0) X(eps) X(head_dim) X(activation) X(gate) X(residual) \
  X(keep_output) X(scale) X(addend) X(multiplicand)
#define DECLARE(n) PyObject* s_##n = nullptr;
NAMES(DECLARE)
#undef DECLARE

// An owned reference, dropped at the end of the scope.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* o) : p(o) {
    if (!p) {
      PyErr_Clear();
      throw Fallback{};
    }
  }
  ~Ref() { Py_DECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};
Ref attr(PyObject* o, PyObject* name) { return Ref(PyObject_GetAttr(o, name)); }
int64_t as_int(PyObject* o) {
  if (!PyLong_CheckExact(o)) throw Fallback{};
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Fallback{};
  }
  return v;
}
float as_float(PyObject* o) {
  if (PyFloat_CheckExact(o)) return (float)PyFloat_AS_DOUBLE(o);
  return (float)as_int(o);
}
int32_t as_int32(PyObject* o) {
  const int64_t v = as_int(o);
  if (v < INT32_MIN || v > INT32_MAX) throw Fallback{};
  return (int32_t)v;
}

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw Fallback{};
  return THPVariable_Unpack(o);
}
const at::Tensor& cuda(PyObject* o, at::ScalarType type) {
  const at::Tensor& t = tensor(o);
  if (!t.is_cuda() || t.scalar_type() != type) throw Fallback{};
  return t;
}
const at::Tensor& half(PyObject* o) { return cuda(o, at::kHalf); }
template <typename T>
T* ptr(const at::Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}
const uint16_t* half_or_null(PyObject* o) { return o == Py_None ? nullptr : ptr<const uint16_t>(half(o)); }

// A list or tuple.
struct Seq {
  PyObject* o;
  Py_ssize_t n;
  explicit Seq(PyObject* s) : o(s), n(0) {
    if (!PyList_CheckExact(s) && !PyTuple_CheckExact(s)) throw Fallback{};
    n = PySequence_Fast_GET_SIZE(s);
  }
  PyObject* operator[](Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(o, i); }
};

// t as an [M, N] matrix with contiguous rows: its row stride.
int64_t matrix(const at::Tensor& t, int64_t M, int64_t N) {
  if (t.dim() == 2) {
    if (t.size(0) != M || t.size(1) != N || t.stride(1) != 1) throw Fallback{};
    return t.stride(0);
  }
  if (t.numel() != M * N || t.dim() < 1 || t.size(-1) != N || !t.is_contiguous()) throw Fallback{};
  return N;
}

struct Problem {
  const at::Tensor* x = nullptr;
  int64_t M = 0, K = 0;
  std::vector<dt_qx_weight> w;
  std::vector<const uint16_t*> bias;
  std::vector<uint16_t*> y;
  std::vector<int64_t> ldy;
  std::vector<dt_head_epilogue> epi;
  std::vector<dt_dense_post> post;
  std::vector<at::Tensor> outs;  // undefined: only accumulates into a residual
};

void epilogue(PyObject* o, int64_t M, dt_head_epilogue& e) {
  e = dt_head_epilogue{};
  e.head_dim = 128;
  if (o == Py_None) return;
  if ((PyObject*)Py_TYPE(o) != g_epi) throw Fallback{};
  const Ref gamma = attr(o, s_gamma), rot = attr(o, s_rot), pos = attr(o, s_rot_pos0), eps = attr(o, s_eps), dim = attr(o, s_head_dim);
  e.rot_pos0 = as_int(pos.p);
  e.eps = as_float(eps.p);
  e.head_dim = as_int32(dim.p);
  if (rot.p != Py_None) {
    const at::Tensor& t = half(rot.p);
    if (t.dim() != 2 || t.size(1) != e.head_dim || !t.is_contiguous() || t.size(0) < e.rot_pos0 + M) throw Fallback{};
    e.rot = ptr<const uint16_t>(t);
  }
  if (gamma.p != Py_None) {
    const at::Tensor& t = half(gamma.p);
    if (t.numel() != e.head_dim || !t.is_contiguous()) throw Fallback{};
    e.gamma = ptr<const uint16_t>(t);
  }
}

// Returns whether the output is kept.
bool post(PyObject* o, int64_t M, int64_t N, dt_dense_post& d) {
  d = dt_dense_post{};
  d.scale = 1.0f;
  if (o == Py_None) return true;
  if ((PyObject*)Py_TYPE(o) != g_post) throw Fallback{};
  const Ref act = attr(o, s_activation), gate = attr(o, s_gate), res = attr(o, s_residual), keep = attr(o, s_keep_output),
            scale = attr(o, s_scale), add = attr(o, s_addend), mul = attr(o, s_multiplicand);
  d.activation = as_int32(act.p);
  d.scale = as_float(scale.p);
  if (d.scale == 0.0f || (keep.p != Py_True && keep.p != Py_False)) throw Fallback{};
  if (gate.p != Py_None) {
    const at::Tensor& t = tensor(gate.p);
    if (!t.is_cuda() || t.numel() != N || !t.is_contiguous()) throw Fallback{};
    if (t.scalar_type() == at::kFloat) d.gate_f32 = ptr<const float>(t);
    else if (t.scalar_type() == at::kHalf) d.gate = ptr<const uint16_t>(t);
    else throw Fallback{};
  }
  if (res.p != Py_None) {
    const at::Tensor& t = cuda(res.p, at::kFloat);
    d.ld_residual = matrix(t, M, N);
    d.residual = ptr<float>(t);
  }
  if (add.p != Py_None) {
    const at::Tensor& t = half(add.p);
    d.ld_addend = matrix(t, M, N);
    d.addend = ptr<const uint16_t>(t);
  }
  if (mul.p != Py_None) {
    const at::Tensor& t = half(mul.p);
    d.ld_multiplicand = matrix(t, M, N);
    d.multiplicand = ptr<const uint16_t>(t);
  }
  return !d.residual || keep.p == Py_True;
}

// (x, weights, biases, outs, epilogues, posts)
void read_problem(PyObject* o, Problem& p) {
  if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 6) throw Fallback{};
  const at::Tensor& x = half(PyTuple_GET_ITEM(o, 0));
  p.x = &x;
  if (x.dim() < 1 || x.numel() == 0) throw Fallback{};
  p.K = x.size(-1);
  p.M = x.numel() / p.K;
  if (x.dim() == 2 ? x.stride(1) != 1 : !x.is_contiguous()) throw Fallback{};
  const Seq ws(PyTuple_GET_ITEM(o, 1)), bs(PyTuple_GET_ITEM(o, 2));
  const size_t n = (size_t)ws.n;
  if (n == 0 || bs.n > ws.n) throw Fallback{};
  p.w.resize(n);
  p.bias.assign(n, nullptr);
  p.y.assign(n, nullptr);
  p.ldy.resize(n);
  p.outs.resize(n);
  for (size_t i = 0; i < n; i++) {
    PyObject* const w = ws[(Py_ssize_t)i];
    if ((PyObject*)Py_TYPE(w) != g_qx) throw Fallback{};
    const Ref data = attr(w, s_data), qbits = attr(w, s_qbits), nib = attr(w, s_nib), shape = attr(w, s_shape);
    if (!PyTuple_Check(shape.p) || PyTuple_GET_SIZE(shape.p) != 2) throw Fallback{};
    const int64_t N = as_int(PyTuple_GET_ITEM(shape.p, 0));
    if (as_int(PyTuple_GET_ITEM(shape.p, 1)) != p.K || N < 0) throw Fallback{};
    p.w[i] = dt_qx_weight{ptr<const void>(tensor(data.p)), as_int32(qbits.p), as_int32(nib.p), N * p.K};
    p.ldy[i] = N;
  }
  for (Py_ssize_t i = 0; i < bs.n; i++) p.bias[(size_t)i] = half_or_null(bs[i]);
  PyObject *const epis = PyTuple_GET_ITEM(o, 4), *const posts = PyTuple_GET_ITEM(o, 5);
  if (epis != Py_None) {
    const Seq s(epis);
    if (s.n > ws.n) throw Fallback{};
    p.epi.resize(n);
    for (size_t i = 0; i < n; i++) epilogue((Py_ssize_t)i < s.n ? s[(Py_ssize_t)i] : Py_None, p.M, p.epi[i]);
  }
  std::vector<bool> keep(n, true);
  if (posts != Py_None) {
    const Seq s(posts);
    if (s.n > ws.n) throw Fallback{};
    p.post.resize(n);
    for (size_t i = 0; i < n; i++) keep[i] = post((Py_ssize_t)i < s.n ? s[(Py_ssize_t)i] : Py_None, p.M, p.ldy[i], p.post[i]);
  }
  if (PyObject* const given = PyTuple_GET_ITEM(o, 3); given != Py_None) {
    const Seq s(given);
    if (s.n != ws.n) throw Fallback{};
    for (size_t i = 0; i < n; i++) {
      const at::Tensor& t = tensor(s[(Py_ssize_t)i]);
      if (t.dim() < 1) throw Fallback{};
      p.ldy[i] = t.stride(0);
      if (!keep[i]) continue;
      p.y[i] = ptr<uint16_t>(t);
      // (in the leading shape of x where that takes no copy)
      if (t.size(0) != p.M || !t.is_contiguous()) {
        p.outs[i] = t;
      } else {
        at::DimVector sizes(x.sizes().begin(), x.sizes().end());
        sizes.back() = t.size(-1);
        p.outs[i] = t.reshape(sizes);
      }
    }
  } else {
    at::DimVector sizes(x.sizes().begin(), x.sizes().end());
    for (size_t i = 0; i < n; i++) {
      if (!keep[i]) continue;
      sizes.back() = p.ldy[i];
      p.outs[i] = at::empty(sizes, x.options());
      p.y[i] = ptr<uint16_t>(p.outs[i]);
    }
  }
}

// Scratch memory as the package's own function for it hands it out: get(like, need, least) -> (what holds it, address, bytes).
struct Scratch {
  PyObject* held = nullptr;
  void* at = nullptr;
  size_t bytes = 0;
  void ask(PyObject* get, PyObject* like, size_t need, size_t least) {
    if (need == 0) return;
    const Ref a(PyLong_FromSize_t(need)), b(PyLong_FromSize_t(least));
    PyObject* const args[3] = {like, a.p, b.p};
    held = PyObject_Vectorcall(get, args, 3, nullptr);
    if (!held) throw Raised{};
    if (!PyTuple_CheckExact(held) || PyTuple_GET_SIZE(held) != 3) throw Fallback{};
    if (PyObject* const p = PyTuple_GET_ITEM(held, 1); p != Py_None) at = reinterpret_cast<void*>(as_int(p));
    bytes = (size_t)as_int(PyTuple_GET_ITEM(held, 2));
  }
  Scratch() = default;
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  ~Scratch() { Py_XDECREF(held); }
};

dt_stream current_stream() { return (dt_stream)c10::hip::getCurrentHIPStream().stream(); }

// dense(problems, flags, scratch): the outputs of each problem, or a status that is not DT_OK as an int (kWithScratch less where it is that of
// the entry point with scratch), or None.
constexpr long kWithScratch = 1000;
PyObject* dense(Py_ssize_t n_args, PyObject* const* args) {
  if (n_args != 3) throw Fallback{};
  const Seq problems(args[0]);
  const uint32_t flags = (uint32_t)as_int32(args[1]);
  std::vector<Problem> ps((size_t)problems.n);
  std::vector<dt_dense_group> groups(ps.size());
  bool many = false;
  for (size_t i = 0; i < ps.size(); i++) {
    Problem& p = ps[i];
    read_problem(problems[(Py_ssize_t)i], p);
    many = many || p.M > kRowsMax;
    groups[i] = dt_dense_group{p.M, p.K, ptr<const uint16_t>(*p.x), p.x->dim() == 2 && p.M > 1 ? p.x->stride(0) : p.K, p.w.data(),
                               (int32_t)p.w.size(), p.bias.data(), p.y.data(), p.ldy.data(), p.epi.empty() ? nullptr : p.epi.data(),
                               p.post.empty() ? nullptr : p.post.data()};
  }
  if (ps.empty()) throw Fallback{};
  const int32_t n = (int32_t)groups.size();
  // (the scratch for copies of the weights; where the device is too full for them, that for cuts, which take less)
  Scratch copies, cuts;
  PyObject* const like = PyTuple_GET_ITEM(problems[0], 0);
  const size_t need = many ? dt_dense_scratch_bytes(n, groups.data()) : 0;
  copies.ask(args[2], like, need, 0);
  if (need && !copies.bytes) cuts.ask(args[2], like, dt_dense_workspace_bytes(n, groups.data()), 0);
  const Scratch& scratch = copies.bytes ? copies : cuts;
  const dt_stream stream = current_stream();
  dt_status st;
  Py_BEGIN_ALLOW_THREADS;
  st = scratch.bytes ? dt_dense_qx_grouped_scratch_f16(stream, n, groups.data(), flags, scratch.at, scratch.bytes)
                     : dt_dense_qx_grouped_ws_f16(stream, n, groups.data(), flags, nullptr, 0);
  Py_END_ALLOW_THREADS;
  if (st != DT_OK) return PyLong_FromLong((long)st - (scratch.bytes ? kWithScratch : 0));
  PyObject* all = PyList_New(n);
  for (int32_t i = 0; all && i < n; i++) {
    Problem& p = ps[(size_t)i];
    PyObject* outs = PyList_New((Py_ssize_t)p.outs.size());
    for (size_t j = 0; outs && j < p.outs.size(); j++) {
      PyObject* t = p.outs[j].defined() ? THPVariable_Wrap(std::move(p.outs[j])) : Py_NewRef(Py_None);
      if (!t) Py_CLEAR(outs);
      else PyList_SET_ITEM(outs, (Py_ssize_t)j, t);
    }
    if (!outs) Py_CLEAR(all);
    else PyList_SET_ITEM(all, i, outs);
  }
  return all;
}

// lora(problem, down, up, rank, ld_up, scale, flags, scratch): a list of the output of the problem's only weight with the low-rank branch
// added, or a status that is not DT_OK as an int, or None.  down, up: both fp16, or both fp32, contiguous.
PyObject* lora(Py_ssize_t n_args, PyObject* const* args) {
  if (n_args != 8) throw Fallback{};
  const at::Tensor &down = tensor(args[1]), &up = tensor(args[2]);
  const bool f32 = down.scalar_type() == at::kFloat;
  for (const at::Tensor* t : {&down, &up})
    if (!t->is_cuda() || !t->is_contiguous() || t->scalar_type() != (f32 ? at::kFloat : at::kHalf)) throw Fallback{};
  Problem p;
  read_problem(args[0], p);
  if (p.w.size() != 1 || !p.epi.empty()) throw Fallback{};
  const dt_lora_pair pair{ptr<const void>(down), ptr<const void>(up), as_int(args[4]), as_int32(args[3]), f32 ? 1 : 0, as_float(args[5])};
  // (of the pair's padded halves the first `rank` rows are read, in up's case columns)
  if (pair.rank <= 0 || down.numel() < pair.rank * p.K || up.numel() != p.ldy[0] * pair.ld_up) throw Fallback{};
  const uint32_t flags = (uint32_t)as_int32(args[6]);
  const uint16_t* const x = ptr<const uint16_t>(*p.x);
  const int64_t ldx = p.x->dim() == 2 && p.M > 1 ? p.x->stride(0) : p.K;
  const dt_dense_post* const post = p.post.empty() ? nullptr : p.post.data();
  const size_t need = dt_lora_dense_scratch_bytes(p.M, p.K, x, ldx, p.w.data(), p.y[0], p.ldy[0], post, &pair);
  if (need == 0) throw Fallback{};
  Scratch scratch;  // (on a device too full for copies of the weights: the intermediate alone)
  scratch.ask(args[7], PyTuple_GET_ITEM(args[0], 0), need, ((size_t)p.M * pair.rank * (f32 ? 4 : 2) + 255) & ~(size_t)255);
  const dt_stream stream = current_stream();
  dt_status st;
  Py_BEGIN_ALLOW_THREADS;
  st = dt_lora_dense_f16(stream, p.M, p.K, x, ldx, p.w.data(), p.bias[0], p.y[0], p.ldy[0], post, &pair, flags, scratch.at, scratch.bytes);
  Py_END_ALLOW_THREADS;
  if (st != DT_OK) return PyLong_FromLong((long)st);
  PyObject* const out = p.outs[0].defined() ? THPVariable_Wrap(std::move(p.outs[0])) : Py_NewRef(Py_None);
  PyObject* const all = out ? PyList_New(1) : nullptr;
  if (!all) Py_XDECREF(out);
  else PyList_SET_ITEM(all, 0, out);
  return all;
}

dt_view4 view4(const at::Tensor& t) {
  if (t.dim() != 4 || t.stride(3) != 1) throw Fallback{};
  return dt_view4{t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}

// sdpa(q_segs, k_segs, v_segs, scale, gamma_q, gamma_k, rot_q, rot_k, eps, out, scratch): the output, or a status as an int, or None.
PyObject* sdpa(Py_ssize_t n_args, PyObject* const* args) {
  if (n_args != 11) throw Fallback{};
  const Seq qs(args[0]), ks(args[1]), vs(args[2]);
  if (qs.n < 1 || ks.n < 1 || vs.n != ks.n || qs.n > 8 || ks.n > 8) throw Fallback{};
  dt_seq_segment q[8] = {}, k[8] = {}, v[8] = {};
  int64_t len[2] = {0, 0};
  bool prep = args[7] != Py_None;
  const auto read = [&](const Seq& ts, PyObject* gammas, dt_seq_segment* out, int64_t* total, bool* any) {
    const bool with = gammas != Py_None;
    if (with && Seq(gammas).n != ts.n) throw Fallback{};
    for (Py_ssize_t i = 0; i < ts.n; i++) {
      const at::Tensor& t = half(ts[i]);
      out[i].view = view4(t);
      out[i].len = t.size(1);
      if (with) out[i].gamma = half_or_null(Seq(gammas)[i]);
      if (any && out[i].gamma) *any = true;
      if (total) *total += t.size(1);
    }
  };
  read(qs, args[4], q, &len[0], nullptr);
  read(ks, args[5], k, &len[1], &prep);
  read(vs, Py_None, v, nullptr, nullptr);
  const at::Tensor& q0 = tensor(qs[0]);
  const int64_t B = q0.size(0), H = q0.size(2), D = q0.size(3), Hk = tensor(ks[0]).size(2);
  if (B > INT32_MAX || H > INT32_MAX || D > INT32_MAX || Hk > INT32_MAX) throw Fallback{};
  const float scale = as_float(args[3]), eps = as_float(args[8]);
  const uint16_t *const rq = half_or_null(args[6]), *const rk = half_or_null(args[7]);
  const Ref out(args[9] == Py_None ? THPVariable_Wrap(at::empty({B, len[0], H, D}, q0.options())) : Py_NewRef(args[9]));
  const dt_view4 ov = view4(tensor(out.p));
  Scratch ws;
  const size_t need = dt_sdpa_workspace_bytes((int32_t)B, (int32_t)H, (int32_t)Hk, (int32_t)D, len[0], len[1], prep, 0);
  ws.ask(args[10], out.p, need, prep ? ((size_t)B * len[1] * Hk * D * 2 + 255) & ~(size_t)255 : 0);
  const dt_stream stream = current_stream();
  dt_status st;
  Py_BEGIN_ALLOW_THREADS;
  st = dt_sdpa_f16(stream, (int32_t)B, (int32_t)H, (int32_t)Hk, (int32_t)D, (int32_t)qs.n, q, (int32_t)ks.n, k, v, rq, rk, eps, ov, scale, nullptr,
                   nullptr, ws.at, ws.bytes);
  Py_END_ALLOW_THREADS;
  if (st != DT_OK) return PyLong_FromLong((long)st);
  return Py_NewRef(out.p);
}

// layernorm16(x, weight, bias, epsilon): the output, or a status as an int, or None.
PyObject* layernorm16(Py_ssize_t n_args, PyObject* const* args) {
  if (n_args != 4) throw Fallback{};
  const at::Tensor& x = half(args[0]);
  if (x.dim() < 1 || x.numel() == 0 || (x.dim() == 2 ? x.stride(1) != 1 : !x.is_contiguous())) throw Fallback{};
  const int64_t C = x.size(-1), M = x.numel() / C;
  const uint16_t* affine[2] = {nullptr, nullptr};
  for (int i = 0; i < 2; i++) {
    if (args[1 + i] == Py_None) continue;
    const at::Tensor& t = half(args[1 + i]);
    if (t.numel() != C || !t.is_contiguous()) throw Fallback{};
    affine[i] = ptr<const uint16_t>(t);
  }
  const float eps = as_float(args[3]);
  at::Tensor out = at::empty(x.sizes(), x.options());
  const dt_stream stream = current_stream();
  dt_status st;
  Py_BEGIN_ALLOW_THREADS;
  st = dt_layernorm_f16(stream, M, C, ptr<const uint16_t>(x), x.dim() == 2 ? x.stride(0) : C, affine[0], affine[1], eps, ptr<uint16_t>(out), C);
  Py_END_ALLOW_THREADS;
  return st == DT_OK ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong((long)st);
}

// Runs one of them; whatever it throws -- before it has enqueued anything -- sends the caller the other way, except for what the
// scratch memory's function raises.
template <PyObject* (*F)(Py_ssize_t, PyObject* const*)>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  try {
    return F(n, args);
  } catch (const Raised&) {
    return nullptr;
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// classes(QxTensor, HeadEpilogue, DensePost)
PyObject* classes(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 3) {
    PyErr_SetString(PyExc_TypeError, "three classes");
    return nullptr;
  }
  g_qx = Py_NewRef(args[0]);
  g_epi = Py_NewRef(args[1]);
  g_post = Py_NewRef(args[2]);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"classes", (PyCFunction)(void*)classes, METH_FASTCALL, nullptr},
                         {"dense", (PyCFunction)(void*)guarded<dense>, METH_FASTCALL, nullptr},
                         {"lora", (PyCFunction)(void*)guarded<lora>, METH_FASTCALL, nullptr},
                         {"sdpa", (PyCFunction)(void*)guarded<sdpa>, METH_FASTCALL, nullptr},
                         {"layernorm16", (PyCFunction)(void*)guarded<layernorm16>, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dthost", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dthost(void) {
#define INTERN(n) \
  if (!(s_##n = PyUnicode_InternFromString(#n))) return nullptr;
  NAMES(INTERN)
#undef INTERN
  return PyModule_Create(&module);
}
