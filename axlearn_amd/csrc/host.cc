// Host side of a layer call in native code: from the layer's tensors and its logit bias to the C ABI in one step.
//
// The classes in axlearn_amd/flash_attention say what the kernels take and how a call reaches them; for one call they run
// some 200 Python functions, 20 to 30 us beside the 3.5 us of each launch, and a decode step of one sequence, a short prompt or a
// small training step takes less than that on the GPU.  `attend` does the same for the calls that need nothing but their own tensors:
// bf16, f16 (decode and self-attention also f32) tensors on the current device, a causal or sliding-window mask or none,
// segment ids, a float32 sink, a dense bias.  Whatever else there is - another mask, dropout, casts, padding, tensor subclasses,
// modes that look at a call by its operations, sizes that do not fit together - is answered with None, and the
// caller goes on in Python, which refuses what it refuses.  So nothing is refused or raised here, and what both would
// take gets the same parameter block (tests/test_host_native.py compares them byte for byte).
//
// Call of the layer before / after, us: decode of one sequence 31 / 12, paged decode step with its page insert 47 / 15, chunk of 9
// rows 36 / 18, prefill of 512 tokens 28 / 15, of 256 with an f16 bias 47 / 20 (all by their kernels now), training step of 256 tokens
// 172 / 94.
#include <Python.h>

#include <algorithm>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/headeronly/version.h>

#include "../../include/axl_attn.h"

namespace {

// The bias classes, handed over once by `register_types`.
PyObject *composite_type, *causal_type, *sliding_type, *segment_type, *tensor_type, *cache_type, *paged_cache_type;
PyObject *s_biases, *s_target, *s_source, *s_window, *s_segments, *s_dtype, *s_internal_value;

// A reference that is given back at the end of the scope.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* x) : p(x) {}
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
};

// Leaves a function with nothing (null, false) where a call does not suit this path.  No exceptions: thrown through
// libraries of this size one takes 4 us, and what goes on in Python is not to pay for that.
#define AXL_WANT(...)              \
  do {                             \
    if (!(__VA_ARGS__)) return {}; \
  } while (0)

// Describe: on any device and without a launch, for the tests; the parameter block is the answer.
struct Context {
  bool describe = false;
  c10::Device device = c10::kCPU;
};

// The tensor behind `x`, or null: exactly a torch.Tensor or Parameter, dense, on the call's device.
const at::Tensor* tensor(PyObject* x) {
  AXL_WANT(THPVariable_CheckExact(x));
  const at::Tensor& t = THPVariable_Unpack(x);
  AXL_WANT(t.defined() && t.layout() == at::kStrided);
  constexpr c10::DispatchKeySet odd({c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor,
                                     c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                     c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched});
  AXL_WANT(!t.key_set().has_any(odd));
  return &t;
}
const at::Tensor* tensor(PyObject* x, const Context& c) {
  const at::Tensor* t = tensor(x);
  return t && t->device() == c.device ? t : nullptr;
}

bool differentiated(std::initializer_list<const at::Tensor*> ts) {
  if (!c10::GradMode::is_enabled()) return false;
  for (const at::Tensor* t : ts)
    if (t && t->requires_grad()) return true;
  return false;
}

// Modes that see a call by the operations it is made of (a trace, function transforms, forward differentiation, dispatch and
// function modes): there are none to see here.
bool plain_mode() {
  const c10::DispatchKeySet in = c10::impl::tls_local_dispatch_key_set().included_;
  return (in - c10::default_included_set).empty() && !c10::impl::dispatch_mode_enabled() &&
         !at::impl::torch_function_mode_enabled() && !torch::autograd::ForwardADLevel::try_get_by_idx(0);
}

bool set_context(Context& c, const at::Tensor& q, bool describe) {
  c = Context{describe, q.device()};
  return describe || (q.is_cuda() && q.get_device() == c10::hip::current_device());
}

bool dtype_code(int32_t& code, const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: code = AXL_BF16; return true;
    case at::kHalf: code = AXL_F16; return true;
    case at::kFloat: code = AXL_F32; return true;
    default: return false;
  }
}

bool strides(AxlStrides& to, const at::Tensor& t) {
  AXL_WANT(t.dim() == 4 && t.stride(3) == 1);
  to = AxlStrides{t.stride(0), t.stride(1), t.stride(2)};
  return true;
}
AxlStrides dense_strides(int64_t rows, int64_t heads, int64_t d) { return AxlStrides{rows * heads * d, heads * d, d}; }

bool fits_int32(std::initializer_list<int64_t> xs) {
  for (const int64_t x : xs)
    if (x < 0 || x > 0x7fffffff) return false;
  return true;
}

// A logit bias that is a mask in closed form, segment ids, a dense tensor, or a sum of one of each, and nothing else.
struct Mask {
  int kind = AXL_MASK_NONE;
  int32_t window = 0;
  PyObject* positions = nullptr;
  PyObject* segments = nullptr;
  PyObject* dense = nullptr;
  Mask() = default;
  Mask(const Mask&) = delete;
  ~Mask() {
    Py_XDECREF(positions);
    Py_XDECREF(segments);
    Py_XDECREF(dense);
  }
};

bool is_rank(PyObject* x, int64_t dims) {
  const at::Tensor* t = x ? tensor(x) : nullptr;
  return t && t->dim() == dims;
}

bool add_member(Mask& m, PyObject* bias) {
  const PyObject* type = (PyObject*)Py_TYPE(bias);
  if (type == segment_type) {
    AXL_WANT(!m.segments);
    m.segments = PyObject_GetAttr(bias, s_segments);
    return is_rank(m.segments, 2);
  }
  if (type == tensor_type) {
    const Ref dtype(PyObject_GetAttr(bias, s_dtype));
    AXL_WANT(!m.dense && dtype.p == Py_None);   // (else it is cast)
    m.dense = PyObject_GetAttr(bias, s_internal_value);
    return is_rank(m.dense, 4);
  }
  AXL_WANT((type == causal_type || type == sliding_type) && m.kind == AXL_MASK_NONE);
  const Ref source(PyObject_GetAttr(bias, s_source));
  m.positions = PyObject_GetAttr(bias, s_target);
  AXL_WANT(is_rank(m.positions, 2) && is_rank(source.p, 2));
  m.kind = AXL_MASK_CAUSAL;
  if (type == sliding_type) {
    const Ref window(PyObject_GetAttr(bias, s_window));
    AXL_WANT(window.p && PyLong_CheckExact(window.p));
    int overflow = 0;
    const long long w = PyLong_AsLongLongAndOverflow(window.p, &overflow);
    AXL_WANT(!overflow && fits_int32({w}));
    m.kind = AXL_MASK_SLIDING_WINDOW;
    m.window = (int32_t)w;
  }
  return true;
}

bool read_bias(Mask& m, PyObject* bias) {
  const PyObject* type = (PyObject*)Py_TYPE(bias);
  if (type != composite_type) return (type == causal_type || type == sliding_type) && add_member(m, bias);
  const Ref members(PyObject_GetAttr(bias, s_biases));
  AXL_WANT(members.p && (PyList_CheckExact(members.p) || PyTuple_CheckExact(members.p)));
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(members.p); i++)
    AXL_WANT(add_member(m, PySequence_Fast_GET_ITEM(members.p, i)));
  return true;
}

// Batch, rows, query heads, head_dim, keys, kv heads of q [B,T,Hq,D], k and v [B,S,Hkv,D].
struct Shape {
  int64_t b, t, hq, d, s, hkv;
};
bool shape(Shape& x, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  AXL_WANT(q.dim() == 4 && k.dim() == 4 && v.dim() == 4);
  x = Shape{q.size(0), q.size(1), q.size(2), q.size(3), k.size(1), k.size(2)};
  AXL_WANT(k.size(0) == x.b && k.size(3) == x.d && v.sizes() == k.sizes() && x.hkv > 0 && x.hq % x.hkv == 0);
  AXL_WANT(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type());
  return q.numel() > 0 && k.numel() > 0 && x.d <= 128 && fits_int32({x.b, x.t, x.hq, x.s, x.hkv});
}

// Rows the kernels read without padded copies (`runs_at_native_head_dim`).
bool native_rows(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int64_t d, bool dense) {
  if (d == 64 || d == 128) return true;
  AXL_WANT(d % 8 == 0 && !dense && q.scalar_type() != at::kFloat);
  const int64_t width = d <= 64 ? 64 : 128;
  for (const at::Tensor* x : {&q, &k, &v}) AXL_WANT(x->stride(1) >= width && x->size(2) * d >= width);
  return true;
}

bool sink_pointer(const float*& p, const at::Tensor*& t, PyObject* sink, const Context& c, int64_t hq) {
  p = nullptr;
  t = nullptr;
  if (sink == Py_None) return true;
  t = tensor(sink, c);
  AXL_WANT(t && t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == hq && t->is_contiguous());
  p = (const float*)t->const_data_ptr();
  return true;
}

bool segment_pointer(const int32_t*& p, PyObject* segments, const Context& c, const Shape& x) {
  p = nullptr;
  if (!segments || segments == Py_None) return true;
  const at::Tensor* ids = tensor(segments, c);
  AXL_WANT(ids && x.t == x.s && ids->dim() == 2 && ids->size(0) == x.b && ids->size(1) == x.t && ids->scalar_type() == at::kInt &&
           ids->is_contiguous());
  p = (const int32_t*)ids->const_data_ptr();
  return true;
}

// A dense bias [B|1,Hq|1,T,S] as the kernels read it: bf16 or fp32 in place, f16 as an fp32 copy that `kept` holds.
bool dense_bias(AxlAttnAux& aux, at::Tensor& kept, PyObject* bias, const Context& c, const Shape& x) {
  if (!bias || bias == Py_None) return true;
  const at::Tensor* t = tensor(bias, c);
  AXL_WANT(t && t->dim() == 4 && (t->size(0) == 1 || t->size(0) == x.b) && (t->size(1) == 1 || t->size(1) == x.hq) &&
           t->size(2) == x.t && t->size(3) == x.s && t->stride(3) == 1);
  kept = t->scalar_type() == at::kHalf ? t->to(at::kFloat) : *t;
  AXL_WANT((kept.scalar_type() == at::kBFloat16 || kept.scalar_type() == at::kFloat) && kept.stride(3) == 1 &&
           dtype_code(aux.bias_dtype, kept));
  aux.bias = kept.const_data_ptr();
  aux.bias_batch_stride = kept.size(0) > 1 ? kept.stride(0) : 0;
  aux.bias_head_stride = kept.size(1) > 1 ? kept.stride(1) : 0;
  aux.bias_row_stride = kept.stride(2);
  return true;
}

at::Tensor empty(at::IntArrayRef sizes, const at::Tensor& like, at::ScalarType type) {
  return at::empty(sizes, like.options().dtype(type).requires_grad(false));
}

// Runs a call of the C ABI as ctypes does, without the interpreter's lock.  A call that is refused is not raised here:
// the caller's way through Python comes to the same refusal and words it.
template <typename P>
bool launch(int (*call)(const P*, void*), const P& p, const Context& c) {
  void* const stream = c10::hip::getCurrentHIPStream(c.device.index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call(&p, stream);
  Py_END_ALLOW_THREADS
  return rc == AXL_OK;
}

template <typename P>
PyObject* block(const P& p) {
  return PyBytes_FromStringAndSize((const char*)&p, sizeof(p));
}

PyObject* with_probs(const at::Tensor& out, int64_t b, int64_t hq, int64_t t, int64_t s) {
  const at::Tensor probs = at::empty({b, hq, t, s}, at::TensorOptions().device(at::kMeta));
  const Ref o(THPVariable_Wrap(out)), p(THPVariable_Wrap(probs));
  return o.p && p.p ? PyTuple_Pack(2, o.p, p.p) : nullptr;
}

// Single-token decode over a contiguous cache (HipDecoding) or a page pool (HipPagedAttention).
PyObject* decode(const at::Tensor& q, PyObject* key, PyObject* value, PyObject* tables, const Mask& m, double scale,
                 int64_t block_size, const Context& c) {
  const at::Tensor *k = tensor(key, c), *v = tensor(value, c), *pos = m.positions ? tensor(m.positions, c) : nullptr;
  AXL_WANT(k && v && pos && !m.segments && !m.dense && !differentiated({&q, k, v}) && q.is_contiguous());
  const int64_t b = q.size(0), hq = q.size(2), d = q.size(3);
  const bool i64 = pos->scalar_type() == at::kLong;
  AXL_WANT((i64 || pos->scalar_type() == at::kInt) && (pos->size(0) == 1 || pos->size(0) == b) && pos->size(1) >= 1);
  AXL_WANT(d % 8 == 0 && fits_int32({b, hq, d}));
  at::Tensor out, workspace;
  auto run = [&](auto& p, auto bytes, auto call) -> bool {
    p.q = q.const_data_ptr();
    // the last position of every sequence, as the bias holds it
    p.lengths = (const int32_t*)((const char*)pos->const_data_ptr() + (pos->size(1) - 1) * pos->stride(1) * (i64 ? 8 : 4));
    p.lengths_stride = pos->size(0) > 1 ? pos->stride(0) : 0;
    p.flags = AXL_DECODE_LENGTHS_ARE_POSITIONS | (i64 ? AXL_DECODE_LENGTHS_I64 : 0);
    p.batch = (int32_t)b; p.num_q_heads = (int32_t)hq; p.head_dim = (int32_t)d;
    AXL_WANT(dtype_code(p.dtype, q));
    p.sliding_window = m.kind == AXL_MASK_SLIDING_WINDOW ? m.window : -1;
    p.softmax_scale = (float)scale;
    if (c.describe) return true;
    out = empty(q.sizes(), q, q.scalar_type());
    p.out = out.mutable_data_ptr();
    workspace = empty({(int64_t)std::max<size_t>(bytes(&p), 16)}, q, at::kByte);
    p.workspace = workspace.mutable_data_ptr();
    p.workspace_bytes = (size_t)workspace.numel();
    return launch(call, p, c);
  };
  if (!tables) {
    Shape x;
    AxlDecodeParams p = {};
    AXL_WANT(shape(x, q, *k, *v) && strides(p.k_strides, *k) && strides(p.v_strides, *v));
    p.k = k->const_data_ptr(); p.v = v->const_data_ptr();
    p.kv_len = (int32_t)x.s; p.num_kv_heads = (int32_t)x.hkv;
    AXL_WANT(run(p, axl_decode_workspace_bytes, axl_decode));
    return c.describe ? block(p) : with_probs(out, b, hq, 1, x.s);
  }
  const at::Tensor* table = tensor(tables, c);
  AXL_WANT(table && k->dim() == 4 && v->sizes() == k->sizes() && k->size(0) > 0 && hq % k->size(0) == 0 && k->size(3) == d && d <= 128);
  AXL_WANT(k->scalar_type() == q.scalar_type() && v->scalar_type() == q.scalar_type() && k->is_contiguous() && v->is_contiguous());
  AXL_WANT(table->dim() == 2 && table->size(0) == b && table->scalar_type() == at::kInt && table->is_contiguous());
  AXL_WANT(q.numel() > 0 && k->numel() > 0 && table->numel() > 0);
  const int64_t page = k->size(2);
  AXL_WANT(page >= 16 && (page & (page - 1)) == 0 && block_size % page == 0 && block_size < 16 * page);
  AXL_WANT(fits_int32({k->size(0), k->size(1), page, table->size(1)}));
  AxlPagedDecodeParams p = {};
  p.k_pages = k->const_data_ptr(); p.v_pages = v->const_data_ptr();
  p.page_tables = (const int32_t*)table->const_data_ptr();
  p.num_kv_heads = (int32_t)k->size(0); p.num_pages = (int32_t)k->size(1); p.page_size = (int32_t)page;
  p.pages_per_seq = (int32_t)table->size(1);
  AXL_WANT(run(p, axl_paged_decode_workspace_bytes, axl_paged_decode));
  return c.describe ? block(p) : with_probs(out, b, hq, 1, page * table->size(1));
}

// What the blocks of the prefill kernels have in common; `out` is dense whatever the strides of q.
template <typename P>
bool prefill_block(P& p, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const Shape& x, double scale) {
  p.q = q.const_data_ptr(); p.k = k.const_data_ptr(); p.v = v.const_data_ptr();
  p.out_strides = dense_strides(x.t, x.hq, x.d);
  p.batch = (int32_t)x.b; p.q_len = (int32_t)x.t; p.kv_len = (int32_t)x.s; p.num_q_heads = (int32_t)x.hq; p.num_kv_heads = (int32_t)x.hkv;
  p.head_dim = (int32_t)x.d;
  p.softmax_scale = (float)scale;
  return strides(p.q_strides, q) && strides(p.k_strides, k) && strides(p.v_strides, v) && dtype_code(p.dtype, q);
}

// A chunk of query rows per sequence over a contiguous cache (HipFlashAttention._incremental_prefill).
PyObject* chunk(const at::Tensor& q, PyObject* key, PyObject* value, const Mask& m, PyObject* logit_sink, double scale, const Context& c) {
  const at::Tensor *k = tensor(key, c), *v = tensor(value, c), *pos = m.positions ? tensor(m.positions, c) : nullptr, *sink;
  AXL_WANT(k && v && pos && !m.segments && !m.dense && !differentiated({&q, k, v}));
  Shape x;
  AXL_WANT(shape(x, q, *k, *v) && x.s % 128 == 0 && q.scalar_type() != at::kFloat && native_rows(q, *k, *v, x.d, false));
  AXL_WANT((uintptr_t)q.const_data_ptr() % 16 == 0 && q.stride(0) % 8 == 0 && q.stride(1) % 8 == 0 && q.stride(2) % 8 == 0);
  const bool i64 = pos->scalar_type() == at::kLong;
  AXL_WANT((i64 || pos->scalar_type() == at::kInt) && (pos->size(0) == 1 || pos->size(0) == x.b) && pos->size(1) == x.t);
  AxlFlashChunkParams p = {};
  AXL_WANT(prefill_block(p, q, *k, *v, x, scale) && sink_pointer(p.logit_sink, sink, logit_sink, c, x.hq));
  p.mask_kind = m.kind; p.sliding_window = m.window;
  p.positions = pos->const_data_ptr();
  p.pos_batch_stride = pos->size(0) > 1 ? pos->stride(0) : 0;
  p.pos_row_stride = pos->stride(1);
  p.pos_is_i64 = i64;
  if (c.describe) return block(p);
  const at::Tensor out = empty(q.sizes(), q, q.scalar_type());
  p.out = out.mutable_data_ptr();
  at::Tensor workspace;
  if (const size_t bytes = axl_flash_chunk_workspace_bytes(&p)) {
    workspace = empty({(int64_t)bytes}, q, at::kByte);
    p.workspace = workspace.mutable_data_ptr();
    p.workspace_bytes = bytes;
  }
  AXL_WANT(launch(axl_flash_chunk, p, c));
  return with_probs(out, x.b, x.hq, x.t, x.s);
}

// Whole sequences (HipFlashAttention.__call__).  With something to differentiate: (None, probs, mask kind, window,
// segment ids or None, dense bias or None), from which the caller makes its autograd node.
PyObject* whole(const at::Tensor& q, PyObject* key, PyObject* value, const Mask& m, PyObject* logit_sink, double scale, const Context& c) {
  const at::Tensor *k = tensor(key, c), *v = tensor(value, c), *dense = m.dense ? tensor(m.dense, c) : nullptr, *sink;
  Shape x;
  AXL_WANT(k && v && shape(x, q, *k, *v) && x.t % 128 == 0 && x.s % 128 == 0 && native_rows(q, *k, *v, x.d, m.dense));
  AxlFlashFwdParams p = {};
  AXL_WANT(prefill_block(p, q, *k, *v, x, scale) && sink_pointer(p.logit_sink, sink, logit_sink, c, x.hq) &&
           segment_pointer(p.segment_ids, m.segments, c, x));
  p.mask_kind = m.kind; p.sliding_window = m.window;
  // (a bias of other rows is copied there)
  AXL_WANT(!m.dense || (dense && dense->is_contiguous() && (uintptr_t)dense->const_data_ptr() % 16 == 0));
  if (!c.describe && differentiated({&q, k, v, sink, dense})) {
    AXL_WANT(!dense || dense->is_floating_point());
    const at::Tensor probs = at::empty({x.b, x.hq, x.t, x.s}, at::TensorOptions().device(at::kMeta));
    const Ref wrapped(THPVariable_Wrap(probs));
    return wrapped.p ? Py_BuildValue("OOiiOO", Py_None, wrapped.p, m.kind, (int)m.window, m.segments ? m.segments : Py_None,
                                     m.dense ? m.dense : Py_None) : nullptr;
  }
  at::Tensor kept;
  AXL_WANT(dense_bias(p.aux, kept, m.dense, c, x));
  if (c.describe) return block(p);
  const at::Tensor out = empty(q.sizes(), q, q.scalar_type());
  p.out = out.mutable_data_ptr();
  AXL_WANT(launch(axl_flash_fwd, p, c));
  return with_probs(out, x.b, x.hq, x.t, x.s);
}

// The boundary to Python: whatever keeps a call off this path, an allocation that fails among it, is None.
template <typename F>
PyObject* guarded(F&& f) {
  PyObject* r = nullptr;
  try {
    if (plain_mode()) r = f();
  } catch (...) {
    r = nullptr;
  }
  if (r) return r;
  PyErr_Clear();
  Py_RETURN_NONE;
}

bool read_scale(double& scale, PyObject* x) {
  AXL_WANT(PyFloat_CheckExact(x));
  scale = PyFloat_AS_DOUBLE(x);
  return scale > 0 && scale < 3.4e38;
}
bool read_int(int64_t& to, PyObject* x) {
  AXL_WANT(PyLong_CheckExact(x));
  int overflow = 0;
  to = PyLong_AsLongLongAndOverflow(x, &overflow);
  return !overflow && to >= 0;
}

// attend(q, k, v, bias, page_indices, kv_cache_type, logit_sink, softmax_scale, gpu_block_size, describe)
PyObject* py_attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    double scale;
    int64_t block_size;
    Context c;
    Mask m;
    AXL_WANT(n == 10 && composite_type && read_scale(scale, a[7]) && read_int(block_size, a[8]) && block_size > 0);
    const at::Tensor* q = tensor(a[0]);
    AXL_WANT(q && q->dim() == 4 && set_context(c, *q, a[9] == Py_True) && read_bias(m, a[3]));
    if (a[5] == Py_None) return a[4] == Py_None ? whole(*q, a[1], a[2], m, a[6], scale, c) : nullptr;
    if (a[5] == paged_cache_type) {
      AXL_WANT(q->size(1) == 1 && a[4] != Py_None && a[6] == Py_None);
      return decode(*q, a[1], a[2], a[4], m, scale, block_size, c);
    }
    AXL_WANT(a[5] == cache_type && a[4] == Py_None);
    if (q->size(1) != 1) return chunk(*q, a[1], a[2], m, a[6], scale, c);
    return a[6] == Py_None ? decode(*q, a[1], a[2], nullptr, m, scale, 0, c) : nullptr;
  });
}

// page_insert(k_pages, v_pages, k_proj, v_proj, page_indices, key_positions, describe) -> True where the step's keys and values
// [B,1,Hkv,D] were written (ops.paged_kv_insert with `single_row`).
PyObject* py_page_insert(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    AXL_WANT(n == 7);
    const at::Tensor* pool = tensor(a[0]);
    Context c;
    AXL_WANT(pool && pool->dim() == 4 && set_context(c, *pool, a[6] == Py_True));
    const at::Tensor *v_pool = tensor(a[1], c), *k = tensor(a[2], c), *v = tensor(a[3], c), *table = tensor(a[4], c), *pos = tensor(a[5], c);
    AXL_WANT(v_pool && k && v && table && pos && !differentiated({pool, v_pool, k, v}));
    AXL_WANT(v_pool->sizes() == pool->sizes() && v_pool->scalar_type() == pool->scalar_type() && pool->is_contiguous() &&
             v_pool->is_contiguous() && pool->numel() > 0);
    AXL_WANT(table->dim() == 2 && table->is_contiguous() && table->scalar_type() == at::kInt && table->numel() > 0);
    const int64_t b = table->size(0), hkv = pool->size(0), d = pool->size(3);
    for (const at::Tensor* x : {k, v})
      AXL_WANT(x->dim() == 4 && x->size(0) == b && x->size(1) == 1 && x->size(2) == hkv && x->size(3) == d && x->stride(3) == 1 &&
               x->scalar_type() == pool->scalar_type());
    AXL_WANT(pos->dim() == 2 && pos->size(1) == 1 && (pos->size(0) == 1 || pos->size(0) == b) && pos->scalar_type() == at::kInt &&
             pos->is_contiguous());
    AXL_WANT(fits_int32({b, hkv, d, pool->size(1), pool->size(2), table->size(1)}));
    AxlPageInsertParams p = {};
    AXL_WANT(dtype_code(p.dtype, *pool));
    p.k_pages = pool->data_ptr(); p.v_pages = v_pool->data_ptr();
    p.k_proj = k->const_data_ptr(); p.v_proj = v->const_data_ptr();
    p.page_indices = (const int32_t*)table->const_data_ptr();
    p.key_positions = (const int32_t*)pos->const_data_ptr();
    p.k_proj_batch_stride = k->stride(0); p.k_proj_head_stride = k->stride(2);
    p.v_proj_batch_stride = v->stride(0); p.v_proj_head_stride = v->stride(2);
    p.batch = (int32_t)b; p.num_kv_heads = (int32_t)hkv; p.head_dim = (int32_t)d;
    p.num_pages = (int32_t)pool->size(1); p.page_size = (int32_t)pool->size(2); p.pages_per_seq = (int32_t)table->size(1);
    p.broadcast_positions = pos->size(0) == 1 && b > 1;
    if (c.describe) return block(p);
    AXL_WANT(launch(axl_paged_kv_insert, p, c));
    Py_RETURN_TRUE;
  });
}

// flash_fwd(q, k, v, segment_ids, logit_sink, softmax_scale, mask_kind, sliding_window, bias, bias_copy, describe) -> (out, lse)
// (ops.flash_fwd without offsets and dropout mask).
PyObject* py_flash_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    double scale;
    int64_t kind, window;
    Context c;
    Shape x;
    AXL_WANT(n == 11 && read_scale(scale, a[5]) && read_int(kind, a[6]) && read_int(window, a[7]) && fits_int32({kind, window}));
    const at::Tensor *q = tensor(a[0]), *sink;
    AXL_WANT(q && set_context(c, *q, a[10] == Py_True));
    const at::Tensor *k = tensor(a[1], c), *v = tensor(a[2], c);
    at::Tensor kept;
    AxlFlashFwdParams p = {};
    AXL_WANT(k && v && shape(x, *q, *k, *v) && prefill_block(p, *q, *k, *v, x, scale) && segment_pointer(p.segment_ids, a[3], c, x) &&
             sink_pointer(p.logit_sink, sink, a[4], c, x.hq) && dense_bias(p.aux, kept, a[8], c, x));
    p.mask_kind = (int32_t)kind; p.sliding_window = (int32_t)window;
    if (a[9] != Py_None) {   // as ops.can_copy_bias says
      const at::Tensor* copy = tensor(a[9], c);
      AXL_WANT(copy && kept.defined() && kept.scalar_type() == at::kBFloat16 && kept.is_contiguous() && !p.segment_ids &&
               q->scalar_type() != at::kFloat && (uintptr_t)p.aux.bias % 16 == 0 && x.t * x.s < (int64_t)1 << 31);
      AXL_WANT(copy->sizes() == kept.sizes() && copy->scalar_type() == at::kBFloat16 && copy->is_contiguous());
      p.bias_copy = copy->data_ptr();
    }
    if (c.describe) return block(p);
    const at::Tensor out = empty(q->sizes(), *q, q->scalar_type()), lse = empty({x.b, x.hq, x.t}, *q, at::kFloat);
    p.out = out.mutable_data_ptr();
    p.lse = (float*)lse.mutable_data_ptr();
    AXL_WANT(launch(axl_flash_fwd, p, c));
    const Ref o(THPVariable_Wrap(out)), l(THPVariable_Wrap(lse));
    return o.p && l.p ? PyTuple_Pack(2, o.p, l.p) : nullptr;
  });
}

// flash_bwd(q, k, v, out, lse, d_out, segment_ids, logit_sink, softmax_scale, mask_kind, sliding_window, limit, bias, describe)
// -> (dq, dk, dv[, d_sink]) (ops.flash_bwd by the size rule, where dS as a whole fits `limit` bytes or does not apply).
PyObject* py_flash_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    double scale;
    int64_t kind, window, limit;
    Context c;
    Shape x;
    AXL_WANT(n == 14 && read_scale(scale, a[8]) && read_int(kind, a[9]) && read_int(window, a[10]) && read_int(limit, a[11]) &&
             fits_int32({kind, window}));
    const at::Tensor *q = tensor(a[0]), *sink;
    AXL_WANT(q && set_context(c, *q, a[13] == Py_True));
    const at::Tensor *k = tensor(a[1], c), *v = tensor(a[2], c), *out = tensor(a[3], c), *lse = tensor(a[4], c), *d_out = tensor(a[5], c);
    AXL_WANT(k && v && out && lse && d_out && shape(x, *q, *k, *v));
    AXL_WANT(out->sizes() == q->sizes() && d_out->sizes() == q->sizes() && out->scalar_type() == q->scalar_type() &&
             d_out->scalar_type() == q->scalar_type());
    AXL_WANT(lse->dim() == 3 && lse->size(0) == x.b && lse->size(1) == x.hq && lse->size(2) == x.t &&
             lse->scalar_type() == at::kFloat && lse->is_contiguous());
    AxlFlashBwdParams p = {};
    AXL_WANT(prefill_block(p, *q, *k, *v, x, scale) && strides(p.out_strides, *out) && strides(p.d_out_strides, *d_out) &&
             segment_pointer(p.segment_ids, a[6], c, x) && sink_pointer(p.logit_sink, sink, a[7], c, x.hq));
    p.out = out->const_data_ptr(); p.d_out = d_out->const_data_ptr(); p.lse = (const float*)lse->const_data_ptr();
    p.dq_strides = dense_strides(x.t, x.hq, x.d);
    p.dk_strides = p.dv_strides = dense_strides(x.s, x.hkv, x.d);
    p.mask_kind = (int32_t)kind; p.sliding_window = (int32_t)window;
    // dS is kept where that is a form of the call (its workspace is larger with the flag) and fits; slices of heads are
    // the caller's business
    const size_t without = axl_flash_bwd_workspace_bytes(&p);
    p.flags = AXL_BWD_DS_WORKSPACE;
    const size_t with = axl_flash_bwd_workspace_bytes(&p);
    AXL_WANT(with == without || with <= (size_t)limit);
    if (with == without) p.flags = 0;
    at::Tensor kept;
    AXL_WANT(dense_bias(p.aux, kept, a[12], c, x));
    if (c.describe) return block(p);
    const at::Tensor dq = empty(q->sizes(), *q, q->scalar_type()), dk = empty(k->sizes(), *k, k->scalar_type()),
                     dv = empty(v->sizes(), *v, v->scalar_type());
    const at::Tensor workspace = empty({(int64_t)std::max<size_t>(with, 256)}, *q, at::kByte);
    at::Tensor d_sink;
    p.dq = dq.mutable_data_ptr(); p.dk = dk.mutable_data_ptr(); p.dv = dv.mutable_data_ptr();
    if (sink) {
      d_sink = empty({x.hq}, *q, at::kFloat);
      p.d_logit_sink = (float*)d_sink.mutable_data_ptr();
    }
    p.workspace = workspace.mutable_data_ptr();
    p.workspace_bytes = (size_t)workspace.numel();
    AXL_WANT(launch(axl_flash_bwd, p, c));
    const Ref g0(THPVariable_Wrap(dq)), g1(THPVariable_Wrap(dk)), g2(THPVariable_Wrap(dv));
    AXL_WANT(g0.p && g1.p && g2.p);
    if (!sink) return PyTuple_Pack(3, g0.p, g1.p, g2.p);
    const Ref g3(THPVariable_Wrap(d_sink));
    return g3.p ? PyTuple_Pack(4, g0.p, g1.p, g2.p, g3.p) : nullptr;
  });
}

// register_types(Composite, Causal, SlidingWindow, SegmentId, Tensor, KVCache, PagedKVCache)
PyObject* py_register_types(PyObject*, PyObject* args) {
  PyObject* t[7];
  if (!PyArg_ParseTuple(args, "OOOOOOO", &t[0], &t[1], &t[2], &t[3], &t[4], &t[5], &t[6])) return nullptr;
  PyObject** const to[7] = {&composite_type, &causal_type, &sliding_type, &segment_type, &tensor_type, &cache_type, &paged_cache_type};
  for (int i = 0; i < 7; i++) {
    Py_INCREF(t[i]);
    Py_XSETREF(*to[i], t[i]);
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"attend", (PyCFunction)(void*)py_attend, METH_FASTCALL, nullptr},
    {"page_insert", (PyCFunction)(void*)py_page_insert, METH_FASTCALL, nullptr},
    {"flash_fwd", (PyCFunction)(void*)py_flash_fwd, METH_FASTCALL, nullptr},
    {"flash_bwd", (PyCFunction)(void*)py_flash_bwd, METH_FASTCALL, nullptr},
    {"register_types", py_register_types, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_axl_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__axl_host() {
  s_biases = PyUnicode_InternFromString("biases");
  s_target = PyUnicode_InternFromString("target_positions");
  s_source = PyUnicode_InternFromString("source_positions");
  s_window = PyUnicode_InternFromString("sliding_window_size");
  s_segments = PyUnicode_InternFromString("segment_ids");
  s_dtype = PyUnicode_InternFromString("dtype");
  s_internal_value = PyUnicode_InternFromString("_internal_value");
  PyObject* const m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
