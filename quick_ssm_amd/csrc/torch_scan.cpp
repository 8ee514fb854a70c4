// Native half of the Python package's scan: output tensors, launch plans, the launches and the autograd nodes.
//
// A training step over a small tensor is bound by the host: two launches keep the GPU busy for under 20 us, and the
// interpreter needed 114 to 142 us to make them (a Python autograd node runs on autograd's own thread, on a core that has to
// be woken and under the interpreter lock).  Here a forward is one call from Python, and the backward node runs without
// the interpreter except for the few bytecodes that number the launch (quick_ssm_amd/hip_scan.py keeps the control
// block and workspace of every stream and is the only place that numbers launches).  Measured, Python node -> this one:
// fp32 B=4 L=2048 D=16 forward + backward 114-142 -> 78 us (of which torch's own hand-over to its thread and back is
// about 45), fp16 B=2 L=8192 D=512 with a carried state 170 -> 95 us, one token of generation 21.8 -> 10.5 us.
//
// Takes the place of the Python bodies of the reference's `_TritonScanFunction` (quick_ssm/scan_interface.py:49-158).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <cstring>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/quick_ssm_hip.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// Python callables of quick_ssm_amd (held for the life of the process).
PyObject* g_take_launch = nullptr;   // (device index, stream, control bytes, workspace bytes) -> see LaunchBuffers
PyObject* g_check = nullptr;         // raises QssmError for a nonzero return code

at::ScalarType scalar_of(int code) {
  return code == QSSM_F32 ? at::kFloat : code == QSSM_F16 ? at::kHalf : at::kBFloat16;
}

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return QSSM_F32;
    case at::kHalf: return QSSM_F16;
    case at::kBFloat16: return QSSM_BF16;
    default: TORCH_CHECK_VALUE(false, "scan operands must be float32, float16 or bfloat16, got ", t);
  }
}

struct Gil {
  PyGILState_STATE s = PyGILState_Ensure();
  ~Gil() { PyGILState_Release(s); }
};

// A launch can block while the stream's queue is full: not with the interpreter lock in hand.
struct Unlocked {
  PyThreadState* s = PyGILState_Check() ? PyEval_SaveThread() : nullptr;
  ~Unlocked() {
    if (s != nullptr) PyEval_RestoreThread(s);
  }
};

[[noreturn]] void throw_python_error() {
  python_error err;
  err.persist();   // fetches the Python error; whoever catches it on a Python thread restores it
  throw err;
}

void check_rc(int rc) {
  if (rc == 0) return;
  Gil gil;
  PyObject* r = PyObject_CallFunction(g_check, "i", rc);
  Py_XDECREF(r);
  if (r == nullptr) throw_python_error();
  TORCH_CHECK(false, "libquick_ssm_hip call failed with code ", rc);
}

// Control block, workspace and number of one launch.  `owner` keeps the two tensors alive until the launch is on its
// stream: another thread may replace them by larger ones at any moment.
struct LaunchBuffers {
  PyObject* owner = nullptr;
  void *control = nullptr, *workspace = nullptr;
  uint64_t control_size = 0, workspace_size = 0;
  uint32_t epoch = 0;
  int32_t* status_to = nullptr;   // pinned word the status is to be copied to behind this launch

  LaunchBuffers(int index, void* stream, uint64_t need_c, uint64_t need_w) {
    Gil gil;
    owner = PyObject_CallFunction(g_take_launch, "iKKK", index, (unsigned long long)(uintptr_t)stream,
                                  (unsigned long long)need_c, (unsigned long long)need_w);
    if (owner == nullptr) throw_python_error();
    unsigned long long v[6];
    for (int k = 0; k < 6; ++k) v[k] = PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(owner, k));
    control = (void*)(uintptr_t)v[0];
    control_size = v[1];
    workspace = (void*)(uintptr_t)v[2];
    workspace_size = v[3];
    epoch = (uint32_t)v[4];
    status_to = (int32_t*)(uintptr_t)v[5];
  }
  ~LaunchBuffers() {
    Gil gil;
    Py_XDECREF(owner);
  }
  LaunchBuffers(const LaunchBuffers&) = delete;
};

// ---- launch plans ------------------------------------------------------------------------------------------------

// Plans depend on nothing but these numbers, so they are kept (per thread, bounded) and handed out as copies: between
// a plan and its launch the interpreter may run, and with it another scan on this thread.
struct PlanKey {
  int32_t B, L, D, in, out, direction, align, ckpt, tune, bwd_tune, keep;
  bool operator==(const PlanKey& o) const { return std::memcmp(this, &o, sizeof(*this)) == 0; }
};
struct PlanHash {
  size_t operator()(const PlanKey& k) const {
    uint64_t h = 1469598103934665603ull;
    const int32_t* p = &k.B;
    for (size_t i = 0; i < sizeof(PlanKey) / sizeof(int32_t); ++i) h = (h ^ (uint32_t)p[i]) * 1099511628211ull;
    return (size_t)(h ^ (h >> 29));
  }
};

// A forward's `ckpt` says whether it saves states (1) or not (0); their spacing is the tile length of the backward
// that `bwd_tune` asks for.  A backward's is the spacing the states were saved with.  `keep` < 0: the planner's cache
// policy; otherwise the most tiles per chain that may leave their operands in the caches.
qssm_plan plan_for(const PlanKey& k) {
  static thread_local std::unordered_map<PlanKey, qssm_plan, PlanHash> plans;
  auto it = plans.find(k);
  if (it != plans.end()) return it->second;
  qssm_plan p;
  int32_t stride = k.ckpt;
  if (k.direction == QSSM_FORWARD && k.ckpt != 0) {
    check_rc(qssm_plan_scan_loose(k.B, k.L, k.D, k.in, k.out, QSSM_BACKWARD, k.align, 0, k.bwd_tune, &p));
    stride = p.seg_len;
  }
  check_rc(qssm_plan_scan_loose(k.B, k.L, k.D, k.in, k.out, k.direction, k.align, stride, k.tune, &p));
  if (k.direction == QSSM_FORWARD && k.keep >= 0 && p.keep_tiles > k.keep) p.keep_tiles = k.keep;
  if (plans.size() >= 1024) plans.clear();
  return plans.emplace(k, p).first->second;
}

// ---- operands ----------------------------------------------------------------------------------------------------

// One operand as a launch takes it; `bits` collects what the alignment of all of them is read from.
struct Operand {
  Tensor t;
  const void* p = nullptr;
  qssm_strides s{0, 0};

  Operand() = default;
  Operand(const Tensor& given, uint64_t& bits) {
    if (!given.defined()) return;
    t = given.stride(2) == 1 ? given : given.contiguous();
    p = t.const_data_ptr();
    s = {t.stride(0), t.stride(1)};
    const uint64_t es = t.element_size(), at = (uint64_t)(uintptr_t)p;
    bits |= at % es != 0 ? 1u : (at / es) | (uint64_t)s.b | (uint64_t)s.l;
  }
};

Tensor fresh(int64_t B, int64_t L, int64_t D, at::ScalarType dtype, const Tensor& like, uint64_t* bits) {
  Tensor t = at::empty({B, L, D}, like.options().dtype(dtype).memory_format(c10::nullopt).requires_grad(c10::nullopt));
  if (bits != nullptr) *bits |= ((uint64_t)(uintptr_t)t.const_data_ptr() / t.element_size()) | (uint64_t)(L * D);
  return t;
}

int align_of(uint64_t bits) {
  const uint64_t low = bits & (~bits + 1);
  return low == 0 || low > 8 ? 8 : (int)low;
}

void require_gpu(std::initializer_list<const Tensor*> ts) {
  const Tensor& first = **ts.begin();
  for (const Tensor* t : ts) {
    if (!t->defined()) continue;
    TORCH_CHECK(t->is_cuda(), "HIP scan backend requires GPU tensors.");
    TORCH_CHECK(t->get_device() == first.get_device(), "all scan operands must live on one GPU");
  }
}

void check_state(const Tensor& t, int64_t B, int64_t D, const Tensor& like, const char* name) {
  if (!t.defined()) return;
  TORCH_CHECK_VALUE(t.dim() == 2 && t.size(0) == B && t.size(1) == D && t.scalar_type() == at::kFloat && t.is_contiguous() &&
                        t.device() == like.device(),
                    name, " must be a contiguous float32 tensor of shape (", B, ", ", D, ") on ", like.device(), ", got ",
                    t.scalar_type(), " ", t.sizes(), " on ", t.device());
}

// A state that the launch reads, as memory of its own when the launch also writes to it (a state carried in place): where
// lanes share columns, and where a chain's first tiles read the state that its last one replaces, the order is nobody's.
Tensor read_state(const Tensor& t, const Tensor& written) {
  if (!t.defined() || !written.defined() || t.numel() == 0) return t;
  const char *r = (const char*)t.const_data_ptr(), *w = (const char*)written.const_data_ptr();
  return r < w + written.nbytes() && w < r + t.nbytes() ? t.clone() : t;
}

void* data_or_null(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
const float* floats_or_null(const Tensor& t) { return t.defined() ? t.const_data_ptr<float>() : nullptr; }

template <typename Call, typename Fn>
void launch(Call& k, const qssm_plan& plan, int index, Fn fn) {
  void* stream = (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)index).stream();
  const LaunchBuffers buf(index, stream, plan.control_bytes, plan.workspace_bytes);
  k.plan = &plan;
  k.control = buf.control;
  k.control_size = buf.control_size;
  k.workspace = buf.workspace;
  k.workspace_bytes = buf.workspace_size;
  k.epoch = buf.epoch;
  k.stream = stream;
  int rc;
  {
    const Unlocked other_threads_may_run;
    rc = fn(&k);
  }
  check_rc(rc);
  if (buf.status_to != nullptr) check_rc(qssm_control_status_async(buf.control, buf.status_to, stream));
}

// A call of the library that makes launches, with the other threads running beside it.
template <typename Fn>
void unlocked(Fn fn) {
  int rc;
  {
    const Unlocked other_threads_may_run;
    rc = fn();
  }
  check_rc(rc);
}

struct ForwardOut {
  Tensor y, h, ckpt;
  int64_t stride = 0;
};

ForwardOut scan_forward(const Tensor& x, const Tensor& a, const Tensor& b, const Tensor& c, int out_code, bool want_y,
                        bool want_h, bool want_ckpt, int keep, int tune, int bwd_tune, const Tensor& h_init,
                        const Tensor& h_final) {
  require_gpu({&x, &a, &b, &c});
  TORCH_CHECK_VALUE(x.dim() == 3, "x, a, b, c must be 3-D tensors [B, L, D].");
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2);
  const c10::OptionalDeviceGuard guard(x.device());
  uint64_t bits = (uint64_t)D;
  ForwardOut out;
  if (want_y) out.y = fresh(B, L, D, scalar_of(out_code), x, &bits);
  if (want_h) out.h = fresh(B, L, D, at::kFloat, x, &bits);
  check_state(h_init, B, D, x, "h_init");
  check_state(h_final, B, D, x, "h_final");
  if (B == 0 || L == 0 || D == 0) {   // nothing happened to the state
    if (h_final.defined()) {
      if (h_init.defined()) h_final.copy_(h_init);
      else h_final.zero_();
    }
    if (want_ckpt) out.ckpt = fresh(B, 0, D, at::kFloat, x, nullptr);
    return out;
  }
  TORCH_CHECK_VALUE(B <= INT32_MAX && L <= INT32_MAX && D <= INT32_MAX, "a dimension of the scan does not fit 32 bits");
  const Operand ox(x, bits), oa(a, bits), ob(b, bits), oc(c, bits);
  const qssm_plan plan = plan_for({(int32_t)B, (int32_t)L, (int32_t)D, code_of(x.scalar_type()), out_code, QSSM_FORWARD,
                                    align_of(bits), want_ckpt, tune, bwd_tune, keep});
  if (want_ckpt) out.ckpt = fresh(B, plan.n_ckpt, D, at::kFloat, x, nullptr);
  out.stride = plan.ckpt_stride;
  const qssm_strides dense{L * D, D};
  qssm_forward_call k{};
  k.x = ox.p; k.a = oa.p; k.b = ob.p; k.c = oc.p;
  k.sx = ox.s; k.sa = oa.s; k.sb = ob.s; k.sc = oc.s;
  k.y = data_or_null(out.y);
  k.h_out = (float*)data_or_null(out.h);
  k.sy = k.sh = dense;
  k.ckpt = (float*)data_or_null(out.ckpt);
  const Tensor h0 = read_state(h_init, h_final);
  k.h_init = floats_or_null(h0);
  k.h_final = (float*)data_or_null(h_final);
  launch(k, plan, x.get_device(), qssm_scan_forward_call);
  return out;
}

struct Grads {
  Tensor g[4];
};

Grads scan_backward(const Tensor& x, const Tensor& a, const Tensor& b, const Tensor& c, const Tensor& dy, const Tensor& h,
                    const Tensor& ckpt, int64_t ckpt_stride, unsigned need, int tune, const Tensor& h_init,
                    const Tensor& dh_final, const Tensor& dh_init) {
  require_gpu({&x, &a, &b, &c, &dy});
  TORCH_CHECK_VALUE(x.dim() == 3 && dy.dim() == 3, "scan operands must be 3-D tensors [B, L, D].");
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2);
  const c10::OptionalDeviceGuard guard(x.device());
  uint64_t bits = (uint64_t)D;
  Grads out;
  for (int i = 0; i < 4; ++i)
    if (need >> i & 1) out.g[i] = fresh(B, L, D, x.scalar_type(), x, &bits);
  check_state(h_init, B, D, x, "h_init");
  check_state(dh_final, B, D, x, "dh_final");
  check_state(dh_init, B, D, x, "dh_init");
  if (B == 0 || L == 0 || D == 0) {   // the state passed through untouched
    if (dh_init.defined()) {
      if (dh_final.defined()) dh_init.copy_(dh_final);
      else dh_init.zero_();
    }
    return out;
  }
  TORCH_CHECK_VALUE(h.defined() != ckpt.defined(), "pass exactly one of h and ckpt");
  TORCH_CHECK_VALUE(B <= INT32_MAX && L <= INT32_MAX && D <= INT32_MAX, "a dimension of the scan does not fit 32 bits");
  const Operand ox(x, bits), oa(a, bits), ob(b, bits), oc(c, bits), og(dy, bits);
  const Operand oh(h.defined() && h.scalar_type() != at::kFloat ? h.to(at::kFloat) : h, bits);
  const Tensor saved = ckpt.defined() ? ckpt.contiguous() : ckpt;
  const qssm_plan plan = plan_for({(int32_t)B, (int32_t)L, (int32_t)D, code_of(x.scalar_type()), code_of(dy.scalar_type()),
                                    QSSM_BACKWARD, align_of(bits), (int32_t)(h.defined() ? 0 : ckpt_stride), tune, 0, -1});
  if (saved.defined())
    TORCH_CHECK_VALUE(saved.dim() == 3 && saved.size(0) == B && saved.size(1) == plan.n_ckpt && saved.size(2) == D &&
                          saved.scalar_type() == at::kFloat,
                      "ckpt has shape ", saved.sizes(), ", expected float32 (", B, ", ", plan.n_ckpt, ", ", D, ")");
  const qssm_strides dense{L * D, D};
  qssm_backward_call k{};
  k.x = ox.p; k.a = oa.p; k.b = ob.p; k.c = oc.p; k.dy = og.p; k.h = (const float*)oh.p;
  k.sx = ox.s; k.sa = oa.s; k.sb = ob.s; k.sc = oc.s; k.sdy = og.s; k.sh = oh.s;
  k.ckpt = floats_or_null(saved);
  const Tensor g_final = read_state(dh_final, dh_init);
  k.h_init = floats_or_null(h_init);
  k.dh_final = floats_or_null(g_final);
  k.dh_init = (float*)data_or_null(dh_init);
  k.dx = data_or_null(out.g[0]); k.da = data_or_null(out.g[1]); k.db = data_or_null(out.g[2]); k.dc = data_or_null(out.g[3]);
  k.sdx = k.sda = k.sdb = k.sdc = dense;
  launch(k, plan, x.get_device(), qssm_scan_backward_call);
  return out;
}

// ---- autograd ----------------------------------------------------------------------------------------------------

Tensor in_dtype(const Tensor& t, at::ScalarType dtype) { return t.scalar_type() == dtype ? t : t.to(dtype); }

// Node of `scan` and `scan_chunk`: (x, a, b, c [, state]) -> y [, final state].  Operands are saved as the caller gave
// them and cast again when the launch stores them in another type; every gradient returns in its operand's type.
struct ScanBackward : public Node {
  SavedVariable x, a, b, c;
  Tensor h, ckpt, h_init;   // what the forward kept: the full fp32 states or those at every `stride`-th step; the state it started from
  int64_t stride = 0;
  int k_in = 0, k_out = 0;
  bool carry = false;                       // second output and fifth input: the states
  at::ScalarType state_dtype = at::kFloat;  // the incoming state's type

  std::string name() const override { return "HipScanBackward"; }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.reset_data();
    a.reset_data();
    b.reset_data();
    c.reset_data();
    h.reset();
    ckpt.reset();
    h_init.reset();
  }

  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const Tensor ox = x.unpack(), oa = a.unpack(), ob = b.unpack(), oc = c.unpack();
    variable_list out(carry ? 5 : 4);
    const bool have_state = carry && grads[1].defined();
    // (no gradient at all, from a function that returns none for y, stands for zeros, as torch.autograd.Function has it)
    c10::AutoGradMode no_grad(false);
    const at::ScalarType in = scalar_of(k_in), go = scalar_of(k_out);
    const Tensor dy = grads[0].defined() ? in_dtype(grads[0], go) : at::zeros(ox.sizes(), ox.options().dtype(go));
    Tensor dh_final, dh_init;
    if (have_state) {
      dh_final = in_dtype(grads[1], at::kFloat).contiguous();
      if ((uintptr_t)dh_final.const_data_ptr() % 16 != 0) dh_final = dh_final.clone();
    }
    if (carry && task_should_compute_output(4)) dh_init = at::empty({ox.size(0), ox.size(2)}, ox.options().dtype(at::kFloat));
    unsigned need = 0;
    for (int i = 0; i < 4; ++i) need |= task_should_compute_output(i) ? 1u << i : 0u;
    Grads g = scan_backward(in_dtype(ox, in), in_dtype(oa, in), in_dtype(ob, in), in_dtype(oc, in), dy, h,
                            h.defined() ? Tensor() : ckpt, stride, need, 0, h_init, dh_final, dh_init);
    const Tensor* like[4] = {&ox, &oa, &ob, &oc};
    for (int i = 0; i < 4; ++i)
      if (g.g[i].defined()) out[i] = in_dtype(g.g[i], like[i]->scalar_type());
    if (dh_init.defined()) out[4] = in_dtype(dh_init, state_dtype);
    return out;
  }
};

// ---- linear maps over fp32 parameters (qssm_gemm_f32) -------------------------------------------------------------

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)t.get_device()).stream(); }

Tensor like_of(std::initializer_list<int64_t> sizes, const Tensor& like, at::ScalarType type) {
  return at::empty(at::IntArrayRef(sizes), like.options().dtype(type).memory_format(c10::nullopt).requires_grad(c10::nullopt));
}

Tensor matrix(int64_t rows, int64_t cols, const Tensor& like) { return like_of({rows, cols}, like, like.scalar_type()); }

// c[i] = a[i] b[i]^T (+ bias[i]), or c[0] = the sum of them all.
void product(const std::vector<Tensor>& a, const std::vector<Tensor>& b, const std::vector<Tensor>& c, int64_t K,
             bool a_kstrided, bool b_kstrided, const std::vector<Tensor>& bias = {}) {
  qssm_gemm_f32_call k{};
  Tensor partial;
  const int batch = (int)c.size();
  for (size_t i = 0; i < a.size(); ++i) {
    k.a[i] = a[i].const_data_ptr<float>();
    k.b[i] = b[i].const_data_ptr<float>();
  }
  for (int i = 0; i < batch; ++i) {
    k.c[i] = c[i].mutable_data_ptr<float>();
    if ((size_t)i < bias.size()) k.bias[i] = floats_or_null(bias[i]);
  }
  k.lda = a[0].stride(0); k.ldb = b[0].stride(0); k.ldc = c[0].stride(0);
  k.M = (int32_t)c[0].size(0); k.N = (int32_t)c[0].size(1); k.K = (int32_t)K;
  k.batch = batch;
  k.segments = batch == 1 ? (int32_t)a.size() : 1;
  k.a_kstrided = a_kstrided;
  k.b_kstrided = b_kstrided;
  uint64_t bytes = 0;
  check_rc(qssm_gemm_f32_packed_plan(&k, &bytes));
  const Tensor packed = like_of({(int64_t)bytes}, c[0], at::kByte);
  if (k.splits > 1) {
    partial = matrix((int64_t)k.splits * batch * k.M, k.N, c[0]);
    k.partial = partial.mutable_data_ptr<float>();
    k.partial_floats = (uint64_t)partial.numel();
  }
  void* const stream = stream_of(c[0]);
  unlocked([&] { return bytes == 0 ? qssm_gemm_f32(&k, stream) : qssm_gemm_f32_packed(&k, packed.mutable_data_ptr(), bytes, stream); });
}

bool matrix_ok(const Tensor& t, int64_t rows, int64_t cols, const Tensor& like) {
  return t.defined() && t.is_cuda() && t.device() == like.device() && t.scalar_type() == at::kFloat && t.dim() == 2 &&
         t.size(0) == rows && t.size(1) == cols && t.stride(1) == 1 && t.stride(0) >= cols && t.stride(0) % 4 == 0 &&
         t.stride(0) < (1 << 20) && (uintptr_t)t.const_data_ptr() % 16 == 0;
}

void check_operands(const Tensor& u, const std::vector<Tensor>& w) {
  TORCH_CHECK_VALUE(!w.empty() && w.size() <= QSSM_GEMM_MANY && u.defined() && u.dim() == 2 && u.size(0) > 0 &&
                        matrix_ok(u, u.size(0), u.size(1), u), "split products need a float32 GPU matrix of 16-byte aligned rows");
  for (const Tensor& t : w)
    TORCH_CHECK_VALUE(matrix_ok(t, w[0].size(0), u.size(1), u) && t.stride(0) == w[0].stride(0),
                      "split products need weights of one shape and layout beside their input");
}

// ---- Python entry points -----------------------------------------------------------------------------------------

const Tensor kNone;

const Tensor& tensor_arg(PyObject* o) {
  if (o == Py_None) return kNone;
  TORCH_CHECK_TYPE(THPVariable_Check(o), "expected a tensor, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}

int64_t int_arg(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred() != nullptr) throw python_error();
  return v;
}

PyObject* wrap_or_none(const Tensor& t) {
  if (t.defined()) return THPVariable_Wrap(t);
  Py_RETURN_NONE;
}

void want_args(Py_ssize_t n, Py_ssize_t want) {
  TORCH_CHECK_TYPE(n == want, "expected ", want, " arguments, got ", n);
}

// (x, a, b, c, out_code, want: 1 y | 2 h | 4 ckpt, keep, tune, bwd_tune, h_init, h_final) -> (y, h, ckpt, stride)
PyObject* py_scan_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 11);
  const Tensor &x = tensor_arg(args[0]), &a = tensor_arg(args[1]), &b = tensor_arg(args[2]), &c = tensor_arg(args[3]);
  const int out_code = (int)int_arg(args[4]), want = (int)int_arg(args[5]), keep = (int)int_arg(args[6]);
  const int tune = (int)int_arg(args[7]), bwd_tune = (int)int_arg(args[8]);
  const Tensor &h_init = tensor_arg(args[9]), &h_final = tensor_arg(args[10]);
  TORCH_CHECK_TYPE(x.defined() && a.defined() && b.defined(), "x, a and b must be tensors");
  ForwardOut out;
  {
    const c10::AutoGradMode no_grad(false);
    out = scan_forward(x, a, b, c, out_code, want & 1, want & 2, want & 4, keep, tune, bwd_tune, h_init, h_final);
  }
  PyObject* r = PyTuple_New(4);
  if (r == nullptr) throw python_error();
  PyTuple_SET_ITEM(r, 0, wrap_or_none(out.y));
  PyTuple_SET_ITEM(r, 1, wrap_or_none(out.h));
  PyTuple_SET_ITEM(r, 2, wrap_or_none(out.ckpt));
  PyTuple_SET_ITEM(r, 3, PyLong_FromLongLong(out.stride));
  return r;
  END_HANDLE_TH_ERRORS
}

// (x, a, b, c, dy, h, ckpt, stride, need, tune, h_init, dh_final, dh_init) -> (dx, da, db, dc)
PyObject* py_scan_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 13);
  for (int i = 0; i < 5; ++i) TORCH_CHECK_TYPE(THPVariable_Check(args[i]), "x, a, b, c and dy must be tensors");
  Grads g;
  {
    const c10::AutoGradMode no_grad(false);
    g = scan_backward(tensor_arg(args[0]), tensor_arg(args[1]), tensor_arg(args[2]), tensor_arg(args[3]), tensor_arg(args[4]),
                      tensor_arg(args[5]), tensor_arg(args[6]), int_arg(args[7]), (unsigned)int_arg(args[8]),
                      (int)int_arg(args[9]), tensor_arg(args[10]), tensor_arg(args[11]), tensor_arg(args[12]));
  }
  PyObject* r = PyTuple_New(4);
  if (r == nullptr) throw python_error();
  for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(r, i, wrap_or_none(g.g[i]));
  return r;
  END_HANDLE_TH_ERRORS
}

// (y, h, ckpt, stride, x, a, b, c, k_in, k_out, final, state, h_init): makes y (and the final state, when there is
// one) outputs of a ScanBackward node over the operands (and the incoming state, or None).  A y of a type that has no
// gradients (integers, bool) stays outside.
PyObject* py_attach_scan(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 13);
  const Tensor y = tensor_arg(args[0]), final_state = tensor_arg(args[10]);
  const Tensor &x = tensor_arg(args[4]), &a = tensor_arg(args[5]), &b = tensor_arg(args[6]), &c = tensor_arg(args[7]);
  const Tensor& state = tensor_arg(args[11]);
  TORCH_CHECK_TYPE(y.defined() && x.defined() && a.defined() && b.defined() && c.defined(), "y, x, a, b, c must be tensors");
  const bool y_has_gradients = torch::autograd::isDifferentiableType(y.scalar_type());
  if (!y_has_gradients && !final_state.defined()) Py_RETURN_NONE;
  std::shared_ptr<ScanBackward> node(new ScanBackward(), torch::autograd::deleteNode);
  node->carry = final_state.defined();
  node->x = SavedVariable(x, false);
  node->a = SavedVariable(a, false);
  node->b = SavedVariable(b, false);
  node->c = SavedVariable(c, false);
  node->h = tensor_arg(args[1]);
  node->ckpt = tensor_arg(args[2]);
  node->stride = int_arg(args[3]);
  node->k_in = (int)int_arg(args[8]);
  node->k_out = (int)int_arg(args[9]);
  node->h_init = tensor_arg(args[12]);
  if (state.defined()) node->state_dtype = state.scalar_type();
  if (node->carry) node->set_next_edges(torch::autograd::collect_next_edges(x, a, b, c, state));
  else node->set_next_edges(torch::autograd::collect_next_edges(x, a, b, c));
  if (y_has_gradients) torch::autograd::set_history(y, node);
  else node->add_input_metadata(Node::undefined_input());
  if (node->carry) torch::autograd::set_history(final_state, node);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

std::vector<Tensor> tensors_arg(PyObject* o) {
  TORCH_CHECK_TYPE(PyTuple_Check(o) || PyList_Check(o), "expected a tuple or list of tensors");
  std::vector<Tensor> v;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
  for (Py_ssize_t i = 0; i < n; ++i) v.push_back(tensor_arg(PySequence_Fast_GET_ITEM(o, i)));
  return v;
}

PyObject* wrap_list(const std::vector<Tensor>& v) {
  PyObject* r = PyList_New((Py_ssize_t)v.size());
  if (r == nullptr) throw python_error();
  for (size_t i = 0; i < v.size(); ++i) PyList_SET_ITEM(r, (Py_ssize_t)i, wrap_or_none(v[i]));
  return r;
}

// (u, weights, biases) -> outputs
PyObject* py_split_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 3);
  const Tensor& u = tensor_arg(args[0]);
  const std::vector<Tensor> w = tensors_arg(args[1]);
  std::vector<Tensor> bias = tensors_arg(args[2]), out;
  check_operands(u, w);
  {
    const c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(u.device());
    const int count = (int)w.size();
    const int64_t N = w[0].size(0);
    TORCH_CHECK_VALUE((int)bias.size() == count, "one bias, or None, for every weight");
    for (Tensor& t : bias)
      if (t.defined()) {
        TORCH_CHECK_VALUE(t.dim() == 1 && t.size(0) == N && t.scalar_type() == at::kFloat && t.device() == u.device(),
                          "a bias must be a float32 vector of the outputs' width");
        t = t.contiguous();
      }
    for (int i = 0; i < count; ++i) out.push_back(matrix(u.size(0), N, u));
    product(std::vector<Tensor>(count, u), w, out, u.size(1), false, false, bias);
  }
  return wrap_list(out);
  END_HANDLE_TH_ERRORS
}

// (gradients of the outputs, u, weights, want: 1 du | 2 dw) -> (du, [dw])
PyObject* py_split_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 4);
  std::vector<Tensor> g = tensors_arg(args[0]), dw;
  const Tensor& u = tensor_arg(args[1]);
  const std::vector<Tensor> w = tensors_arg(args[2]);
  const int64_t want = int_arg(args[3]);
  check_operands(u, w);
  Tensor du;
  {
    const c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(u.device());
    const int count = (int)w.size();
    const int64_t rows = u.size(0), N = w[0].size(0), K = u.size(1);
    TORCH_CHECK_VALUE((int)g.size() == count, "one gradient for every weight");
    bool whole = true;
    for (const Tensor& t : g) {
      TORCH_CHECK_VALUE(t.defined() && t.dim() == 2 && t.size(0) == rows && t.size(1) == N, "a gradient has its output's shape");
      whole = whole && matrix_ok(t, rows, N, u) && t.stride(0) == g[0].stride(0);
    }
    if (!whole)
      for (Tensor& t : g) t = matrix(rows, N, u).copy_(t);
    if (want & 1) {
      du = matrix(rows, K, u);
      product(g, w, {du}, N, false, true);
    }
    if (want & 2) {
      for (int i = 0; i < count; ++i) dw.push_back(matrix(N, K, u));
      product(g, std::vector<Tensor>(count, u), dw, rows, true, true);
    }
  }
  PyObject* r = PyTuple_New(2);
  if (r == nullptr) throw python_error();
  PyTuple_SET_ITEM(r, 0, wrap_or_none(du));
  PyTuple_SET_ITEM(r, 1, wrap_list(dw));
  return r;
  END_HANDLE_TH_ERRORS
}

// Rows of 16-byte pieces next to each other, in one of the storage types of qssm_weight_gradient.
bool rows_of_16_bytes(const Tensor& t) {
  return t.defined() && t.is_cuda() && t.dim() == 2 && t.size(0) > 0 && t.size(1) > 0 &&
         t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.size(1) % 8 == 0 && t.stride(0) % 8 == 0 && t.stride(0) < (1 << 24) &&
         t.size(0) < (1 << 30) && t.size(1) < (1 << 30) && (uintptr_t)t.const_data_ptr() % 16 == 0;
}

// (gradient of a linear map's outputs [rows, N], its inputs [rows, K]) -> the weight's gradient [N, K], or None where the
// library's product is the faster one or this has no kernel for the operands.
PyObject* py_weight_gradient(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 2);
  const Tensor &g = tensor_arg(args[0]), &u = tensor_arg(args[1]);
  Tensor dw;
  if (g.defined() && u.defined() && g.dim() == 2 && u.dim() == 2 && g.size(0) == u.size(0) && g.device() == u.device() &&
      g.scalar_type() == u.scalar_type()) {
    const c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(g.device());
    const at::ScalarType type = g.scalar_type();
    const int64_t rows = g.size(0), N = g.size(1), K = u.size(1);
    if (type == at::kFloat) {
      // (Up to 16 columns of either the library's product is the faster one, us against this: 8192 rows 8 x 8 17 / 25, 80 x 16
      // 26 / 29, 262144 rows 8 x 8 217 / 372, 80 x 16 291 / 371; from 20 on 8192 rows 20 x 20 44 / 27, 262144 rows 32 x 32 453 /
      // 375.)
      if (rows > 0 && matrix_ok(g, rows, N, u) && matrix_ok(u, rows, K, g) && N % 4 == 0 && K % 4 == 0 && N >= 20 && K >= 20 &&
          N < (1 << 30) && K < (1 << 30) && rows < (1 << 30)) {
        dw = matrix(N, K, u);
        product({g}, {u}, {dw}, rows, true, true);
      }
    } else if ((type == at::kHalf || type == at::kBFloat16) && rows_of_16_bytes(g) && rows_of_16_bytes(u) &&
               qssm_weight_gradient_suits((int32_t)N, (int32_t)K, (int32_t)rows) != 0) {
      dw = matrix(N, K, u);
      const uint64_t floats = qssm_weight_gradient_floats((int32_t)N, (int32_t)K, (int32_t)rows);
      Tensor partial;
      if (floats > 0) partial = like_of({(int64_t)floats}, u, at::kFloat);
      unlocked([&] {
        return qssm_weight_gradient(g.const_data_ptr(), g.stride(0), u.const_data_ptr(), u.stride(0), dw.mutable_data_ptr(),
                                    dw.stride(0), (int32_t)N, (int32_t)K, (int32_t)rows, type == at::kHalf ? QSSM_F16 : QSSM_BF16,
                                    floats > 0 ? partial.mutable_data_ptr<float>() : nullptr, floats, stream_of(dw));
      });
    }
  }
  return wrap_or_none(dw);
  END_HANDLE_TH_ERRORS
}

// ---- the layer's other launches ------------------------------------------------------------------------------------
//
// Called inside the layer's autograd functions, which stay in Python; here are the outputs, the scratch and the arguments of
// their launches.  Through ctypes a layer's forward and backward spent about 110 us of the interpreter's time on these.

// Five tensors, or the five column blocks of one.
struct FiveBlocks {
  std::vector<Tensor> t;
  const char* p[5];
  qssm_strides s[5];
};

FiveBlocks blocks_arg(PyObject* o, bool written) {
  FiveBlocks b;
  if (THPVariable_Check(o)) {
    const Tensor& wide = THPVariable_Unpack(o);
    TORCH_CHECK_VALUE(wide.dim() == 3, "expected a [B, L, 5 S] tensor");   // (columns behind the last block are not touched)
    b.t.push_back(wide);
    const int64_t step = wide.size(2) / 5 * wide.element_size();
    for (int k = 0; k < 5; ++k) {
      b.p[k] = (const char*)(written ? wide.mutable_data_ptr() : wide.const_data_ptr()) + k * step;
      b.s[k] = {wide.stride(0), wide.stride(1)};
    }
    return b;
  }
  b.t = tensors_arg(o);
  TORCH_CHECK_VALUE(b.t.size() == 5, "expected five tensors");
  for (int k = 0; k < 5; ++k) {
    TORCH_CHECK_VALUE(b.t[k].defined() && b.t[k].dim() == 3, "expected five tensors [B, L, S]");
    b.p[k] = (const char*)(written ? b.t[k].mutable_data_ptr() : b.t[k].const_data_ptr());
    b.s[k] = {b.t[k].stride(0), b.t[k].stride(1)};
  }
  return b;
}

qssm_strides strides3(const Tensor& t) {
  TORCH_CHECK_VALUE(t.defined() && t.dim() == 3, "expected a tensor [B, L, S]");
  return {t.stride(0), t.stride(1)};
}

// What gated_scan._launch hands on behind a launch's own arguments: control block, workspace, epoch and stream.
struct Taken {
  void* control;
  uint64_t control_size;
  void* workspace;
  uint64_t workspace_size;
  uint32_t epoch;
  void* stream;
  explicit Taken(PyObject* const* a) {
    unsigned long long v[6];
    for (int k = 0; k < 6; ++k) {
      v[k] = PyLong_AsUnsignedLongLong(a[k]);
      if (v[k] == (unsigned long long)-1 && PyErr_Occurred() != nullptr) throw python_error();
    }
    control = (void*)(uintptr_t)v[0];
    control_size = v[1];
    workspace = (void*)(uintptr_t)v[2];
    workspace_size = v[3];
    epoch = (uint32_t)v[4];
    stream = (void*)(uintptr_t)v[5];
  }
};

const qssm_plan* plan_arg(PyObject* o) {
  const unsigned long long v = PyLong_AsUnsignedLongLong(o);
  if (v == (unsigned long long)-1 && PyErr_Occurred() != nullptr) throw python_error();
  return (const qssm_plan*)(uintptr_t)v;
}

// (plan's address, projection outputs: five or one wide, y, ckpt, control ...) -> return code
PyObject* py_gated_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 10);
  const qssm_plan* plan = plan_arg(args[0]);
  const FiveBlocks pre = blocks_arg(args[1], false);
  const Tensor &y = tensor_arg(args[2]), &ckpt = tensor_arg(args[3]);
  const Taken to(args + 4);
  const qssm_strides sy = strides3(y);
  void* yp = y.mutable_data_ptr();
  float* cp = ckpt.mutable_data_ptr<float>();
  int rc;
  {
    const Unlocked other_threads_may_run;
    rc = qssm_scan_gated_forward(plan, pre.p[0], pre.s[0], pre.p[1], pre.s[1], pre.p[2], pre.s[2], pre.p[3], pre.s[3], pre.p[4],
                                 pre.s[4], yp, sy, cp, to.control, to.control_size, to.workspace, to.workspace_size, to.epoch,
                                 to.stream);
  }
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

// (plan's address, projection outputs, dy, ckpt, gradients: five or one wide, control ...) -> return code
PyObject* py_gated_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 11);
  const qssm_plan* plan = plan_arg(args[0]);
  const FiveBlocks pre = blocks_arg(args[1], false), grad = blocks_arg(args[4], true);
  const Tensor &dy = tensor_arg(args[2]), &ckpt = tensor_arg(args[3]);
  const Taken to(args + 5);
  const qssm_strides sdy = strides3(dy);
  const void* dyp = dy.const_data_ptr();
  const float* cp = ckpt.const_data_ptr<float>();
  void* g[5];
  for (int k = 0; k < 5; ++k) g[k] = const_cast<char*>(grad.p[k]);
  int rc;
  {
    const Unlocked other_threads_may_run;
    rc = qssm_scan_gated_backward(plan, pre.p[0], pre.s[0], pre.p[1], pre.s[1], pre.p[2], pre.s[2], pre.p[3], pre.s[3], pre.p[4],
                                  pre.s[4], dyp, sdy, cp, g[0], grad.s[0], g[1], grad.s[1], g[2], grad.s[2], g[3], grad.s[3],
                                  g[4], grad.s[4], to.control, to.control_size, to.workspace, to.workspace_size, to.epoch,
                                  to.stream);
  }
  return PyLong_FromLong(rc);
  END_HANDLE_TH_ERRORS
}

int64_t row_stride(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }

// (x [rows, H], weight, eps) -> (y, rstd)
PyObject* py_rmsnorm_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 3);
  const Tensor &x = tensor_arg(args[0]), &w = tensor_arg(args[1]);
  const double eps = PyFloat_AsDouble(args[2]);
  if (eps == -1.0 && PyErr_Occurred() != nullptr) throw python_error();
  TORCH_CHECK_VALUE(x.defined() && w.defined() && x.dim() == 2, "expected a [rows, H] matrix and its weight");
  Tensor y, rstd;
  {
    const c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(x.device());
    const int64_t rows = x.size(0), H = x.size(1);
    TORCH_CHECK_VALUE(H <= INT32_MAX, "a row does not fit 32 bits");
    y = like_of({rows, H}, x, x.scalar_type());
    rstd = like_of({rows}, x, at::kFloat);
    const int type = code_of(x.scalar_type());
    unlocked([&] {
      return qssm_rmsnorm_forward(x.const_data_ptr(), row_stride(x), w.const_data_ptr(), y.mutable_data_ptr(),
                                  rstd.mutable_data_ptr<float>(), rows, (int32_t)H, (float)eps, type, stream_of(x));
    });
  }
  return Py_BuildValue("(NN)", THPVariable_Wrap(y), THPVariable_Wrap(rstd));
  END_HANDLE_TH_ERRORS
}

// (dy [rows, H], x [rows, H], weight, rstd, eps, rows of scratch) -> (dx, dweight)
PyObject* py_rmsnorm_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 6);
  const Tensor &dy = tensor_arg(args[0]), &x = tensor_arg(args[1]), &w = tensor_arg(args[2]), &rstd = tensor_arg(args[3]);
  const double eps = PyFloat_AsDouble(args[4]);
  if (eps == -1.0 && PyErr_Occurred() != nullptr) throw python_error();
  const int64_t scratch = int_arg(args[5]);
  TORCH_CHECK_VALUE(dy.defined() && x.defined() && w.defined() && rstd.defined() && x.dim() == 2 && dy.sizes() == x.sizes(),
                    "expected two [rows, H] matrices, the weight and what the forward saved");
  Tensor dx, dw;
  {
    const c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(x.device());
    const int64_t rows = x.size(0), H = x.size(1);
    TORCH_CHECK_VALUE(H <= INT32_MAX && scratch <= INT32_MAX, "a row does not fit 32 bits");
    dx = like_of({rows, H}, x, x.scalar_type());
    dw = like_of({H}, x, w.scalar_type());
    const Tensor partial = like_of({scratch, H}, x, at::kFloat);
    const int type = code_of(x.scalar_type());
    unlocked([&] {
      return qssm_rmsnorm_backward(dy.const_data_ptr(), row_stride(dy), x.const_data_ptr(), row_stride(x), w.const_data_ptr(),
                                   rstd.const_data_ptr<float>(), dx.mutable_data_ptr(), dw.mutable_data_ptr(),
                                   partial.mutable_data_ptr<float>(), (int32_t)scratch, rows, (int32_t)H, (float)eps, type,
                                   stream_of(x));
    });
  }
  return Py_BuildValue("(NN)", THPVariable_Wrap(dx), THPVariable_Wrap(dw));
  END_HANDLE_TH_ERRORS
}

// ([rows, S] matrix, rows of scratch) -> its column sums
PyObject* py_column_sum(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 2);
  const Tensor& g = tensor_arg(args[0]);
  const int64_t scratch = int_arg(args[1]);
  TORCH_CHECK_VALUE(g.defined() && g.dim() == 2 && g.size(1) <= INT32_MAX && scratch <= INT32_MAX, "expected a [rows, S] matrix");
  Tensor out;
  {
    const c10::AutoGradMode no_grad(false);
    const c10::OptionalDeviceGuard guard(g.device());
    out = like_of({g.size(1)}, g, g.scalar_type());
    const Tensor partial = like_of({scratch, g.size(1)}, g, at::kFloat);
    const int type = code_of(g.scalar_type());
    unlocked([&] {
      return qssm_colsum(g.const_data_ptr(), g.stride(0), g.size(0), (int32_t)g.size(1), type, partial.mutable_data_ptr<float>(),
                         (int32_t)scratch, out.mutable_data_ptr(), stream_of(g));
    });
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject* node_h_saved(PyObject* self, void*) {
  HANDLE_TH_ERRORS
  auto* node = static_cast<ScanBackward*>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get());
  return wrap_or_none(node->h);
  END_HANDLE_TH_ERRORS
}

PyTypeObject g_node_type;
PyMethodDef g_node_methods[] = {{"_register_hook_dict", torch::autograd::THPCppFunction_register_hook_dict, METH_O, nullptr},
                                {"register_hook", torch::autograd::THPCppFunction_register_hook, METH_O, nullptr},
                                {"register_prehook", torch::autograd::THPCppFunction_register_prehook, METH_O, nullptr},
                                {"name", torch::autograd::THPCppFunction_name, METH_NOARGS, nullptr},
                                {"_sequence_nr", torch::autograd::THPCppFunction_sequence_nr, METH_NOARGS, nullptr},
                                {nullptr, nullptr, 0, nullptr}};
PyGetSetDef g_node_properties[] = {{"next_functions", torch::autograd::THPCppFunction_next_functions, nullptr, nullptr, nullptr},
                                   {"requires_grad", torch::autograd::THPCppFunction_requires_grad, nullptr, nullptr, nullptr},
                                   {"metadata", torch::autograd::THPCppFunction_metadata, nullptr, nullptr, nullptr},
                                   {"_input_metadata", torch::autograd::THPCppFunction_input_metadata, nullptr, nullptr, nullptr},
                                   {"h_saved", node_h_saved, nullptr, nullptr, nullptr},
                                   {nullptr, nullptr, nullptr, nullptr, nullptr}};

// (take_launch, check): the callables of quick_ssm_amd this module works with.
PyObject* py_set_hooks(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  want_args(n, 2);
  Py_INCREF(args[0]);
  Py_INCREF(args[1]);
  g_take_launch = args[0];
  g_check = args[1];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define QSSM_METHOD(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {QSSM_METHOD("set_hooks", py_set_hooks), QSSM_METHOD("scan_forward", py_scan_forward),
                           QSSM_METHOD("scan_backward", py_scan_backward), QSSM_METHOD("attach_scan", py_attach_scan),
                           QSSM_METHOD("split_forward", py_split_forward), QSSM_METHOD("split_backward", py_split_backward),
                           QSSM_METHOD("weight_gradient", py_weight_gradient), QSSM_METHOD("gated_forward", py_gated_forward),
                           QSSM_METHOD("gated_backward", py_gated_backward), QSSM_METHOD("rmsnorm_forward", py_rmsnorm_forward),
                           QSSM_METHOD("rmsnorm_backward", py_rmsnorm_backward), QSSM_METHOD("column_sum", py_column_sum),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_qssm_torch", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__qssm_torch() {
  PyObject* m = PyModule_Create(&g_module);
  if (m == nullptr) return nullptr;
  torch::autograd::_initFunctionPyTypeObject(g_node_type, "HipScanBackward", g_node_properties, g_node_methods);
  Py_INCREF(&g_node_type);
  if (PyModule_AddObject(m, "HipScanBackward", reinterpret_cast<PyObject*>(&g_node_type)) < 0) return nullptr;
  torch::autograd::registerCppFunction(typeid(ScanBackward), &g_node_type);
  PyModule_AddIntConstant(m, "abi_version", QSSM_VERSION);
  return m;
}
