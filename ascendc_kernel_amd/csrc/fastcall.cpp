// Calls of the modules' forwards with the layouts of the calls before them, natively: the
// checks, the output's allocation and the launches. A Python module checks and marshals a call
// (_native.Prepared, task2_indexer._IndexerPlan) in 40-100 us of host time, or takes 4-8 us
// besides the launches where it finds the very same tensors again. Once two calls in a row that
// no plan served have had the same layouts it hands its marshalled launches to make(), and run() serves further
// calls of those layouts, whatever their tensors, stream and decode position. Repeated calls,
// before and after: 160 tokens x 64 heads over 32 rows 7.2 -> 5.7 us, an 8-token decode step of
// the 16-head indexer 15.5 -> 10.7 us, the kernels' own time in both.
//
// Nothing of a plan depends on an address or on a tensor's identity: every pointer, the
// stream, the positions and the scratch memory (fresh from torch's caching allocator) are
// filled in per call, into a copy of the arguments of the call's own, so that a plan serves
// several threads and streams.
//
// run() returns None, and the module takes its Python path (which prepares anew, or raises),
// wherever a layout differs: sizes, strides, dtype, device, dispatch keys (wrapped or batched
// tensors), a pointer that is not 16-byte aligned, a scalar, an active dispatch or function
// mode, a position out of the plan's range, a launch that was refused.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <memory>
#include <vector>

#include "../../include/dsa_abi.h"

namespace py = pybind11;

namespace {

constexpr int kMaxArgs = 24;

// The entry points by their declarations in include/dsa_abi.h, argument positions as there. (The
// _i64 ones, and dsa_indexer_decode_projections_rope of kProj, differ from the one called in what
// pointers point to.)
enum Kind { kAttn = 0, kMla = 1, kMlaWs = 2, kScore = 3, kScoreWs = 4, kProj = 5 };
constexpr int kArgs[] = {14, 15, 17, 19, 21, 17};

constexpr int kMaxCalls = 2, kMaxTensors = 8;

struct Call {
  int kind;
  void* fn;
  int64_t a[kMaxArgs];
  float f;  // the one float argument (its position in `a` is unused)
};

// A pointer argument, whatever it points to.
struct Ptr {
  int64_t v;
  template <typename T>
  operator T*() const {
    return reinterpret_cast<T*>(static_cast<uintptr_t>(v));
  }
};

int invoke(const Call& c) {
  const int64_t* a = c.a;
  auto p = [a](int i) { return Ptr{a[i]}; };
  auto i32 = [a](int i) { return static_cast<int32_t>(a[i]); };
  switch (c.kind) {
    case kAttn:
      return reinterpret_cast<decltype(&dsa_sparse_attn_fwd)>(c.fn)(
          p(0), p(1), p(2), p(3), p(4), a[5], a[6], a[7], a[8], a[9], a[10], c.f, i32(12), p(13));
    case kMla:
      return reinterpret_cast<decltype(&dsa_sparse_mla_fwd)>(c.fn)(
          p(0), p(1), p(2), p(3), p(4), a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], c.f, p(14));
    case kMlaWs:
      return reinterpret_cast<decltype(&dsa_sparse_mla_fwd_ws)>(c.fn)(
          p(0), p(1), p(2), p(3), p(4), a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], c.f, p(14), a[15],
          p(16));
    case kScore:
      return reinterpret_cast<decltype(&dsa_indexer_score_topk)>(c.fn)(
          p(0), p(1), a[2], p(3), c.f, p(5), i32(6), p(7), a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15],
          i32(16), a[17], p(18));
    case kScoreWs:
      return reinterpret_cast<decltype(&dsa_indexer_score_topk_ws)>(c.fn)(
          p(0), p(1), a[2], p(3), c.f, p(5), i32(6), p(7), a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15],
          i32(16), a[17], p(18), a[19], p(20));
    case kProj:
      return reinterpret_cast<decltype(&dsa_indexer_projections_splitk)>(c.fn)(
          p(0), p(1), p(2), i32(3), p(4), p(5), p(6), p(7), a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15],
          p(16));
  }
  return -1;
}

struct Layout {
  uint64_t keys;
  std::vector<int64_t> sizes, strides;
  at::ScalarType dtype;
  c10::Device device = c10::kCPU;
};

// What a pointer argument is filled with: a tensor of the call (its index) or one of these.
constexpr int kOut = -1, kTemp = -2, kStream = -3;
struct Patch {
  int call, slot, source;
  int64_t offset;  // bytes
};

// An indexer's forward: start_pos and offset vary from call to call (the last two ints of run).
struct Positions {
  bool causal;                    // start_pos == 0; a plan stays with one of the two
  int64_t s, ratio, topk;
  int64_t table_rows, row_bytes;  // RoPE table: the call's rows begin at start_pos
  int64_t kv_rows;
  int proj, freqs_slot, score;    // the calls, and the projection's table argument
  int64_t ws_off;                 // the score workspace in the temporary (-1: none)
};

constexpr int kScoreCand = 13, kScoreK = 14, kScoreOffset = 17, kScoreWsPtr = 18, kScoreWsBytes = 19;

struct Plan {
  std::vector<Layout> tensors;
  std::vector<py::object> scalars;
  c10::Device device = c10::kCPU;
  std::vector<Call> calls;
  std::vector<Patch> patches;
  std::vector<int64_t> out_sizes;
  at::TensorOptions out_options;
  int64_t temp_bytes = 0;
  bool positioned = false;
  Positions pos{};
  int64_t (*ws_bytes)(int64_t, int64_t, int64_t, int64_t, int64_t) = nullptr;
};

bool same(const at::Tensor& t, const Layout& e) {
  return t.unsafeGetTensorImpl()->key_set().raw_repr() == e.keys && t.scalar_type() == e.dtype &&
         t.device() == e.device && t.sizes().equals(e.sizes) && t.strides().equals(e.strides) &&
         reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

bool same(PyObject* got, PyObject* want) {
  if (got == want) return true;
  if (Py_TYPE(got) != Py_TYPE(want)) return false;
  if (PyFloat_CheckExact(got)) return PyFloat_AS_DOUBLE(got) == PyFloat_AS_DOUBLE(want);
  if (!PyLong_CheckExact(got)) return false;
  int a = 0, b = 0;
  return PyLong_AsLongLongAndOverflow(got, &a) == PyLong_AsLongLongAndOverflow(want, &b) && !a && !b;
}

constexpr const char* kCapsule = "dsa_fastcall_plan";
void destroy(PyObject* o) { delete static_cast<Plan*>(PyCapsule_GetPointer(o, kCapsule)); }

// make(tensors, scalars, calls, patches, out_sizes, out_like, temp_bytes, positions, ws_fn):
//   calls      [(kind, address, [args], float)]
//   patches    [(call, slot, source, byte offset)]
//   out_like   index of the tensor whose dtype the output has (-1: int64)
//   positions  None or Positions' fields in order; ws_fn dsa_indexer_workspace_bytes
// The plan, or None where a tensor could not be served.
py::object make(py::tuple tensors, py::tuple scalars, py::list calls, py::list patches, std::vector<int64_t> out_sizes,
                int out_like, int64_t temp_bytes, py::object positions, uintptr_t ws_fn) {
  auto plan = std::make_unique<Plan>();
  for (auto h : tensors) {
    if (!THPVariable_CheckExact(h.ptr())) return py::none();
    const at::Tensor& t = THPVariable_Unpack(h.ptr());
    Layout e;
    e.keys = t.unsafeGetTensorImpl()->key_set().raw_repr();
    e.sizes = t.sizes().vec();
    e.strides = t.strides().vec();
    e.dtype = t.scalar_type();
    e.device = t.device();
    if (!same(t, e)) return py::none();  // misaligned
    plan->tensors.push_back(std::move(e));
  }
  for (auto h : scalars) {
    PyObject* o = h.ptr();
    // Plain values only: an object that can change in place would still be the plan's own.
    if (o != Py_None && !PyLong_Check(o) && !PyFloat_Check(o)) return py::none();
    plan->scalars.push_back(py::reinterpret_borrow<py::object>(h));
  }
  plan->device = plan->tensors.at(0).device;
  for (const Layout& e : plan->tensors)
    if (e.device != plan->device) return py::none();
  for (auto h : calls) {
    auto c = py::cast<py::tuple>(h);
    Call call{};
    call.kind = c[0].cast<int>();
    call.fn = reinterpret_cast<void*>(c[1].cast<uintptr_t>());
    const auto args = c[2].cast<std::vector<int64_t>>();
    if (call.kind < 0 || call.kind > kProj || (int)args.size() != kArgs[call.kind])
      throw std::invalid_argument("fastcall: call");
    std::copy(args.begin(), args.end(), call.a);
    call.f = c[3].cast<float>();
    plan->calls.push_back(call);
  }
  const int n_calls = (int)plan->calls.size(), n_tensors = (int)plan->tensors.size();
  if (n_calls > kMaxCalls) throw std::invalid_argument("fastcall: calls");
  for (auto h : patches) {
    auto t = py::cast<py::tuple>(h);
    Patch p{t[0].cast<int>(), t[1].cast<int>(), t[2].cast<int>(), t[3].cast<int64_t>()};
    if (p.call < 0 || p.call >= n_calls || p.slot < 0 || p.slot >= kArgs[plan->calls[p.call].kind] ||
        p.source < kStream || p.source >= n_tensors)
      throw std::invalid_argument("fastcall: patch");
    plan->patches.push_back(p);
  }
  plan->out_sizes = std::move(out_sizes);
  plan->out_options = at::TensorOptions().device(plan->device).dtype(
      out_like < 0 ? at::kLong : plan->tensors.at(out_like).dtype);
  plan->temp_bytes = temp_bytes;
  if (!positions.is_none()) {
    auto t = py::cast<py::tuple>(positions);
    plan->positioned = true;
    plan->pos = Positions{t[0].cast<bool>(),    t[1].cast<int64_t>(), t[2].cast<int64_t>(), t[3].cast<int64_t>(),
                          t[4].cast<int64_t>(), t[5].cast<int64_t>(), t[6].cast<int64_t>(), t[7].cast<int>(),
                          t[8].cast<int>(),     t[9].cast<int>(),     t[10].cast<int64_t>()};
    const Positions& p = plan->pos;
    const int want = p.ws_off < 0 ? kScore : kScoreWs;
    if (p.ratio < 1 || p.s < 1 || p.row_bytes % 16 || p.proj < 0 || p.proj >= n_calls || p.score < 0 ||
        p.score >= n_calls || plan->calls[p.proj].kind != kProj || plan->calls[p.score].kind != want ||
        p.freqs_slot < 0 || p.freqs_slot >= kArgs[kProj] || plan->out_sizes.empty())
      throw std::invalid_argument("fastcall: positions");
    plan->ws_bytes = reinterpret_cast<decltype(plan->ws_bytes)>(ws_fn);
  }
  return py::reinterpret_steal<py::object>(PyCapsule_New(plan.release(), kCapsule, destroy));
}

// Output and launches of one call; an undefined tensor where a launch was refused.
at::Tensor launch(const Plan& plan, const void* const* ptrs, int64_t start_pos, int64_t offset) {
  Call calls[kMaxCalls];
  std::copy(plan.calls.begin(), plan.calls.end(), calls);
  int64_t out_last = plan.out_sizes.back(), temp_bytes = plan.temp_bytes;
  if (plan.positioned) {
    const Positions& p = plan.pos;
    if (start_pos < 0 || (start_pos == 0) != p.causal || start_pos > p.table_rows - p.s) return {};
    const int64_t n_cand = (start_pos + p.s) / p.ratio;
    out_last = std::min(p.topk, n_cand);
    if (out_last < 1 || n_cand > p.kv_rows) return {};
    int64_t* a = calls[p.score].a;
    a[kScoreCand] = n_cand;
    a[kScoreK] = out_last;
    a[kScoreOffset] = offset;
    const int64_t need = plan.ws_bytes(a[8], a[9], a[10], a[11], n_cand);
    if (need < 0 || (need > 0) != (p.ws_off >= 0)) return {};
    if (need > 0) {
      a[kScoreWsBytes] = need;
      temp_bytes = p.ws_off + need;
    }
  }
  at::Tensor temp;
  uintptr_t temp_ptr = 0, stream = 0;
  if (plan.device.is_cuda()) {
    if (c10::hip::current_device() != plan.device.index()) return {};
    stream = reinterpret_cast<uintptr_t>(c10::hip::getCurrentHIPStream(plan.device.index()).stream());
  }
  if (temp_bytes > 0) {
    temp = at::empty({temp_bytes}, plan.out_options.dtype(at::kByte));
    temp_ptr = reinterpret_cast<uintptr_t>(temp.const_data_ptr());
  }
  c10::SmallVector<int64_t, 5> sizes(plan.out_sizes.begin(), plan.out_sizes.end());
  sizes.back() = out_last;
  at::Tensor out = at::empty(sizes, plan.out_options);
  for (const Patch& p : plan.patches) {
    const uintptr_t base = p.source == kOut      ? reinterpret_cast<uintptr_t>(out.const_data_ptr())
                           : p.source == kTemp   ? temp_ptr
                           : p.source == kStream ? stream
                                                 : reinterpret_cast<uintptr_t>(ptrs[p.source]);
    calls[p.call].a[p.slot] = static_cast<int64_t>(base + p.offset);
  }
  if (plan.positioned) calls[plan.pos.proj].a[plan.pos.freqs_slot] += start_pos * plan.pos.row_bytes;
  for (size_t i = 0; i < plan.calls.size(); ++i)
    if (invoke(calls[i]) != 0) return {};
  // (The temporary is released here: the caching allocator hands its memory only to later
  // work on this stream.)
  return out;
}

// An active dispatch or function mode sees every call of torch, so calls take the Python path.
bool mode_active() { return c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled(); }

// The plan of args = (plan, tensors..., scalars..., ...) if the tensors' layouts (their pointers in
// ptrs) and the scalars are its own, else null. positions: the call's two follow.
const Plan* match(PyObject* const* args, Py_ssize_t nargs, const void** ptrs, bool positions) {
  const auto* plan = nargs > 0 ? static_cast<const Plan*>(PyCapsule_GetPointer(args[0], kCapsule)) : nullptr;
  if (plan == nullptr) {
    PyErr_Clear();
    return nullptr;
  }
  const size_t nt = plan->tensors.size(), ns = plan->scalars.size(), np = positions && plan->positioned ? 2 : 0;
  if ((size_t)nargs != 1 + nt + ns + np || nt > kMaxTensors || mode_active()) return nullptr;
  for (size_t i = 0; i < nt; ++i) {
    if (!THPVariable_CheckExact(args[1 + i])) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(args[1 + i]);
    if (!same(t, plan->tensors[i])) return nullptr;
    ptrs[i] = t.const_data_ptr();
  }
  for (size_t i = 0; i < ns; ++i)
    if (!same(args[1 + nt + i], plan->scalars[i].ptr())) return nullptr;
  return plan;
}

// run(plan, tensors..., scalars..., [start_pos, offset]): the output, or None.
PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const void* ptrs[kMaxTensors];
  const Plan* plan = match(args, nargs, ptrs, true);
  if (plan == nullptr) Py_RETURN_NONE;
  int64_t pos[2] = {0, 0};
  for (int i = 0; i < (plan->positioned ? 2 : 0); ++i) {
    PyObject* o = args[nargs - 2 + i];
    int overflow = 0;
    if (!PyLong_CheckExact(o)) Py_RETURN_NONE;
    pos[i] = PyLong_AsLongLongAndOverflow(o, &overflow);
    if (overflow) Py_RETURN_NONE;
  }
  at::Tensor out;
  {
    py::gil_scoped_release no_gil;  // (the caller's argument list keeps plan and tensors alive)
    out = launch(*plan, ptrs, pos[0], pos[1]);
  }
  if (!out.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// serves(plan, tensors..., scalars...): whether run() takes these (positions aside).
PyObject* serves(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const void* ptrs[kMaxTensors];
  return PyBool_FromLong(match(args, nargs, ptrs, false) != nullptr);
  END_HANDLE_TH_ERRORS
}

PyMethodDef kRun = {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(run)), METH_FASTCALL, nullptr};
PyMethodDef kServes = {"serves", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(serves)),
                       METH_FASTCALL, nullptr};

}  // namespace

PYBIND11_MODULE(_fastcall, m) {
  m.def("make", &make);
  // Whether calls of tensors on this device are served now, whatever their layout.
  m.def("ready", [](int device) { return !mode_active() && c10::hip::current_device() == device; });
  m.attr("MAX_TENSORS") = kMaxTensors;
  m.attr("ABI_VERSION") = DSA_ABI_VERSION;
  m.add_object("run", py::reinterpret_steal<py::object>(PyCFunction_NewEx(&kRun, nullptr, nullptr)));
  m.add_object("serves", py::reinterpret_steal<py::object>(PyCFunction_NewEx(&kServes, nullptr, nullptr)));
}
