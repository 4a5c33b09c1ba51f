// Host side of the usual call of HipLoRABackend.add_lora (nanovllm_voxcpm_amd/lora.py), in C++.
//
// The backend mirrors the reference's LoRABackend.add_lora (reference: nanovllm_voxcpm/lora.py:43-54,
// body :241-381): one Python call per LoRA linear and step.  Such a call costs the interpreter
// several microseconds of tensor attribute reads and checks before the launch, which takes about
// four; a decode step of 96 calls is then bound by the host, not by the GPU.  This module does the
// same reads and checks on the tensors' C++ objects.  It decides nothing by itself: it handles a
// call only when everything the Python path would look up for it is what the Python path looked up
// last time (the argument block of these weight buffers, the plan of this step's slot vector, the
// scratch buffer of this stream), fills the per-step fields of the block and calls mlora_add_lora_counts.
// One lookup it makes itself: the first call of a step whose slot vector carries a plan (take_step below).
// Everything else - a first call of these buffers, a step without a plan, a capture in progress, anything
// that has to raise - is answered with "not handled", and the Python path runs as if this module did not
// exist, then tells it what it found (register_site, set_step, set_scratch).
//
// One state object per backend and thread; every function runs under the interpreter lock.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

#include "mlora.h"

namespace {

constexpr long kNotHandled = 1;  // what call() returns when the Python path has to run

struct Site {
  MloraAddArgs* args = nullptr;
  PyObject* keep = nullptr;  // the object that owns the block
  int k = 0, rank = 0, num_slots = 0, num_slices = 0, device = 0, form = 0, dtype_code = 0;
  bool vectorisable = false;
  c10::ScalarType dtype = c10::ScalarType::Undefined;
  std::vector<int64_t> widths;
};

struct State {
  int (*add_lora)(const MloraAddArgs*, int32_t, int32_t) = nullptr;  // mlora_add_lora_counts
  size_t (*workspace_bytes)(int32_t, int32_t, int32_t, int32_t) = nullptr;
  std::unordered_map<std::string, Site> sites;
  // what the last call of the Python path looked up for its step
  const PyObject* metadata = nullptr;
  const PyObject* source = nullptr;
  uint32_t version = 0;
  void* stream = nullptr;
  int num_slots = 0, active_slots = 0, active_tokens = 0;
  int64_t rows = -1;
  const void* plan = nullptr;
  PyObject* held[3] = {};  // metadata, slot vector and plan of a step that was taken here (set_step's are its caller's to hold)
  // the eager scratch buffer of a stream
  void* sc_stream = nullptr;
  int sc_device = -1;
  void* sc_ptr = nullptr;
  int64_t sc_bytes = 0;
  // bytes of scratch a shape asks for
  std::unordered_map<uint64_t, int64_t> need;
  long long handled = 0, passed_on = 0;  // calls enqueued here / left to the Python path

  ~State() {
    for (PyObject* o : held) Py_XDECREF(o);
    for (auto& kv : sites) Py_XDECREF(kv.second.keep);
  }
};

const char* kCapsule = "mlora.fastcall.state";

State* state_of(PyObject* capsule) { return static_cast<State*>(PyCapsule_GetPointer(capsule, kCapsule)); }

void destroy(PyObject* capsule) { delete static_cast<State*>(PyCapsule_GetPointer(capsule, kCapsule)); }

// Key of a set of weight buffers: address and shape of every A and B slice, and the element type.
// False when something in the lists is not a contiguous tensor.
bool weights_key(PyObject* a_list, PyObject* b_list, Py_ssize_t n, std::string* key, const at::Tensor** a0) {
  int64_t buf[2 * MLORA_MAX_SLICES * 5 + 1];
  int at = 0;
  for (PyObject* list : {a_list, b_list}) {
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* o = PySequence_Fast_GET_ITEM(list, i);
      if (!THPVariable_Check(o)) return false;
      const at::Tensor& t = THPVariable_Unpack(o);
      if (t.dim() != 3 || !t.is_contiguous()) return false;
      if (list == a_list && i == 0) *a0 = &t;
      buf[at++] = reinterpret_cast<int64_t>(t.data_ptr());
      buf[at++] = t.size(0);
      buf[at++] = t.size(1);
      buf[at++] = t.size(2);
    }
  }
  buf[at++] = static_cast<int64_t>((*a0)->scalar_type());
  key->assign(reinterpret_cast<const char*>(buf), static_cast<size_t>(at) * sizeof(int64_t));
  return true;
}

struct Ref {  // an owned reference, given back at the end of the scope
  PyObject* p;
  ~Ref() { Py_XDECREF(p); }
};

// Gives back, at the end of the scope, the objects of a step that stands no longer: the state is consistent by then.
struct Released {
  PyObject* p[3] = {};
  explicit Released(State* s) { std::swap(p, s->held); }
  ~Released() { for (PyObject* o : p) Py_XDECREF(o); }
};

bool on_device(const at::Tensor& t, int device) { return t.is_cuda() && t.device().index() == device; }

PyObject* py_create(PyObject*, PyObject* args) {
  unsigned long long add = 0, ws = 0;
  if (!PyArg_ParseTuple(args, "KK", &add, &ws)) return nullptr;
  State* s = new State();
  s->add_lora = reinterpret_cast<int (*)(const MloraAddArgs*, int32_t, int32_t)>(static_cast<uintptr_t>(add));
  s->workspace_bytes = reinterpret_cast<size_t (*)(int32_t, int32_t, int32_t, int32_t)>(static_cast<uintptr_t>(ws));
  return PyCapsule_New(s, kCapsule, destroy);
}

// register_site(state, a_list, b_list, widths, block address, block owner, vectorisable)
PyObject* py_register_site(PyObject*, PyObject* args) {
  PyObject *cap, *a_list, *b_list, *widths, *keep;
  unsigned long long addr = 0;
  int vectorisable = 0;
  if (!PyArg_ParseTuple(args, "OOOOKOp", &cap, &a_list, &b_list, &widths, &addr, &keep, &vectorisable)) return nullptr;
  State* s = state_of(cap);
  if (!s) return nullptr;
  PyObject* af = PySequence_Fast(a_list, "lora_a slices");
  PyObject* bf = af ? PySequence_Fast(b_list, "lora_b slices") : nullptr;
  PyObject* wf = bf ? PySequence_Fast(widths, "widths") : nullptr;
  bool ok = false;
  if (wf) {
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(af);
    std::string key;
    const at::Tensor* a0 = nullptr;
    if (n >= 1 && n <= MLORA_MAX_SLICES && PySequence_Fast_GET_SIZE(bf) == n && PySequence_Fast_GET_SIZE(wf) == n &&
        weights_key(af, bf, n, &key, &a0) && a0->is_cuda()) {
      Site site;
      site.args = reinterpret_cast<MloraAddArgs*>(static_cast<uintptr_t>(addr));
      site.k = site.args->k; site.rank = site.args->r; site.num_slots = site.args->num_slots; site.num_slices = site.args->num_slices;
      site.form = site.args->form; site.dtype_code = site.args->dtype;
      site.device = a0->device().index();
      site.dtype = a0->scalar_type();
      site.vectorisable = vectorisable != 0;
      ok = site.num_slices == n;
      for (Py_ssize_t i = 0; ok && i < n; ++i) {
        const long long w = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(wf, i));
        if (w == -1 && PyErr_Occurred()) { PyErr_Clear(); ok = false; }
        site.widths.push_back(w);
      }
      if (ok) {
        auto it = s->sites.find(key);
        if (it != s->sites.end()) {
          Py_XDECREF(it->second.keep);
          s->sites.erase(it);
        }
        Py_INCREF(keep);
        site.keep = keep;
        s->sites.emplace(std::move(key), std::move(site));
      }
    }
  }
  Py_XDECREF(wf); Py_XDECREF(bf); Py_XDECREF(af);
  if (PyErr_Occurred()) return nullptr;
  return PyBool_FromLong(ok);
}

PyObject* py_clear_sites(PyObject*, PyObject* cap) {
  State* s = state_of(cap);
  if (!s) return nullptr;
  for (auto& kv : s->sites) Py_XDECREF(kv.second.keep);
  s->sites.clear();
  Py_RETURN_NONE;
}

// set_step(state, metadata, source, version, stream, num_slots, rows, plan address, tokens with a slot, active slots): what a call
// outside any capture looked up; the caller keeps metadata, source and the plan alive for as long
// as this stands.  forget_step(state) withdraws it.
PyObject* py_set_step(PyObject*, PyObject* args) {
  PyObject *cap, *metadata, *source;
  unsigned long version = 0;
  unsigned long long stream = 0, plan = 0;
  int num_slots = 0, active_tokens = 0, active_slots = 0;
  long long rows = 0;
  if (!PyArg_ParseTuple(args, "OOOkKiLKii", &cap, &metadata, &source, &version, &stream, &num_slots, &rows, &plan, &active_tokens, &active_slots)) return nullptr;
  State* s = state_of(cap);
  if (!s) return nullptr;
  const Released before(s);
  s->metadata = metadata; s->source = source; s->version = static_cast<uint32_t>(version);
  s->stream = reinterpret_cast<void*>(static_cast<uintptr_t>(stream));
  s->num_slots = num_slots; s->rows = rows; s->active_slots = active_slots < 0 ? 0 : active_slots;
  s->active_tokens = active_tokens < 0 ? 0 : active_tokens;
  s->plan = reinterpret_cast<const void*>(static_cast<uintptr_t>(plan));
  Py_RETURN_NONE;
}

PyObject* py_forget_step(PyObject*, PyObject* cap) {
  State* s = state_of(cap);
  if (!s) return nullptr;
  const Released before(s);
  s->metadata = nullptr; s->source = nullptr; s->rows = -1; s->plan = nullptr;
  Py_RETURN_NONE;
}

// set_scratch(state, device index, stream, address, bytes): the eager scratch buffer of a stream
PyObject* py_set_scratch(PyObject*, PyObject* args) {
  PyObject* cap;
  int device = 0;
  unsigned long long stream = 0, ptr = 0;
  long long bytes = 0;
  if (!PyArg_ParseTuple(args, "OiKKL", &cap, &device, &stream, &ptr, &bytes)) return nullptr;
  State* s = state_of(cap);
  if (!s) return nullptr;
  s->sc_device = device;
  s->sc_stream = reinterpret_cast<void*>(static_cast<uintptr_t>(stream));
  s->sc_ptr = reinterpret_cast<void*>(static_cast<uintptr_t>(ptr));
  s->sc_bytes = bytes;
  Py_RETURN_NONE;
}

// What a Python object has been given under this name (its own attributes alone); nullptr without.  Borrowed.
PyObject* given(PyObject* o, PyObject* name) {
  PyObject** dict = _PyObject_GetDictPtr(o);
  return dict && *dict ? PyDict_GetItem(*dict, name) : nullptr;
}

// The first call of a step: what the Python path looks up for it (HipLoRABackend._plan_for, known_active_slots), where
// the metadata's own slot vector of exactly these rows carries the plan of the launch that made it
// (segment_meta.attach_plan) and has not been rewritten since.  The state holds the three objects from then
// on, until the next step, forget_step or its own end.  Eager calls only.  In Python this lookup cost 15 us of every step on one fast
// host (passes back to back: sixteen calls in fp32 134 us, 119 with this; sixteen linears of 1234 tokens 500, 479); on another host, paced by its
// launches, the difference was within two runs' (172.4, 172.9 and 537, 528).
bool take_step(State* s, const Site& site, PyObject* metadata, PyObject* source_obj, const at::Tensor& source, uint32_t version, void* stream, int64_t rows) {
  static PyObject* const kPlan = PyUnicode_InternFromString("_mlora_plan");
  static PyObject* const kCapacity = PyUnicode_InternFromString("_mlora_capacity");
  static PyObject* const kActiveIds = PyUnicode_InternFromString("active_slot_ids");
  static PyObject* const kActive = PyUnicode_InternFromString("num_active_loras");
  static PyObject* const kSorted = PyUnicode_InternFromString("token_indices_sorted_by_slot");
  if (source.numel() != rows) return false;
  PyObject* made = given(source_obj, kPlan);  // (workspace, max_slots, version)
  if (!made || !PyTuple_Check(made) || PyTuple_GET_SIZE(made) != 3 || !THPVariable_Check(PyTuple_GET_ITEM(made, 0))) return false;
  const at::Tensor& plan = THPVariable_Unpack(PyTuple_GET_ITEM(made, 0));
  const long slots = PyLong_AsLong(PyTuple_GET_ITEM(made, 1));
  const unsigned long at = PyLong_AsUnsignedLong(PyTuple_GET_ITEM(made, 2));
  if (PyErr_Occurred() || slots != site.num_slots || at != version || !on_device(plan, site.device)) return false;
  const Ref plan_held{(Py_INCREF(made), made)};  // (the attribute reads below can run Python code)
  long active = 0;
  const Ref ids{PyObject_GetAttr(metadata, kActiveIds)}, number{PyObject_GetAttr(metadata, kActive)}, sorted{PyObject_GetAttr(metadata, kSorted)};
  PyErr_Clear();
  PyObject* capacity = ids.p ? given(ids.p, kCapacity) : nullptr;
  if (number.p && !(capacity && PyObject_IsTrue(capacity) == 1)) active = PyLong_AsLong(number.p);
  if (PyErr_Occurred()) return false;
  const Released before(s);
  s->held[0] = metadata; s->held[1] = source_obj; s->held[2] = made;
  for (PyObject* o : s->held) Py_INCREF(o);
  s->metadata = metadata; s->source = source_obj; s->version = version; s->stream = stream;
  s->num_slots = site.num_slots; s->rows = rows; s->plan = plan.data_ptr();
  s->active_slots = active > 0 && active <= site.num_slots ? static_cast<int>(active) : 0;
  const int64_t tokens = s->active_slots && sorted.p && THPVariable_Check(sorted.p) ? THPVariable_Unpack(sorted.p).numel() : 0;
  s->active_tokens = tokens <= rows ? static_cast<int>(tokens) : 0;
  return true;
}

// The call itself, at the site of its weight buffers.  Returns 0 (enqueued), a negative code of the library
// (the caller raises with the library's message), or kNotHandled.
long call_at(State* s, const Site& site, PyObject* x_obj, PyObject* target_obj, PyObject* indices, PyObject* metadata, double scaling, PyObject* eff_obj) {
  const at::Tensor& x = THPVariable_Unpack(x_obj);
  const at::Tensor& target = THPVariable_Unpack(target_obj);
  if (x.dim() != 2 || x.stride(1) != 1 || target.dim() != 2 || target.stride(1) != 1) return kNotHandled;
  const int64_t rows = x.size(0);
  if (rows <= 0 || rows > INT32_MAX) return kNotHandled;

  // the flag and the slot vector of the step's metadata (attribute reads: the object is the engine's)
  static PyObject* const kNoLora = PyUnicode_InternFromString("no_lora_flag");
  static PyObject* const kSlots = PyUnicode_InternFromString("token_to_slot");
  PyObject* flag = PyObject_GetAttr(metadata, kNoLora);
  if (!flag) { PyErr_Clear(); return kNotHandled; }
  const int no_lora = PyObject_IsTrue(flag);
  Py_DECREF(flag);
  if (no_lora != 0) { PyErr_Clear(); return kNotHandled; }
  const Ref tts{PyObject_GetAttr(metadata, kSlots)};
  if (!tts.p) { PyErr_Clear(); return kNotHandled; }
  PyObject* source_obj = tts.p != Py_None ? tts.p : indices;
  if (!THPVariable_Check(source_obj)) return kNotHandled;
  const at::Tensor& source = THPVariable_Unpack(source_obj);

  const int dev = site.device;
  if (x.size(1) != site.k || x.scalar_type() != site.dtype || target.scalar_type() != site.dtype || !on_device(x, dev) ||
      !on_device(target, dev) || !on_device(source, dev) || source.numel() < rows || target.size(0) < rows ||
      source.scalar_type() != c10::ScalarType::Int || source.dim() != 1 || !source.is_contiguous())
    return kNotHandled;
  const void* eff_ptr = nullptr;
  if (eff_obj != Py_None) {
    if (!THPVariable_Check(eff_obj)) return kNotHandled;
    const at::Tensor& eff = THPVariable_Unpack(eff_obj);
    if (eff.scalar_type() != c10::ScalarType::Int || !eff.is_contiguous() || eff.numel() < site.num_slots || !on_device(eff, dev)) return kNotHandled;
    eff_ptr = eff.data_ptr();
  }
  if (c10::hip::current_device() != dev) return kNotHandled;  // another GPU of this process: the Python path makes it current
  hipStream_t stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();

  const void* x_ptr = x.data_ptr();
  void* y_ptr = target.data_ptr();
  const int64_t xs = x.stride(0), ys = target.stride(0);
  const void* plan = nullptr;
  void* ws = nullptr;
  int64_t ws_bytes = 0;
  if (site.vectorisable && site.form != MLORA_FORM_TOKEN &&
      !(xs % 8 || ys % 8 || reinterpret_cast<uintptr_t>(x_ptr) % 16 || reinterpret_cast<uintptr_t>(y_ptr) % 16)) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess) { (void)hipGetLastError(); return kNotHandled; }
    if (capturing != hipStreamCaptureStatusNone) return kNotHandled;
    if (source.is_inference()) return kNotHandled;  // no version counter: nothing is remembered for them
    const uint32_t version = source._version();
    const bool known = s->metadata == metadata && s->source == source_obj && s->version == version && s->stream == stream &&
                       s->num_slots == site.num_slots && s->rows == rows && s->plan;
    if (!known && (tts.p == Py_None || !take_step(s, site, metadata, source_obj, source, version, stream, rows))) return kNotHandled;
    plan = s->plan;
    const uint64_t shape = (static_cast<uint64_t>(rows) << 24) | (static_cast<uint64_t>(site.num_slices) << 16) |
                           (static_cast<uint64_t>(site.rank) << 4) | static_cast<uint64_t>(site.dtype_code);
    int64_t need;
    const auto nit = s->need.find(shape);
    if (nit != s->need.end()) {
      need = nit->second;
    } else {
      if (s->need.size() >= 256) s->need.clear();
      need = static_cast<int64_t>(s->workspace_bytes(static_cast<int32_t>(rows), site.num_slices, site.rank, site.dtype_code));
      s->need.emplace(shape, need);
    }
    if (s->sc_device != dev || s->sc_stream != stream || !s->sc_ptr || s->sc_bytes < need) return kNotHandled;
    ws = s->sc_ptr;
    ws_bytes = s->sc_bytes;
  }

  MloraAddArgs* a = site.args;
  a->stream = stream;
  a->x = x_ptr;
  a->y = y_ptr;
  a->x_stride = xs;
  a->y_stride = ys;
  a->token_to_slot = static_cast<const int32_t*>(source.data_ptr());
  a->plan = static_cast<const int32_t*>(plan);
  a->num_tokens = static_cast<int32_t>(rows);
  a->scaling = static_cast<float>(scaling);
  a->workspace = ws;
  a->workspace_bytes = ws_bytes;
  a->effective_rank = static_cast<const int32_t*>(eff_ptr);
  return s->add_lora(a, plan ? s->active_slots : 0, plan ? s->active_tokens : 0);
}

// A call with lists of slices.
long call(State* s, PyObject* y_slices, PyObject* x_obj, PyObject* a_list, PyObject* b_list, PyObject* indices, PyObject* metadata,
          double scaling, PyObject* y_packed, PyObject* eff_obj) {
  if (metadata == Py_None || !THPVariable_Check(x_obj)) return kNotHandled;
  if (!(PyList_Check(y_slices) || PyTuple_Check(y_slices)) || !(PyList_Check(a_list) || PyTuple_Check(a_list)) ||
      !(PyList_Check(b_list) || PyTuple_Check(b_list)))
    return kNotHandled;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(y_slices);
  if (n < 1 || n > MLORA_MAX_SLICES || PySequence_Fast_GET_SIZE(a_list) != n || PySequence_Fast_GET_SIZE(b_list) != n) return kNotHandled;
  PyObject* target_obj = y_packed != Py_None ? y_packed : (n == 1 ? PySequence_Fast_GET_ITEM(y_slices, 0) : nullptr);
  if (!target_obj || !THPVariable_Check(target_obj)) return kNotHandled;

  std::string key;
  const at::Tensor* a0 = nullptr;
  if (!weights_key(a_list, b_list, n, &key, &a0)) return kNotHandled;
  const auto it = s->sites.find(key);
  if (it == s->sites.end()) return kNotHandled;
  const Site& site = it->second;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PySequence_Fast_GET_ITEM(y_slices, i);
    if (!THPVariable_Check(o)) return kNotHandled;
    const at::Tensor& y = THPVariable_Unpack(o);
    if (y.dim() < 1 || y.size(-1) != site.widths[static_cast<size_t>(i)]) return kNotHandled;
  }
  return call_at(s, site, x_obj, target_obj, indices, metadata, scaling, eff_obj);
}

// A call with the buffers of a LoRA linear as the layer holds them: one A buffer [targets, slots, r, K] (or
// [slots, r, K]), its B buffers, and an output whose columns are the targets' blocks in order.  It saves the
// layer the views that the lists are made of.
long call_stacked(State* s, PyObject* target_obj, PyObject* x_obj, PyObject* a_obj, PyObject* b_tuple, PyObject* indices, PyObject* metadata,
                  double scaling, PyObject* eff_obj) {
  if (metadata == Py_None || !THPVariable_Check(x_obj) || !THPVariable_Check(target_obj) || !THPVariable_Check(a_obj) || !PyTuple_Check(b_tuple))
    return kNotHandled;
  const Py_ssize_t n = PyTuple_GET_SIZE(b_tuple);
  const at::Tensor& a = THPVariable_Unpack(a_obj);
  if (n < 1 || n > MLORA_MAX_SLICES || !a.is_contiguous() || (a.dim() == 4 ? a.size(0) != n : a.dim() != 3 || n != 1)) return kNotHandled;
  int64_t buf[2 * MLORA_MAX_SLICES * 4 + 1];
  int at = 0;
  const int64_t one = a.size(-3) * a.size(-2) * a.size(-1) * static_cast<int64_t>(a.element_size());
  for (Py_ssize_t i = 0; i < n; ++i) {
    buf[at++] = reinterpret_cast<int64_t>(a.data_ptr()) + i * one;
    buf[at++] = a.size(-3);
    buf[at++] = a.size(-2);
    buf[at++] = a.size(-1);
  }
  int64_t width = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyTuple_GET_ITEM(b_tuple, i);
    if (!THPVariable_Check(o)) return kNotHandled;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (t.dim() != 3 || !t.is_contiguous()) return kNotHandled;
    buf[at++] = reinterpret_cast<int64_t>(t.data_ptr());
    buf[at++] = t.size(0);
    buf[at++] = t.size(1);
    buf[at++] = t.size(2);
    width += t.size(1);
  }
  buf[at++] = static_cast<int64_t>(a.scalar_type());
  const auto it = s->sites.find(std::string(reinterpret_cast<const char*>(buf), static_cast<size_t>(at) * sizeof(int64_t)));
  if (it == s->sites.end()) return kNotHandled;
  const at::Tensor& target = THPVariable_Unpack(target_obj);
  if (target.dim() != 2 || target.size(1) != width) return kNotHandled;
  return call_at(s, it->second, x_obj, target_obj, indices, metadata, scaling, eff_obj);
}

// call(state, y_slices, x, lora_a_slices, lora_b_slices, indices, metadata, scaling, y_packed, effective_rank)
PyObject* py_call(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 10) {
    PyErr_SetString(PyExc_TypeError, "call() takes ten arguments");
    return nullptr;
  }
  State* s = state_of(args[0]);
  if (!s) return nullptr;
  const double scaling = PyFloat_AsDouble(args[7]);
  if (scaling == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return PyLong_FromLong(kNotHandled); }
  long rc;
  try {
    rc = call(s, args[1], args[2], args[3], args[4], args[5], args[6], scaling, args[8], args[9]);
  } catch (...) {  // whatever a tensor accessor objects to: the Python path says it in its own words
    rc = kNotHandled;
  }
  if (PyErr_Occurred()) PyErr_Clear();
  if (rc == kNotHandled) ++s->passed_on;
  else ++s->handled;
  return PyLong_FromLong(rc);
}

// call_stacked(state, target, x, A, Bs, indices, metadata, scaling, effective_rank)
PyObject* py_call_stacked(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 9) {
    PyErr_SetString(PyExc_TypeError, "call_stacked() takes nine arguments");
    return nullptr;
  }
  State* s = state_of(args[0]);
  if (!s) return nullptr;
  long rc;
  try {
    const double scaling = PyFloat_AsDouble(args[7]);
    rc = PyErr_Occurred() ? kNotHandled : call_stacked(s, args[1], args[2], args[3], args[4], args[5], args[6], scaling, args[8]);
  } catch (...) {
    rc = kNotHandled;
  }
  if (PyErr_Occurred()) PyErr_Clear();
  if (rc == kNotHandled) ++s->passed_on;
  else ++s->handled;
  return PyLong_FromLong(rc);
}

PyObject* py_counters(PyObject*, PyObject* cap) {
  State* s = state_of(cap);
  if (!s) return nullptr;
  return Py_BuildValue("(LL)", s->handled, s->passed_on);
}

// ---- the low-level ops -------------------------------------------------------------------------------
// shrink(address of mlora_shrink, inputs, lora_a weights, output, slot vector, scaling) and
// expand(address of mlora_expand, inputs, lora_b weights, output, slot vector, offset, add): the usual call
// of lora_ops.lora_shrink / lora_expand, checked and enqueued; NOT_HANDLED for anything that
// needs a view, a copy, a conversion or an exception.

// The weights of a call: contiguous [slots, rows, cols] tensors of one element type on `dev`.
bool op_weights(PyObject* list, int dev, c10::ScalarType dtype, Py_ssize_t* n, const at::Tensor* (&w)[MLORA_MAX_SLICES]) {
  if (!(PyList_Check(list) || PyTuple_Check(list))) return false;
  *n = PySequence_Fast_GET_SIZE(list);
  if (*n < 1 || *n > MLORA_MAX_SLICES) return false;
  for (Py_ssize_t i = 0; i < *n; ++i) {
    PyObject* o = PySequence_Fast_GET_ITEM(list, i);
    if (!THPVariable_Check(o)) return false;
    w[i] = &THPVariable_Unpack(o);
    if (w[i]->dim() != 3 || !w[i]->is_contiguous() || w[i]->scalar_type() != dtype || !on_device(*w[i], dev)) return false;
  }
  return true;
}

int code_of(c10::ScalarType t) {
  return t == c10::ScalarType::Float ? MLORA_DTYPE_F32 : t == c10::ScalarType::Half ? MLORA_DTYPE_F16 : t == c10::ScalarType::BFloat16 ? MLORA_DTYPE_BF16 : -1;
}

bool op_slots(const at::Tensor& slots, int64_t rows, int dev) {
  return slots.scalar_type() == c10::ScalarType::Int && slots.dim() == 1 && slots.is_contiguous() && slots.numel() >= rows && on_device(slots, dev);
}

long op_shrink(PyObject* const* args) {
  if (!THPVariable_Check(args[1]) || !THPVariable_Check(args[3]) || !THPVariable_Check(args[4])) return kNotHandled;
  const at::Tensor &x = THPVariable_Unpack(args[1]), &out = THPVariable_Unpack(args[3]), &slots = THPVariable_Unpack(args[4]);
  if (x.dim() != 2 || !x.is_cuda() || x.stride(1) != 1 || x.size(0) < 1 || x.size(0) > INT32_MAX) return kNotHandled;
  const int dev = x.device().index();
  const at::Tensor* w[MLORA_MAX_SLICES];
  Py_ssize_t n;
  if (!op_weights(args[2], dev, x.scalar_type(), &n, w) || !op_slots(slots, x.size(0), dev)) return kNotHandled;
  for (Py_ssize_t i = 1; i < n; ++i)
    if (w[i]->sizes() != w[0]->sizes()) return kNotHandled;
  const int dtype = code_of(x.scalar_type()), out_dtype = code_of(out.scalar_type());
  if (dtype < 0 || out_dtype < 0 || w[0]->size(2) != x.size(1) || out.dim() != 3 || !out.is_contiguous() || !on_device(out, dev) || out.size(0) != n ||
      out.size(1) != x.size(0) || out.size(2) != w[0]->size(1) || c10::hip::current_device() != dev)
    return kNotHandled;
  MloraShrinkArgs a = {};
  a.scaling = static_cast<float>(PyFloat_AsDouble(args[5]));
  if (PyErr_Occurred()) return kNotHandled;
  a.stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
  a.x = x.data_ptr(); a.out = out.data_ptr(); a.x_stride = x.stride(0);
  a.token_to_slot = static_cast<const int32_t*>(slots.data_ptr());
  a.num_tokens = static_cast<int32_t>(x.size(0)); a.k = static_cast<int32_t>(x.size(1));
  a.r = static_cast<int32_t>(w[0]->size(1)); a.num_slots = static_cast<int32_t>(w[0]->size(0)); a.num_slices = static_cast<int32_t>(n);
  a.dtype = dtype; a.out_dtype = out_dtype;
  for (Py_ssize_t i = 0; i < n; ++i) a.a[i] = w[i]->data_ptr();
  const auto fn = reinterpret_cast<int (*)(const MloraShrinkArgs*)>(PyLong_AsSize_t(args[0]));
  return PyErr_Occurred() ? kNotHandled : fn(&a);
}

long op_expand(PyObject* const* args) {
  if (!THPVariable_Check(args[1]) || !THPVariable_Check(args[3]) || !THPVariable_Check(args[4])) return kNotHandled;
  const at::Tensor &h = THPVariable_Unpack(args[1]), &y = THPVariable_Unpack(args[3]), &slots = THPVariable_Unpack(args[4]);
  if (h.dim() != 3 || !h.is_cuda() || !h.is_contiguous() || h.size(1) < 1 || h.size(1) > INT32_MAX) return kNotHandled;
  const int dev = h.device().index();
  const at::Tensor* w[MLORA_MAX_SLICES];
  Py_ssize_t n;
  if (!op_weights(args[2], dev, y.scalar_type(), &n, w) || n != h.size(0) || !op_slots(slots, h.size(1), dev)) return kNotHandled;
  const int dtype = code_of(y.scalar_type()), h_dtype = code_of(h.scalar_type());
  if (dtype < 0 || h_dtype < 0 || y.dim() != 2 || y.stride(1) != 1 || y.size(0) < h.size(1) || !on_device(y, dev) || c10::hip::current_device() != dev)
    return kNotHandled;
  MloraExpandArgs a = {};
  a.offset_start = static_cast<int32_t>(PyLong_AsLong(args[5]));
  a.add_inputs = PyObject_IsTrue(args[6]) == 1;
  if (PyErr_Occurred() || a.offset_start < 0) return kNotHandled;
  int64_t width = a.offset_start;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (w[i]->size(2) != h.size(2) || w[i]->size(0) != w[0]->size(0)) return kNotHandled;
    a.b[i] = w[i]->data_ptr();
    a.n[i] = static_cast<int32_t>(w[i]->size(1));
    width += w[i]->size(1);
  }
  if (width > y.size(1)) return kNotHandled;
  a.stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
  a.h = h.data_ptr(); a.y = y.data_ptr(); a.y_stride = y.stride(0);
  a.token_to_slot = static_cast<const int32_t*>(slots.data_ptr());
  a.num_tokens = static_cast<int32_t>(h.size(1)); a.r = static_cast<int32_t>(h.size(2));
  a.num_slots = static_cast<int32_t>(w[0]->size(0)); a.num_slices = static_cast<int32_t>(n);
  a.dtype = dtype; a.h_dtype = h_dtype;
  const auto fn = reinterpret_cast<int (*)(const MloraExpandArgs*)>(PyLong_AsSize_t(args[0]));
  return PyErr_Occurred() ? kNotHandled : fn(&a);
}

template <typename F> PyObject* run_op(F f, PyObject* const* args, Py_ssize_t nargs, Py_ssize_t want) {
  if (nargs != want) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments", want);
    return nullptr;
  }
  long rc;
  try {
    rc = f(args);
  } catch (...) {
    rc = kNotHandled;
  }
  if (PyErr_Occurred()) PyErr_Clear();
  return PyLong_FromLong(rc);
}
PyObject* py_shrink(PyObject*, PyObject* const* args, Py_ssize_t nargs) { return run_op(op_shrink, args, nargs, 6); }
PyObject* py_expand(PyObject*, PyObject* const* args, Py_ssize_t nargs) { return run_op(op_expand, args, nargs, 7); }

// ---- batch contexts --------------------------------------------------------------------------------------
// The runs of a batch (slot ids and token counts as Python lists) as arrays.
bool read_runs(PyObject* slots, PyObject* counts, std::vector<int32_t>* s, std::vector<int32_t>* c) {
  if (!PyList_Check(slots) || !PyList_Check(counts) || PyList_GET_SIZE(slots) != PyList_GET_SIZE(counts)) return false;
  const Py_ssize_t n = PyList_GET_SIZE(slots);
  if (n > MLORA_META_SINGLES) return false;
  s->resize(static_cast<size_t>(n));
  c->resize(static_cast<size_t>(n));
  for (Py_ssize_t i = 0; i < n; ++i) {
    const long a = PyLong_AsLong(PyList_GET_ITEM(slots, i)), b = PyLong_AsLong(PyList_GET_ITEM(counts, i));
    if ((a == -1 || b == -1) && PyErr_Occurred()) return false;
    if (b < 0 || b > INT32_MAX || a < INT32_MIN || a > INT32_MAX) return false;
    (*s)[static_cast<size_t>(i)] = static_cast<int32_t>(a);
    (*c)[static_cast<size_t>(i)] = static_cast<int32_t>(b);
  }
  return true;
}

// run_totals(slots, counts) -> (tokens, tokens with a slot, slots with tokens, largest slot with tokens), or None for
// what the Python path has to see to
PyObject* py_run_totals(PyObject*, PyObject* args) {
  PyObject *slots, *counts;
  if (!PyArg_ParseTuple(args, "OO", &slots, &counts)) return nullptr;
  std::vector<int32_t> s, c;
  if (!read_runs(slots, counts, &s, &c)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  long long tokens = 0, with_slot = 0;
  int active = 0, largest = -1;
  bool seen[MLORA_MAX_SLOTS] = {}, singles = true;
  for (size_t i = 0; i < s.size(); ++i) {
    tokens += c[i];
    singles &= c[i] == 1;
    if (s[i] < 0 || c[i] == 0) continue;
    if (s[i] >= MLORA_MAX_SLOTS) Py_RETURN_NONE;
    with_slot += c[i];
    if (!seen[s[i]]) { seen[s[i]] = true; ++active; }
    if (s[i] > largest) largest = s[i];
  }
  if (tokens > INT32_MAX || (!singles && s.size() > MLORA_META_RUNS)) Py_RETURN_NONE;
  return Py_BuildValue("LLii", tokens, with_slot, active, largest);
}

// build_context(address of mlora_meta_build_runs, slots, counts, device index, max_slots, capacity, addresses of slot vector, sorted
// indices, ids, counts, offsets and plan) -> 0 or a library error code: slot vector, index arrays and plan in one launch on
// the current stream
PyObject* py_build_context(PyObject*, PyObject* args) {
  PyObject *slots, *counts;
  unsigned long long fn, tts, sorted, ids, per_slot, offsets, plan;
  int device, max_slots, capacity;
  if (!PyArg_ParseTuple(args, "KOOiiiKKKKKK", &fn, &slots, &counts, &device, &max_slots, &capacity, &tts, &sorted, &ids, &per_slot, &offsets, &plan))
    return nullptr;
  std::vector<int32_t> s, c;
  if (!read_runs(slots, counts, &s, &c)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "runs of a batch: two lists of equal length");
    return nullptr;
  }
  int64_t tokens = 0;
  for (const int32_t n : c) tokens += n;
  MloraMetaArgs a[2] = {};
  auto at = [](unsigned long long address) { return reinterpret_cast<int32_t*>(static_cast<uintptr_t>(address)); };
  a[0].stream = a[1].stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream();
  a[0].num_tokens = a[1].num_tokens = static_cast<int32_t>(tokens);
  a[0].max_slots = a[1].max_slots = max_slots;
  a[0].padded_token_to_slot = at(tts);
  a[0].padded_len = static_cast<int32_t>(tokens);
  a[0].sorted_idx = at(sorted);
  a[0].compact_ids = at(ids); a[0].compact_counts = at(per_slot); a[0].compact_offsets = at(offsets);
  a[0].compact_capacity = capacity;
  a[1].plan = at(plan);
  return PyLong_FromLong(reinterpret_cast<int (*)(const MloraMetaArgs*, int32_t, const int32_t*, const int32_t*, int32_t)>(static_cast<uintptr_t>(fn))(
      a, 2, s.data(), c.data(), static_cast<int32_t>(s.size())));
}

// ---- slot installs -----------------------------------------------------------------------------------
// An adapter's targets, collected module by module and handed to mlora_install_slots together.
struct InstallBatch {
  std::vector<MloraInstallArgs> args;
  std::vector<MloraInstallState> states;
  int device = -1;
};
const char* kInstallCapsule = "mlora.fastcall.installs";
void destroy_installs(PyObject* capsule) { delete static_cast<InstallBatch*>(PyCapsule_GetPointer(capsule, kInstallCapsule)); }

PyObject* py_install_batch(PyObject*, PyObject*) { return PyCapsule_New(new InstallBatch(), kInstallCapsule, destroy_installs); }

// Address of a payload tensor on `dev`: its own, or that of its copy where it lies in the packed host buffer.
const void* source_on(const at::Tensor& t, int dev, const at::Tensor* packed, const at::Tensor* staged) {
  if (t.is_cuda()) return t.device().index() == dev ? t.data_ptr() : nullptr;
  if (!packed || !staged || !t.is_cpu() || t.scalar_type() != packed->scalar_type() || !t.is_contiguous()) return nullptr;
  const char* at = static_cast<const char*>(t.data_ptr());
  const char* base = static_cast<const char*>(packed->data_ptr());
  if (at < base || at + t.numel() * t.element_size() > base + packed->numel() * packed->element_size()) return nullptr;
  return static_cast<const char*>(staged->data_ptr()) + (at - base);
}

// install_add(batch, A buffer, tuple of B buffers, lora_a, lora_b, slot, rank, scaling, packed, its device copy,
// rank vector, scaling vector, second scaling vector) -> bool: everything set_slot_lora and the payload check of the
// layer look at is in order and the module's targets are in the batch; False: nothing was added and the
// layer's own methods say what is wrong, or do it.
bool install_add(InstallBatch* batch, PyObject* const* args) {
  if (!THPVariable_Check(args[1]) || !PyTuple_Check(args[2]) || !THPVariable_Check(args[3])) return false;
  const at::Tensor &A = THPVariable_Unpack(args[1]), &a_src = THPVariable_Unpack(args[3]);
  if (!A.is_cuda() || !A.is_contiguous()) return false;
  const bool multi = A.dim() == 4;
  if (!multi && A.dim() != 3) return false;
  const Py_ssize_t n = PyTuple_GET_SIZE(args[2]);
  const int64_t slots = A.size(-3), r = A.size(-2), k = A.size(-1);
  if (n < 1 || (multi ? A.size(0) != n : n != 1)) return false;
  if (multi ? !PyList_Check(args[4]) || PyList_GET_SIZE(args[4]) != n : !THPVariable_Check(args[4])) return false;
  const long long slot = PyLong_AsLongLong(args[5]), rank = PyLong_AsLongLong(args[6]);
  const double scaling = PyFloat_AsDouble(args[7]);
  if (PyErr_Occurred() || slot < 0 || slot >= slots || rank < 1 || rank > r || !std::isfinite(scaling)) return false;
  const at::Tensor* packed = THPVariable_Check(args[8]) ? &THPVariable_Unpack(args[8]) : nullptr;
  const at::Tensor* staged = THPVariable_Check(args[9]) ? &THPVariable_Unpack(args[9]) : nullptr;
  const int dev = A.device().index();
  if (dev != c10::hip::current_device() || (batch->device >= 0 && batch->device != dev)) return false;
  if (staged && (!on_device(*staged, dev) || staged->numel() != packed->numel() || staged->scalar_type() != packed->scalar_type())) return false;
  if (a_src.dim() != (multi ? 3 : 2) || (multi && a_src.size(0) != n) || a_src.size(-2) < rank || a_src.size(-1) != k || a_src.stride(-1) != 1) return false;
  const int dtype = code_of(A.scalar_type()), src_dtype = code_of(a_src.scalar_type());
  if (dtype < 0 || src_dtype < 0) return false;
  const void* a_base = source_on(a_src, dev, packed, staged);
  if (!a_base) return false;
  MloraInstallState state = {};
  for (int i = 10; i < 13; ++i) {
    if (!THPVariable_Check(args[i])) return false;
    const at::Tensor& t = THPVariable_Unpack(args[i]);
    if (!on_device(t, dev) || t.dim() != 1 || t.size(0) != slots || !t.is_contiguous()) return false;
    if (i == 10) {
      if (t.scalar_type() != c10::ScalarType::Int) return false;
      state.rank = static_cast<int32_t*>(t.data_ptr());
    } else {
      const int code = code_of(t.scalar_type());
      if (code < 0 || (i == 12 && code != state.dtype)) return false;
      state.dtype = code;
      state.scaling[i - 11] = t.data_ptr();
    }
  }
  const size_t before = batch->args.size();
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* bo = PyTuple_GET_ITEM(args[2], i);
    PyObject* so = multi ? PyList_GET_ITEM(args[4], i) : args[4];
    bool ok = THPVariable_Check(bo) && THPVariable_Check(so);
    if (ok) {
      const at::Tensor &B = THPVariable_Unpack(bo), &b_src = THPVariable_Unpack(so);
      const void* b_base = source_on(b_src, dev, packed, staged);
      ok = b_base && B.dim() == 3 && B.is_contiguous() && on_device(B, dev) && B.scalar_type() == A.scalar_type() && B.size(0) == slots &&
           B.size(2) == r && b_src.dim() == 2 && b_src.scalar_type() == a_src.scalar_type() && b_src.size(0) == B.size(1) &&
           b_src.size(1) >= rank && b_src.stride(1) == 1;
      if (ok) {
        MloraInstallArgs m = {};
        m.a_dst = static_cast<char*>(A.data_ptr()) + i * slots * r * k * static_cast<int64_t>(A.element_size());
        m.b_dst = B.data_ptr();
        m.a_src = static_cast<const char*>(a_base) + (multi ? i * a_src.stride(0) * static_cast<int64_t>(a_src.element_size()) : 0);
        m.b_src = b_base;
        m.a_src_stride = a_src.stride(-2); m.b_src_stride = b_src.stride(0);
        m.slot = static_cast<int32_t>(slot); m.k = static_cast<int32_t>(k); m.n = static_cast<int32_t>(B.size(1)); m.r = static_cast<int32_t>(r);
        m.rank = static_cast<int32_t>(rank); m.dtype = dtype; m.src_dtype = src_dtype; m.scaling = static_cast<float>(scaling);
        m.num_slots = static_cast<int32_t>(slots);
        ok = m.a_src_stride >= k && m.b_src_stride >= rank;
        if (ok) {
          batch->args.push_back(m);
          batch->states.push_back(i == 0 ? state : MloraInstallState{});
        }
      }
    }
    if (!ok) {
      batch->args.resize(before);
      batch->states.resize(before);
      return false;
    }
  }
  batch->device = dev;
  return true;
}

PyObject* py_install_add(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 13) {
    PyErr_SetString(PyExc_TypeError, "install_add() takes thirteen arguments");
    return nullptr;
  }
  auto* batch = static_cast<InstallBatch*>(PyCapsule_GetPointer(args[0], kInstallCapsule));
  if (!batch) return nullptr;
  bool ok;
  try {
    ok = install_add(batch, args);
  } catch (...) {
    ok = false;
  }
  if (PyErr_Occurred()) PyErr_Clear();
  return PyBool_FromLong(ok);
}

// install_flush(batch, address of mlora_install_slots) -> 0 or a library error code; the batch is empty then
PyObject* py_install_flush(PyObject*, PyObject* args) {
  PyObject* cap;
  unsigned long long fn = 0;
  if (!PyArg_ParseTuple(args, "OK", &cap, &fn)) return nullptr;
  auto* batch = static_cast<InstallBatch*>(PyCapsule_GetPointer(cap, kInstallCapsule));
  if (!batch) return nullptr;
  long rc = 0;
  if (!batch->args.empty()) {
    void* stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(batch->device)).stream();
    for (auto& m : batch->args) m.stream = stream;
    rc = reinterpret_cast<int (*)(const MloraInstallArgs*, const MloraInstallState*, int32_t)>(static_cast<uintptr_t>(fn))(
        batch->args.data(), batch->states.data(), static_cast<int32_t>(batch->args.size()));
  }
  batch->args.clear();
  batch->states.clear();
  return PyLong_FromLong(rc);
}

template <typename F> PyCFunction method(F* f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef kMethods[] = {
    {"call_stacked", method(py_call_stacked), METH_FASTCALL,
     "call_stacked(state, target, x, A, Bs, indices, metadata, scaling, effective_rank) -> 0, a library error code, or NOT_HANDLED"},
    {"shrink", method(py_shrink), METH_FASTCALL, "shrink(address of mlora_shrink, inputs, weights, output, slots, scaling) -> 0, a library error code, or NOT_HANDLED"},
    {"expand", method(py_expand), METH_FASTCALL, "expand(address of mlora_expand, inputs, weights, output, slots, offset, add) -> 0, a library error code, or NOT_HANDLED"},
    {"run_totals", py_run_totals, METH_VARARGS, "run_totals(slots, counts) -> (tokens, with a slot, active slots, largest slot) or None"},
    {"build_context", py_build_context, METH_VARARGS, "build_context(address of mlora_meta_build_runs, slots, counts, device, max_slots, capacity, six addresses) -> rc"},
    {"install_batch", py_install_batch, METH_NOARGS, "install_batch() -> an empty batch of slot installs"},
    {"install_add", method(py_install_add), METH_FASTCALL, "install_add(batch, A, Bs, lora_a, lora_b, slot, rank, scaling, packed, staged, ranks, scalings, base scalings) -> bool"},
    {"install_flush", py_install_flush, METH_VARARGS, "install_flush(batch, address of mlora_install_slots) -> 0 or a library error code"},
    {"create", py_create, METH_VARARGS, "create(address of mlora_add_lora_counts, address of mlora_add_workspace_bytes) -> state"},
    {"register_site", py_register_site, METH_VARARGS, "register_site(state, a_list, b_list, widths, block address, block owner, vectorisable) -> bool"},
    {"clear_sites", py_clear_sites, METH_O, "clear_sites(state)"},
    {"set_step", py_set_step, METH_VARARGS, "set_step(state, metadata, source, version, stream, num_slots, rows, plan address, tokens with a slot, active slots)"},
    {"forget_step", py_forget_step, METH_O, "forget_step(state)"},
    {"set_scratch", py_set_scratch, METH_VARARGS, "set_scratch(state, device index, stream, address, bytes)"},
    {"counters", py_counters, METH_O, "counters(state) -> (calls enqueued here, calls left to the Python path)"},
    {"call", method(py_call), METH_FASTCALL,
     "call(state, y_slices, x, lora_a_slices, lora_b_slices, indices, metadata, scaling, y_packed, effective_rank) -> 0, a library error code, or NOT_HANDLED"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mlora_fastcall", "C++ host path of the usual add_lora call", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mlora_fastcall(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m) PyModule_AddIntConstant(m, "NOT_HANDLED", kNotHandled);
  return m;
}
