// Native call path of the Python API: argument checks, allocation and the C-ABI call of an ordinary
// call in one step.
//
// A call of the package is a handful of tensors and numbers.  Checked attribute by attribute in Python
// and passed through ctypes (25 + 45 arguments for one attention call), its host side took 15 us per
// GEMM and 39 us per attention call, more than the GPU needs for a small one (attention over 384 tokens
// of two heads: 28 us of kernels).  Here the same checks read the tensors' C++ fields.
//
// Every function returns None when a call is not an ordinary one (another device than the current one, a
// tensor that has to be converted first, a wrong shape or type): the Python code then goes through its
// own checks, converts or raises, so that errors have one source and this file none.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <thread>
#include <vector>

#include "../../include/flashomni_hip.h"

namespace {

using at::Tensor;

// None or a tensor
bool opt_tensor(PyObject* o, const Tensor** t) {
  if (o == Py_None) {
    *t = nullptr;
    return true;
  }
  if (!THPVariable_Check(o)) return false;
  *t = &THPVariable_Unpack(o);
  return true;
}

bool whole(PyObject* o, int64_t* v) {
  if (!PyLong_Check(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool real(PyObject* o, double* v) {
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  *v = PyFloat_AsDouble(o);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool truth(PyObject* o) { return PyObject_IsTrue(o) == 1; }

void* data(const Tensor* t) { return t ? t->data_ptr() : nullptr; }

bool on(const Tensor& t, int dev) { return t.is_cuda() && t.get_device() == dev; }

// a contiguous tensor of the given type on the device
bool flat(const Tensor& t, at::ScalarType type, int dev) {
  return on(t, dev) && t.scalar_type() == type && t.is_contiguous();
}

int act_code(at::ScalarType t) { return t == at::kBFloat16 ? FO_BF16 : t == at::kHalf ? FO_F16 : -1; }

void* stream_of(int dev) { return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream(); }

Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType type, int dev) {
  return at::empty(sizes, at::TensorOptions().dtype(type).device(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(dev))));
}

PyObject* raise_last() {
  PyErr_SetString(PyExc_RuntimeError, fo_last_error());
  return nullptr;
}

#define FALL_BACK_UNLESS(cond) \
  do {                         \
    if (!(cond)) Py_RETURN_NONE; \
  } while (0)

#define TORCH_GUARD_BEGIN try {
#define TORCH_GUARD_END                              \
  }                                                  \
  catch (const std::exception& e) {                  \
    PyErr_SetString(PyExc_RuntimeError, e.what());   \
    return nullptr;                                  \
  }

// x [B, M, K] and w [N, K] of a GEMM: contiguous, one 16-bit type, on the current device
bool gemm_operands(const Tensor& a, const Tensor& b, int* dev, int* code) {
  if (!a.is_cuda() || a.dim() != 3 || b.dim() != 2) return false;
  *dev = a.get_device();
  *code = act_code(a.scalar_type());
  return *code >= 0 && *dev == c10::hip::current_device() && a.is_contiguous() && flat(b, a.scalar_type(), *dev) &&
         a.size(2) == b.size(1) && a.size(0) > 0 && a.size(1) > 0 && a.size(0) < (1 << 30) && a.size(1) < (1 << 30) &&
         b.size(0) < (1 << 30) && a.size(2) < (1 << 30);
}

bool gemm_symbols(const Tensor* info, const Tensor* indptr, int dev, int64_t batch, int64_t m, int64_t heads,
                  int64_t text, int64_t q_size) {
  if (!info || !indptr || !flat(*info, at::kByte, dev) || !flat(*indptr, at::kInt, dev)) return false;
  const int64_t last = (text + m - 1) / q_size;
  return indptr->numel() == batch + 1 && info->numel() >= ((last + 1) * heads + 7) / 8;
}

// scratch of the long launches: the pool that the Python side keeps per device and stream
PyObject* g_gemm_scratch = nullptr;  // callable (device index, stream, bytes) -> tensor

PyObject* set_gemm_scratch(PyObject*, PyObject* fn) {
  Py_INCREF(fn);
  Py_XDECREF(g_gemm_scratch);
  g_gemm_scratch = fn;
  Py_RETURN_NONE;
}

bool gemm_scratch(int dev, void* stream, int64_t bytes, Tensor* out) {
  PyObject* r = PyObject_CallFunction(g_gemm_scratch, "iKL", dev, static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(stream)),
                                      static_cast<long long>(bytes));
  if (!r) return false;
  *out = THPVariable_Unpack(r);
  Py_DECREF(r);
  return true;
}

// (A, B, num_qo_heads, sparse_info, sparse_info_indptr, num_text_tokens, bias, out, sparse_q_size, is_full)
PyObject* gemm_q(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor *a, *b, *info, *indptr, *bias, *out;
  int64_t heads, text, q_size;
  FALL_BACK_UNLESS(n == 10 && opt_tensor(args[0], &a) && a && opt_tensor(args[1], &b) && b && whole(args[2], &heads) &&
                   opt_tensor(args[3], &info) && opt_tensor(args[4], &indptr) && whole(args[5], &text) &&
                   opt_tensor(args[6], &bias) && opt_tensor(args[7], &out) && whole(args[8], &q_size));
  const bool full = truth(args[9]);
  int dev, code;
  FALL_BACK_UNLESS(gemm_operands(*a, *b, &dev, &code));
  const int64_t batch = a->size(0), m = a->size(1), k = a->size(2), cols = b->size(0);
  FALL_BACK_UNLESS(heads > 0 && heads < (1 << 20) && cols % heads == 0 && text >= 0 && text < (1 << 30) && q_size > 0 &&
                   q_size < (1 << 30));
  FALL_BACK_UNLESS(full || gemm_symbols(info, indptr, dev, batch, m, heads, text, q_size));
  FALL_BACK_UNLESS(!bias || (flat(*bias, a->scalar_type(), dev) && bias->numel() == cols));
  FALL_BACK_UNLESS(!out || (flat(*out, a->scalar_type(), dev) && out->dim() == 3 && out->size(0) == batch &&
                            out->size(1) == m && out->size(2) == cols));
  Tensor fresh, scratch;
  if (!out) fresh = new_tensor({batch, m, cols}, a->scalar_type(), dev);
  const Tensor& y = out ? *out : fresh;
  void* stream = stream_of(dev);
  const int64_t need = full ? 0 : fo_gemm_workspace_bytes(batch, m, cols);
  if (need && !gemm_scratch(dev, stream, need, &scratch)) return nullptr;
  if (fo_gemm_q(a->data_ptr(), b->data_ptr(), data(bias), y.data_ptr(), code, batch, m, cols, k, q_size, heads,
                full ? nullptr : static_cast<const uint8_t*>(data(info)),
                full ? nullptr : static_cast<const int32_t*>(data(indptr)), text, full, need ? scratch.data_ptr() : nullptr,
                need, stream))
    return raise_last();
  if (out) {
    Py_INCREF(args[7]);
    return args[7];
  }
  return THPVariable_Wrap(std::move(fresh));
  TORCH_GUARD_END
}

// (A, B, num_qo_heads, sparse_info, sparse_info_indptr, num_text_tokens, bias, is_for_cache, sparse_q_size,
//  fp32 output)
PyObject* gemm_o(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor *a, *b, *info, *indptr, *bias;
  int64_t heads, text, q_size;
  FALL_BACK_UNLESS(n == 10 && opt_tensor(args[0], &a) && a && opt_tensor(args[1], &b) && b && whole(args[2], &heads) &&
                   opt_tensor(args[3], &info) && opt_tensor(args[4], &indptr) && whole(args[5], &text) &&
                   opt_tensor(args[6], &bias) && whole(args[8], &q_size));
  const bool cache = truth(args[7]), f32 = truth(args[9]);
  int dev, code;
  FALL_BACK_UNLESS(gemm_operands(*a, *b, &dev, &code));
  const int64_t batch = a->size(0), m = a->size(1), k = a->size(2), cols = b->size(0);
  FALL_BACK_UNLESS(heads > 0 && heads < (1 << 20) && text >= 0 && text < (1 << 30) && q_size > 0 && q_size < (1 << 30) &&
                   cols % heads == 0 && gemm_symbols(info, indptr, dev, batch, m, heads, text, q_size));
  int kind = FO_BIAS_NONE, bias_code = code;
  if (bias && cache) {
    FALL_BACK_UNLESS(flat(*bias, a->scalar_type(), dev) && bias->numel() == cols);
    kind = FO_BIAS_VECTOR;
  } else if (bias) {
    FALL_BACK_UNLESS(on(*bias, dev) && bias->is_contiguous() && bias->numel() == batch * m * cols &&
                     (bias->scalar_type() == a->scalar_type() || bias->scalar_type() == at::kFloat));
    kind = FO_BIAS_MATRIX;
    if (bias->scalar_type() == at::kFloat) bias_code = FO_F32;
  }
  Tensor y = new_tensor({batch, m, cols}, f32 ? at::kFloat : a->scalar_type(), dev);
  if (fo_gemm_o(a->data_ptr(), b->data_ptr(), data(bias), y.data_ptr(), code, kind, bias_code, f32 ? FO_F32 : code, batch,
                m, cols, k, q_size, heads, static_cast<const uint8_t*>(data(info)),
                static_cast<const int32_t*>(data(indptr)), text, cache, nullptr, 0, stream_of(dev)))
    return raise_last();
  return THPVariable_Wrap(std::move(y));
  TORCH_GUARD_END
}

// ---- attention -----------------------------------------------------------------------------------
// A word of pinned memory that a plan's launch leaves its ticket in (not on the default stream, see Plan).
// Tickets ascend and a word is handed out again only when its ticket is there, so that a word and a ticket stay
// comparable after that.  There are as many as plans have ever been alive or under way at a time, in pages of
// 512 (guarded by the interpreter's lock).
struct Word {
  uint64_t* at;
  uint32_t ticket;
  bool arrived() const {  // (false without a word)
    return at && static_cast<int32_t>(static_cast<uint32_t>(__atomic_load_n(at, __ATOMIC_ACQUIRE) >> 32) - ticket) >= 0;
  }
};
std::vector<uint64_t*> g_free_words;
std::vector<Word> g_words_under_way;  // of plans that are gone
uint32_t g_plan_ticket = 0;

bool take_word(Word* w) {
  if (g_free_words.empty()) {
    auto& v = g_words_under_way;
    auto there = std::partition(v.begin(), v.end(), [](const Word& u) { return !u.arrived(); });
    for (auto i = there; i != v.end(); ++i) g_free_words.push_back(i->at);
    v.erase(there, v.end());
  }
  if (g_free_words.empty()) {
    c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);  // (another thread may be capturing)
    void* page = nullptr;
    if (hipHostMalloc(&page, 4096, hipHostMallocCoherent) != hipSuccess) return false;
    for (int i = 0; i < 512; ++i) g_free_words.push_back(static_cast<uint64_t*>(page) + i);
  }
  w->at = g_free_words.back();
  g_free_words.pop_back();
  w->ticket = ++g_plan_ticket;
  __atomic_store_n(w->at, static_cast<uint64_t>(w->ticket - 1) << 32, __ATOMIC_RELEASE);
  return true;
}

// no launch will write it
void settle_word(const Word& w) {
  if (w.at) __atomic_store_n(w.at, static_cast<uint64_t>(w.ticket) << 32, __ATOMIC_RELEASE);
}

void give_word(const Word& w) {
  if (!w.at) return;
  if (w.arrived()) g_free_words.push_back(w.at);
  else g_words_under_way.push_back(w);
}

// The host waits for a word, other threads go on.  (A device that is lost ends the process; the limit is for one
// that hangs.)
bool wait_word(const Word& w) {
  if (w.arrived()) return true;
  bool ok = false;
  Py_BEGIN_ALLOW_THREADS
  const auto limit = std::chrono::steady_clock::now() + std::chrono::minutes(10);
  while (!(ok = w.arrived()) && std::chrono::steady_clock::now() < limit)
    std::this_thread::sleep_for(std::chrono::microseconds(20));
  Py_END_ALLOW_THREADS
  return ok;
}

// kv tokens of a request whose rows the kernel without a decoded list can hold (4096 blocks; the decoder takes
// longer requests)
constexpr int64_t kMaxListed = 4096 * 128;

hipError_t host_wait(hipEvent_t event) {
  hipError_t e;
  Py_BEGIN_ALLOW_THREADS
  e = hipEventSynchronize(event);
  Py_END_ALLOW_THREADS
  return e;
}

// What plan() derives from a batch: sizes, and one int32 tensor on the device that holds every table
// (see fo_plan_tables).
struct Plan {
  PyObject_HEAD
  Tensor tables;
  // plan() queues the tables on the stream that is current there, `home`, and does not wait.  Another stream
  // waits for `behind`, an event recorded on `home` when one first asks.  A stream that is being captured by then
  // takes no such event; the host can still see `word`, which the launch writes.  The default stream cannot be
  // captured and needs no word (0.5 us of a batch of four requests planned anew for each call, 33.5 us; an event
  // recorded in advance 3.3 us).  `used`: the other streams that the allocator holds `tables` for.
  hipStream_t home;
  hipEvent_t behind;
  Word word;
  bool complete;
  std::vector<hipStream_t> used;
  const int32_t *qo_indptr, *kv_indptr;  // the tables' own, or the caller's (graph mode)
  Tensor qo_keep, kv_keep;
  int dev, batch, num_qo, num_kv, symbol_heads, packed;
  bool from_zero;  // the first request begins at token 0
  // What the last run (not: recorded in a graph) left behind.  state 0: the list that the Python side decoded; 1:
  // rows taken straight from the symbols, of which a copy is kept; 2: every row (is_full).  stream: where it ran.
  int state;
  long long stream;
  // Launches of the plan's that a graph holds run at times the host does not know: once there are any
  // (`captured`), whether the list or the kept symbols are newer is read on the device (sched[33]).
  // listed_in: the capture whose last launch on this plan was a decode; recorded_in, recorded_full: the last
  // capture that recorded a decode or run, and its is_full.
  // recording: the last launch was recorded.
  // taken: rows have been taken straight from the symbols, or a graph holds a launch that does so.  Until then
  // there is nothing that could be newer than the list.
  // list_only: a graph holds a reuse that runs the list without looking for something newer, so that no run of the plan
  // takes its rows from the symbols from then on.
  int captured, recorded_full, recording, taken, list_only;
  unsigned long long listed_in, recorded_in;
  // The copy lies behind the tables, in one place for as long as the plan lives (a graph writes it at every
  // replay): room for the symbols that such a run takes, at keep_at[0] info, [1] kv_info, [2] the indptrs (bytes
  // from the start of the tables; keep_at[0] = 0: a batch that is always decoded).
  int64_t keep_at[3], keep_room[2];
  // Partial results of the longer lists that are taken from the symbols, which leave the float workspace to others: made when first
  // needed (66 MiB on 256 CUs).  no_parts: the allocator has refused it, and such runs are decoded from then on.
  Tensor parts;
  bool no_parts;
  fo_batch_sizes z;
};

PyTypeObject* g_plan_type = nullptr;

void plan_dealloc(PyObject* self) {
  Plan* p = reinterpret_cast<Plan*>(self);
  if (p->behind) (void)hipEventDestroy(p->behind);
  give_word(p->word);
  p->used.~vector();
  p->tables.~Tensor();
  p->qo_keep.~Tensor();
  p->kv_keep.~Tensor();
  p->parts.~Tensor();
  PyTypeObject* t = Py_TYPE(self);
  t->tp_free(self);
  Py_DECREF(t);
}

// (the default stream cannot be captured)
bool capturing(hipStream_t stream) {
  if (!stream) return false;
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(stream, &s) == hipSuccess && s != hipStreamCaptureStatusNone;
}

// the capture that the stream is in, 0: none
unsigned long long capture_of(hipStream_t stream) {
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (!stream || hipStreamGetCaptureInfo(stream, &s, &id) != hipSuccess || s == hipStreamCaptureStatusNone) return 0;
  return id ? id : ~0ull;
}

// Whether a run of the plan with 16-bit operands may be taken straight from the symbols.
bool may_take(const Plan* p, int64_t ws_bytes, double cap) {
  return fo_sparse_attention_direct_may_serve(static_cast<int32_t>(p->z.n_q_blocks), p->symbol_heads, p->batch, p->z.max_nnz,
                                              ws_bytes, static_cast<float>(cap));
}

// A launch that leaves a list (state 0) or takes rows without one (1, 2) has been queued on the stream.
void note(Plan* p, hipStream_t stream, int state, bool full) {
  const unsigned long long id = capture_of(stream);
  p->recording = id != 0;
  if (state) p->taken = 1;
  if (id) {
    p->captured = 1;
    p->recorded_in = id;
    p->recorded_full = full;
    p->listed_in = state == 0 ? id : 0;
  } else {
    p->state = state;
    p->stream = reinterpret_cast<long long>(stream);
  }
}

// host_plan()'s arrays, until plan() sends them
thread_local std::unique_ptr<char[]> t_planned;
thread_local size_t t_planned_size = 0;

// The pinned mirror of an integer workspace.  Plans are laid out in it one behind the other: the copy that an
// earlier plan queued may still be reading its part, and waiting for it would mean waiting for everything queued
// before it.  A half of the mirror is written again when the copies out of it are done, which is looked at (and
// fenced, on the default stream) only where a plan enters the other half: half a lap ago, so that there is rarely
// anything left to wait for, and never for other streams.
struct Ring {
  PyObject_HEAD
  size_t off;
  int half;
  struct Half {
    bool on_default;                                    // copies on the default stream, fenced by ...
    hipEvent_t fence;                                   // ... this, recorded when the half is left
    std::vector<std::pair<hipStream_t, Word>> others;   // other streams: the last plan's word (written behind its copy)
  } halves[2];
};
PyTypeObject* g_ring_type = nullptr;

void ring_dealloc(PyObject* self) {
  Ring* r = reinterpret_cast<Ring*>(self);
  for (Ring::Half& h : r->halves) {
    if (h.fence) (void)hipEventDestroy(h.fence);
    h.others.~vector();
  }
  PyTypeObject* t = Py_TYPE(self);
  t->tp_free(self);
  Py_DECREF(t);
}

PyObject* new_ring(PyObject*, PyObject*) {
  PyObject* self = g_ring_type->tp_alloc(g_ring_type, 0);
  if (!self) return nullptr;
  for (Ring::Half& h : reinterpret_cast<Ring*>(self)->halves) new (&h.others) std::vector<std::pair<hipStream_t, Word>>();
  return self;
}

hipError_t leave_half(Ring::Half& h) {
  if (!h.on_default) return hipSuccess;
  c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);  // (another thread may be capturing)
  if (!h.fence) {
    const hipError_t e = hipEventCreateWithFlags(&h.fence, hipEventDisableTiming);
    if (e != hipSuccess) return e;
  }
  return hipEventRecord(h.fence, nullptr);
}

hipError_t enter_half(Ring::Half& h) {
  if (h.on_default) {
    c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
    const hipError_t e = host_wait(h.fence);
    if (e != hipSuccess) return e;
    h.on_default = false;
  }
  const auto others = std::move(h.others);
  h.others.clear();
  for (const auto& o : others)
    if (!wait_word(o.second)) return hipErrorNotReady;
  return hipSuccess;
}

// a part of the mirror for `used` bytes
hipError_t ring_take(Ring* r, size_t size, size_t used, size_t* at) {
  const size_t mid = size / 2;
  const bool large = used > mid;  // (then the whole mirror, alone)
  size_t off = r->off;
  int half = r->half;
  if (large) {
    hipError_t e = leave_half(r->halves[half]);
    if (e == hipSuccess) e = enter_half(r->halves[half]);
    if (e == hipSuccess) e = enter_half(r->halves[1 - half]);
    if (e != hipSuccess) return e;
    off = 0;
    half = 1;
  } else if (off + used > (half ? size : mid)) {
    hipError_t e = leave_half(r->halves[half]);
    if (e == hipSuccess) e = enter_half(r->halves[1 - half]);
    if (e != hipSuccess) return e;
    half = 1 - half;
    off = half ? mid : 0;
  }
  *at = off;
  r->off = large ? size : (off + used + 255) / 256 * 256;
  r->half = half;
  return hipSuccess;
}

// the copy out of the part just taken has been queued, and `word`'s launch behind it
void ring_note(Ring* r, bool large, hipStream_t stream, const Word& word) {
  for (int i = 0; i < 2; ++i) {
    Ring::Half& h = r->halves[i];
    if (i != r->half && !large) continue;
    if (!stream) {
      h.on_default = true;
      if (i != r->half) (void)leave_half(h);
      continue;
    }
    auto o = std::find_if(h.others.begin(), h.others.end(), [&](const auto& v) { return v.first == stream; });
    if (o == h.others.end()) h.others.emplace_back(stream, word);
    else o->second = word;
  }
}

PyObject* raise_captured_plan() {
  PyErr_SetString(PyExc_RuntimeError, "plan() cannot be captured in a graph");
  return nullptr;
}

// Work of the plan's is about to be queued on the current stream: behind the tables, which may still be on
// their way on the stream that planned them, and with their memory held until it is done.  Under capture the
// host waits for the tables: a graph does not know of work queued before it and is replayed on any stream, and a
// stream that is capturing takes no event for others.
hipError_t enter(Plan* p) {
  const c10::hip::HIPStream cur = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(p->dev));
  const hipStream_t s = cur.stream();
  if (s != p->home && std::find(p->used.begin(), p->used.end(), s) == p->used.end()) {
    c10::hip::HIPCachingAllocator::recordStream(p->tables.storage().data_ptr(), cur);
    p->used.push_back(s);
  }
  if (p->complete || (s == p->home && !capturing(s))) return hipSuccess;
  p->complete = p->word.arrived();
  if (p->complete) return hipSuccess;
  const bool by_host = capturing(s) || capturing(p->home);
  if (by_host && p->word.at) {
    p->complete = wait_word(p->word);
    return p->complete ? hipSuccess : hipErrorNotReady;
  }
  const c10::hip::HIPGuard device(static_cast<c10::DeviceIndex>(p->dev));  // (whose default stream is meant)
  c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);  // (this thread or another is capturing)
  if (!p->behind) {
    hipError_t e = hipEventCreateWithFlags(&p->behind, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(p->behind, p->home);
    if (e != hipSuccess) {
      if (p->behind) (void)hipEventDestroy(p->behind);
      p->behind = nullptr;
      return e;
    }
  } else {
    const hipError_t e = hipEventQuery(p->behind);
    p->complete = e == hipSuccess;
    if (e != hipErrorNotReady) return e;
    (void)hipGetLastError();
  }
  if (!by_host) return hipStreamWaitEvent(s, p->behind, 0);
  const hipError_t e = host_wait(p->behind);
  p->complete = e == hipSuccess;
  return e;
}

PyObject* raise_hip(hipError_t e) {
  PyErr_Format(PyExc_RuntimeError, "flashomni_amd: %s", hipGetErrorString(e));
  return nullptr;
}

void hold(const Tensor& t, int dev) {
  c10::hip::HIPCachingAllocator::recordStream(t.storage().data_ptr(),
                                              c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)));
}

// (Plan, work-list tensor or None): the current stream is about to use the plan's tables and the list's storage
PyObject* enter_plan(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor* list;
  if (n != 2 || Py_TYPE(args[0]) != g_plan_type || !opt_tensor(args[1], &list)) {
    PyErr_SetString(PyExc_RuntimeError, "enter_plan: bad argument");
    return nullptr;
  }
  Plan* p = reinterpret_cast<Plan*>(args[0]);
  const hipError_t e = enter(p);
  if (e != hipSuccess) return raise_hip(e);
  if (list) hold(*list, p->dev);
  Py_RETURN_NONE;
  TORCH_GUARD_END
}

// (qo_indptr, kv_indptr: int32 on the host; num_qo_heads, num_kv_heads, packed, device index,
//  qo_indptr, kv_indptr of the device or None; to send host_plan()'s arrays: their bytes, the integer
//  workspace, its pinned mirror and the mirror's Ring, or 0 and None; and whether runs may take their rows straight from
//  the symbols, if the float workspace and the soft cap of the moment, which can change, let them) -> (Plan, tables, sizes)
PyObject* plan(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor *qo, *kv, *qo_dev, *kv_dev, *iws, *pin;
  int64_t hq, hkv, dev, sent;
  if (!(n == 13 && opt_tensor(args[0], &qo) && qo && opt_tensor(args[1], &kv) && kv && whole(args[2], &hq) &&
        whole(args[3], &hkv) && whole(args[5], &dev) && whole(args[8], &sent) && opt_tensor(args[9], &iws) &&
        opt_tensor(args[10], &pin) && (sent == 0 || (iws && pin && Py_TYPE(args[11]) == g_ring_type)) &&
        opt_tensor(args[6], &qo_dev) && opt_tensor(args[7], &kv_dev) &&
        qo->scalar_type() == at::kInt && kv->scalar_type() == at::kInt && qo->is_contiguous() && kv->is_contiguous() &&
        qo->is_cpu() && kv->is_cpu() && qo->numel() == kv->numel() && qo->numel() >= 1)) {
    PyErr_SetString(PyExc_RuntimeError, "plan: bad argument");
    return nullptr;
  }
  hipStream_t home = static_cast<hipStream_t>(stream_of(dev));
  if (capturing(home)) return raise_captured_plan();
  const int batch = static_cast<int>(qo->numel()) - 1;
  const bool packed = truth(args[4]);
  fo_batch_sizes z;
  if (fo_plan_batch(qo->data_ptr<int32_t>(), kv->data_ptr<int32_t>(), batch, hq, hkv, packed, &z)) return raise_last();
  PyObject* self = g_plan_type->tp_alloc(g_plan_type, 0);
  if (!self) return nullptr;
  Plan* p = reinterpret_cast<Plan*>(self);
  new (&p->tables) Tensor();
  new (&p->used) std::vector<hipStream_t>();
  new (&p->qo_keep) Tensor();
  new (&p->kv_keep) Tensor();
  new (&p->parts) Tensor();
  p->dev = dev;
  p->batch = batch;
  p->num_qo = hq;
  p->num_kv = hkv;
  p->packed = packed;
  p->symbol_heads = packed ? hkv : hq;
  p->z = z;
  p->from_zero = qo->data_ptr<int32_t>()[0] == 0;
  p->state = 0;
  int rc = 0;
  int64_t ints = z.table_ints;
  if (truth(args[12]) && z.max_rows <= fo_sparse_attention_direct_max_pairs() && z.max_kv_len <= kMaxListed &&
      may_take(p, INT64_MAX, 0.)) {
    auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    // (symbol tensors much larger than the batch needs are not worth copying)
    p->keep_room[0] = z.min_info + 4096;
    p->keep_room[1] = z.min_kv_info + 4096;
    p->keep_at[0] = up(4 * ints);
    p->keep_at[1] = p->keep_at[0] + up(p->keep_room[0]);
    p->keep_at[2] = p->keep_at[1] + up(p->keep_room[1]);
    ints = p->keep_at[2] / 4 + 2 * (batch + 1);
  }
  try {
    p->tables = new_tensor({ints}, at::kInt, dev);
    p->home = home;
    if (home && !take_word(&p->word)) {
      Py_DECREF(self);
      PyErr_SetString(PyExc_RuntimeError, "hipHostMalloc failed");
      return nullptr;
    }
    Ring* ring = sent ? reinterpret_cast<Ring*>(args[11]) : nullptr;
    const size_t mirror = sent ? pin->numel() * pin->element_size() : 0;
    if (ring) {
      size_t at = 0;
      hipError_t e = static_cast<size_t>(sent) > mirror ? hipErrorInvalidValue : ring_take(ring, mirror, sent, &at);
      if (e == hipSuccess) {
        char* host = static_cast<char*>(pin->data_ptr()) + at;
        std::memcpy(host, t_planned.get(), sent);
        e = hipMemcpyAsync(iws->data_ptr(), host, sent, hipMemcpyHostToDevice, home);
      }
      if (e != hipSuccess) {
        settle_word(p->word);
        Py_DECREF(self);
        PyErr_Format(PyExc_RuntimeError, "the copy into the integer workspace failed: %s", hipGetErrorString(e));
        return nullptr;
      }
    }
    rc = fo_plan_tables_signal(qo->data_ptr<int32_t>(), kv->data_ptr<int32_t>(), batch, hq, hkv, packed,
                               p->tables.data_ptr<int32_t>(), p->word.at, p->word.ticket, p->home);
    if (rc) {
      (void)hipStreamSynchronize(home);  // (the copy has no word to be waited for by)
      settle_word(p->word);
    } else if (ring) {
      ring_note(ring, static_cast<size_t>(sent) > mirror / 2, home, p->word);
    }
  } catch (...) {
    Py_DECREF(self);
    throw;
  }
  if (rc) {
    Py_DECREF(self);
    return raise_last();
  }
  int32_t* t = p->tables.data_ptr<int32_t>();
  p->qo_indptr = t + z.qo_indptr;
  p->kv_indptr = t + z.kv_indptr;
  if (qo_dev && kv_dev) {  // (graph mode: a replay reads the caller's buffers)
    p->qo_keep = *qo_dev;
    p->kv_keep = *kv_dev;
    p->qo_indptr = qo_dev->data_ptr<int32_t>();
    p->kv_indptr = kv_dev->data_ptr<int32_t>();
  }
  const int64_t v[] = {z.n_q_blocks, z.n_kv_blocks, z.max_rows,   z.max_nnz,       z.total_q,     z.total_kv,
                       z.min_info,   z.min_kv_info, z.max_kv_len, z.qo_indptr,     z.kv_indptr,   z.blk_req,
                       z.blk_qb,     z.q_blk_base,  z.kv_blk_base, z.info_indptr,  z.kv_info_indptr};
  PyObject* sizes = PyTuple_New(17);
  for (int i = 0; i < 17; ++i) PyTuple_SET_ITEM(sizes, i, PyLong_FromLongLong(v[i]));
  return Py_BuildValue("(NNN)", self, THPVariable_Wrap(p->tables), sizes);
  TORCH_GUARD_END
}

// The host planner: (float workspace, integer workspace, qo_indptr, kv_indptr (host), rows, heads, kv heads, graph
// mode, element size, plan vector) -> bytes of its arrays, which plan() sends to the integer workspace from this
// thread's scratch.
PyObject* host_plan(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor *fws, *iws, *qo, *kv, *info;
  int64_t rows, hq, hkv, elem;
  if (!(n == 10 && opt_tensor(args[0], &fws) && fws && opt_tensor(args[1], &iws) && iws && opt_tensor(args[2], &qo) && qo &&
        opt_tensor(args[3], &kv) && kv && whole(args[4], &rows) && whole(args[5], &hq) && whole(args[6], &hkv) &&
        whole(args[8], &elem) && opt_tensor(args[9], &info) && info && info->scalar_type() == at::kLong && info->numel() == 15)) {
    PyErr_SetString(PyExc_RuntimeError, "plan: bad argument");
    return nullptr;
  }
  const bool graph = truth(args[7]);
  const int batch = static_cast<int>(qo->numel()) - 1;
  const size_t bytes = iws->numel() * iws->element_size();
  // (the planner writes the used prefix only: the rest of the scratch is never touched)
  if (t_planned_size < bytes) {
    t_planned.reset(new char[bytes]);
    t_planned_size = bytes;
  }
  int64_t* v = info->data_ptr<int64_t>();
  if (fo_prefill_plan(fws->data_ptr(), fws->numel() * fws->element_size(), nullptr, t_planned.get(), bytes,
                      qo->data_ptr<int32_t>(), kv->data_ptr<int32_t>(), rows, batch, hq, hkv, 128, 128, 1, graph, elem, 0,
                      v, nullptr))
    return raise_last();
  // end of the last array: block_valid_mask, else the row count (graph mode), else the chunk size
  return PyLong_FromLongLong(v[14] ? v[12] + v[0] : (v[13] ? v[2] : v[9]) + 4);
  TORCH_GUARD_END
}

// (Plan): the current stream waits for the stream of the last run (by its handle: torch has no stream object for
// the default stream's, 0, but hands out one of its pool).  Under capture nothing is waited for: a replay is
// ordered by whoever makes it.
PyObject* follow_run(PyObject*, PyObject* arg) {
  TORCH_GUARD_BEGIN
  if (Py_TYPE(arg) != g_plan_type) {
    PyErr_SetString(PyExc_RuntimeError, "not a plan");
    return nullptr;
  }
  Plan* p = reinterpret_cast<Plan*>(arg);
  const hipStream_t cur = static_cast<hipStream_t>(stream_of(p->dev)), ran = reinterpret_cast<hipStream_t>(p->stream);
  if (cur == ran || capturing(cur)) Py_RETURN_NONE;
  if (capturing(ran)) {
    PyErr_SetString(PyExc_RuntimeError, "the stream of the last run() is being captured: its list cannot be reused on another");
    return nullptr;
  }
  const c10::hip::HIPGuard device(static_cast<c10::DeviceIndex>(p->dev));  // (whose default stream is meant)
  hipEvent_t ev;
  hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  if (e != hipSuccess) return raise_hip(e);
  e = hipEventRecord(ev, ran);
  if (e == hipSuccess) e = hipStreamWaitEvent(cur, ev, 0);
  const hipError_t destroyed = hipEventDestroy(ev);  // (what was queued stays)
  if (e == hipSuccess) e = destroyed;
  if (e != hipSuccess) return raise_hip(e);
  Py_RETURN_NONE;
  TORCH_GUARD_END
}

// (Plan, is_full): a list has been decoded on the current stream
PyObject* note_list(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  if (n != 2 || Py_TYPE(args[0]) != g_plan_type) {
    PyErr_SetString(PyExc_RuntimeError, "note_list: bad argument");
    return nullptr;
  }
  Plan* p = reinterpret_cast<Plan*>(args[0]);
  note(p, static_cast<hipStream_t>(stream_of(p->dev)), 0, truth(args[1]));
  Py_RETURN_NONE;
  TORCH_GUARD_END
}

// (Plan, bytes of the float workspace that parts of rows may lie in, soft cap) -> how a reuse on the current stream gets
// its list: 0: as it is; 1: decoded from what the last run left behind; 2: the device decides between the two
// (fo_decode_sparse_kept).
PyObject* list_source(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  int64_t ws_bytes;
  double cap;
  if (!(n == 3 && Py_TYPE(args[0]) == g_plan_type && whole(args[1], &ws_bytes) && real(args[2], &cap))) {
    PyErr_SetString(PyExc_RuntimeError, "list_source: bad argument");
    return nullptr;
  }
  Plan* p = reinterpret_cast<Plan*>(args[0]);
  const unsigned long long id = capture_of(static_cast<hipStream_t>(stream_of(p->dev)));
  if (id) p->captured = 1;
  // A reuse that is recorded now may be replayed behind a run that takes its rows from the symbols later on.  Where runs like
  // this one never do, there will be none: should workspace or cap change, such runs are decoded.
  if (id && p->keep_at[0] && p->listed_in != id && !p->taken && !may_take(p, ws_bytes, cap)) p->list_only = 1;
  const bool list = !p->keep_at[0] || p->list_only || (id ? p->listed_in == id : !p->taken);
  const int source = list ? 0 : p->captured ? 2 : p->state != 0;
  return PyLong_FromLong(source);
  TORCH_GUARD_END
}

// (Plan) -> the capture that the current stream is in, 0: none
PyObject* capture(PyObject*, PyObject* arg) {
  TORCH_GUARD_BEGIN
  if (Py_TYPE(arg) != g_plan_type) {
    PyErr_SetString(PyExc_RuntimeError, "not a plan");
    return nullptr;
  }
  return PyLong_FromUnsignedLongLong(capture_of(static_cast<hipStream_t>(stream_of(reinterpret_cast<Plan*>(arg)->dev))));
  TORCH_GUARD_END
}

// (Plan) -> room for (sparse_info, sparse_kv_info, the two indptrs) as the last run without a list read them
PyObject* kept_symbols(PyObject*, PyObject* arg) {
  TORCH_GUARD_BEGIN
  if (Py_TYPE(arg) != g_plan_type || !reinterpret_cast<Plan*>(arg)->keep_at[0]) {
    PyErr_SetString(PyExc_RuntimeError, "no symbols kept");
    return nullptr;
  }
  Plan* p = reinterpret_cast<Plan*>(arg);
  const int64_t n = p->batch + 1, ip = p->keep_at[2] / 4;
  const Tensor bytes = p->tables.view(at::kByte);
  return Py_BuildValue("(NNNN)", THPVariable_Wrap(bytes.narrow(0, p->keep_at[0], p->keep_room[0])),
                       THPVariable_Wrap(bytes.narrow(0, p->keep_at[1], p->keep_room[1])),
                       THPVariable_Wrap(p->tables.narrow(0, ip, n)), THPVariable_Wrap(p->tables.narrow(0, ip + n, n)));
  TORCH_GUARD_END
}

// attention of an ordinary call: (plan, q, k, v, sparse_info, sparse_kv_info, sparse_info_indptr,
// sparse_kv_info_indptr, is_full, out, lse, return_lse, sm_scale, logits_soft_cap, HND, work-list tensors
// or None, float workspace or None, indptrs of the q and kv tokens or None: the plan's) -> out or (out, lse);
// False: needs the work-list tensors
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  FALL_BACK_UNLESS(n == 19 && Py_TYPE(args[0]) == g_plan_type);
  Plan* p = reinterpret_cast<Plan*>(args[0]);
  const int dev = p->dev;
  const Tensor *q, *k, *v, *sym[4], *out, *lse, *ws, *ip[2];
  double sm_scale, cap;
  FALL_BACK_UNLESS(dev == c10::hip::current_device() && opt_tensor(args[1], &q) && q && opt_tensor(args[2], &k) && k &&
                   opt_tensor(args[3], &v) && v && opt_tensor(args[4], &sym[0]) && opt_tensor(args[5], &sym[1]) &&
                   opt_tensor(args[6], &sym[2]) && opt_tensor(args[7], &sym[3]) && opt_tensor(args[9], &out) &&
                   opt_tensor(args[10], &lse) && real(args[13], &cap) && opt_tensor(args[16], &ws) &&
                   opt_tensor(args[17], &ip[0]) && opt_tensor(args[18], &ip[1]));
  for (const Tensor* t : ip)
    FALL_BACK_UNLESS(!t || (flat(*t, at::kInt, dev) && t->numel() == p->batch + 1));
  const bool full = truth(args[8]), want_lse = truth(args[11]), hnd = truth(args[14]);
  const int code = act_code(q->scalar_type());
  FALL_BACK_UNLESS(code >= 0 && on(*q, dev) && on(*k, dev) && on(*v, dev) && k->scalar_type() == q->scalar_type() &&
                   v->scalar_type() == q->scalar_type() && q->dim() == 3 && k->dim() == 3 && v->dim() == 3);
  const int kn = hnd ? 1 : 0, kh = 1 - kn;
  FALL_BACK_UNLESS(q->size(1) == p->num_qo && q->size(2) == 128 && k->size(2) == 128 && v->size(2) == 128 &&
                   k->size(kh) == p->num_kv && v->size(kh) == p->num_kv && q->size(0) >= p->z.total_q &&
                   k->size(kn) >= p->z.total_kv && v->size(kn) >= p->z.total_kv && q->stride(2) == 1 &&
                   k->stride(2) == 1 && v->stride(2) == 1);
  if (args[12] == Py_None) {
    sm_scale = 1.0 / std::sqrt(128.0);
  } else {
    FALL_BACK_UNLESS(real(args[12], &sm_scale));
  }
  if (!full) {
    FALL_BACK_UNLESS(sym[0] && sym[1] && sym[2] && sym[3] && flat(*sym[0], at::kByte, dev) &&
                     flat(*sym[1], at::kByte, dev) && flat(*sym[2], at::kInt, dev) && flat(*sym[3], at::kInt, dev) &&
                     sym[0]->numel() >= p->z.min_info && sym[1]->numel() >= p->z.min_kv_info &&
                     sym[2]->numel() == p->batch + 1 && sym[3]->numel() == p->batch + 1);
  }
  FALL_BACK_UNLESS(!out || (on(*out, dev) && out->scalar_type() == q->scalar_type() && out->sizes() == q->sizes() &&
                            out->stride(2) == 1));
  FALL_BACK_UNLESS(!want_lse || !lse || (flat(*lse, at::kFloat, dev) && lse->dim() == 2 && lse->size(0) == q->size(0) &&
                                         lse->size(1) == q->size(1)));
  // work-list buffers, in the order of fo_decode_sparse's outputs
  int32_t* wl[10] = {};
  if (args[15] != Py_None) {
    FALL_BACK_UNLESS(PyTuple_Check(args[15]) && PyTuple_GET_SIZE(args[15]) == 10);
    for (int i = 0; i < 10; ++i) {
      PyObject* o = PyTuple_GET_ITEM(args[15], i);
      FALL_BACK_UNLESS(THPVariable_Check(o));
      wl[i] = static_cast<int32_t*>(THPVariable_Unpack(o).data_ptr());
    }
  }

  const hipError_t entered = enter(p);
  if (entered != hipSuccess) return raise_hip(entered);
  void* stream = stream_of(dev);
  int32_t* t = p->tables.data_ptr<int32_t>();
  auto bytes = [&](int i) { return full ? nullptr : static_cast<const uint8_t*>(sym[i]->data_ptr()); };
  auto ints = [&](int i) { return full ? nullptr : static_cast<const int32_t*>(sym[i]->data_ptr()); };
  Tensor fresh_lse;
  if (want_lse && !lse) fresh_lse = new_tensor({q->size(0), q->size(1)}, at::kFloat, dev);

  fo_attention_args a{};
  a.q = q->data_ptr(); a.k = k->data_ptr(); a.v = v->data_ptr();
  a.lse = !want_lse ? nullptr : lse ? lse->data_ptr<float>() : fresh_lse.data_ptr<float>();
  a.q_stride_n = q->stride(0); a.q_stride_h = q->stride(1);
  a.k_stride_n = k->stride(kn); a.k_stride_h = k->stride(kh);
  a.v_stride_n = v->stride(kn); a.v_stride_h = v->stride(kh);
  a.info = bytes(0); a.kv_info = bytes(1); a.info_indptr = ints(2); a.kv_info_indptr = ints(3);
  a.qo_indptr = ip[0] ? ip[0]->data_ptr<int32_t>() : p->qo_indptr;
  a.kv_indptr = ip[1] ? ip[1]->data_ptr<int32_t>() : p->kv_indptr;
  a.blk_req = t + p->z.blk_req; a.blk_qb = t + p->z.blk_qb;
  a.sched = t + p->z.sched;
  a.split_ws = ws ? ws->data_ptr() : nullptr;
  a.split_ws_bytes = ws ? ws->numel() * ws->element_size() : 0;
  a.max_nnz = p->z.max_nnz;
  a.dtype = code; a.n_blk = p->z.n_q_blocks; a.batch = p->batch; a.symbol_heads = p->symbol_heads;
  a.num_heads = p->num_qo; a.num_kv_heads = p->num_kv; a.gqa_packed = p->packed; a.is_full = full;
  a.sm_scale = static_cast<float>(sm_scale); a.logits_soft_cap = static_cast<float>(cap);
  a.stream = stream;

  Tensor fresh;
  // the launch without a decoded list (it clears what it skips: every row of a fresh output is its own)
  const bool own = !out && p->from_zero && q->size(0) == p->z.total_q;
  const bool small = p->keep_at[0] && !p->list_only && (full || (sym[0]->numel() <= p->keep_room[0] && sym[1]->numel() <= p->keep_room[1]));
  int rc = FO_NOT_DIRECT;
  const int64_t parts = small && !p->no_parts ? fo_sparse_attention_direct_own_bytes(&a) : 0;
  if (parts && !p->parts.defined()) {
    try {
      p->parts = new_tensor({parts}, at::kByte, dev);
    } catch (const c10::OutOfMemoryError&) {
      p->no_parts = true;  // (a request that fails has the allocator give its cached blocks back first, which waits)
    }
  }
  const bool own_parts = parts && p->parts.defined();
  if (own_parts || (small && fo_sparse_attention_direct_serves(&a))) {
    if (own_parts) {
      hold(p->parts, dev);
      a.split_ws = p->parts.data_ptr();
      a.split_ws_bytes = p->parts.numel();
    }
    if (!out) fresh = own ? at::empty(q->sizes(), q->options()) : at::zeros(q->sizes(), q->options());
    const Tensor& o = out ? *out : fresh;
    a.o = o.data_ptr();
    a.o_stride_n = o.stride(0);
    a.o_stride_h = o.stride(1);
    a.zero_skipped = own;
    if (!full) {
      a.keep_info = reinterpret_cast<uint8_t*>(t) + p->keep_at[0];
      a.keep_kv_info = reinterpret_cast<uint8_t*>(t) + p->keep_at[1];
      a.info_bytes = sym[0]->numel();
      a.kv_info_bytes = sym[1]->numel();
    }
    a.keep_indptr = t + p->keep_at[2] / 4;
    rc = own_parts ? fo_sparse_attention_direct_own(&a) : fo_sparse_attention_direct(&a);
    if (rc < 0) return raise_last();
    if (rc == FO_OK) note(p, static_cast<hipStream_t>(stream), full ? 2 : 1, full);
  }
  if (rc == FO_NOT_DIRECT) {
    if (args[15] == Py_None) Py_RETURN_FALSE;
    hold(THPVariable_Unpack(PyTuple_GET_ITEM(args[15], 0)), dev);  // (the ten share one storage)
    // (the decoder's launches for longer lists clear the rows of a fresh output that nothing computes)
    const bool clears = own && int64_t(p->z.n_q_blocks) * p->symbol_heads >= fo_decode_sparse_clear_min_pairs();
    if (!out) fresh = clears ? at::empty(q->sizes(), q->options()) : at::zeros(q->sizes(), q->options());
    const Tensor& o = out ? *out : fresh;
    int32_t* shares = ws ? wl[9] : nullptr;
    if (clears ? fo_decode_sparse_clear(a.info, a.kv_info, a.info_indptr, a.kv_info_indptr, a.blk_req, a.blk_qb,
                                        a.kv_indptr, p->z.n_q_blocks, p->symbol_heads, 128, full, wl[0], wl[1], wl[2],
                                        wl[3], wl[4], wl[5], wl[6], wl[7], wl[8], shares, o.data_ptr(), o.stride(0),
                                        o.stride(1), a.qo_indptr, p->packed ? p->num_qo / p->num_kv : 1, stream)
               : fo_decode_sparse(a.info, a.kv_info, a.info_indptr, a.kv_info_indptr, a.blk_req, a.blk_qb, a.kv_indptr,
                                  p->z.n_q_blocks, p->symbol_heads, 128, full, wl[0], wl[1], wl[2], wl[3], wl[4], wl[5],
                                  wl[6], wl[7], wl[8], shares, stream))
      return raise_last();
    if (fo_sparse_fa_run(a.q, a.k, a.v, o.data_ptr(), a.lse, code, nullptr, nullptr, nullptr, nullptr, a.q_stride_n,
                         a.q_stride_h, a.k_stride_n, a.k_stride_h, a.v_stride_n, a.v_stride_h, o.stride(0), o.stride(1),
                         a.qo_indptr, a.kv_indptr, t + p->z.q_blk_base, t + p->z.kv_blk_base, p->z.n_q_blocks,
                         p->z.n_kv_blocks, wl[0], wl[1], wl[2], wl[3], wl[4], wl[6], wl[7], p->z.max_rows, p->num_qo,
                         p->num_kv, p->packed, 128, 128, 128, a.sm_scale, a.logits_soft_cap, shares, a.split_ws,
                         a.split_ws_bytes, stream))
      return raise_last();
    note(p, static_cast<hipStream_t>(stream), 0, full);
  }
  PyObject* ret = args[9];
  if (out) {
    Py_INCREF(ret);
  } else {
    ret = THPVariable_Wrap(std::move(fresh));
  }
  if (!want_lse || !ret) return ret;
  PyObject* l = args[10];
  if (lse) {
    Py_INCREF(l);
  } else {
    l = THPVariable_Wrap(std::move(fresh_lse));
  }
  return Py_BuildValue("(NN)", ret, l);
  TORCH_GUARD_END
}

// ---- bit packing ---------------------------------------------------------------------------------
bool bool_bytes(const Tensor* x, int* dev) {
  if (!x || !x->is_cuda() || !x->is_contiguous()) return false;
  *dev = x->get_device();
  const auto t = x->scalar_type();
  return *dev == c10::hip::current_device() && (t == at::kBool || t == at::kByte || t == at::kChar);
}

// (x, bit order code) -> y
PyObject* packbits(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor* x;
  int64_t code;
  int dev;
  FALL_BACK_UNLESS(n == 2 && opt_tensor(args[0], &x) && bool_bytes(x, &dev) && whole(args[1], &code));
  Tensor y = new_tensor({(x->numel() + 7) / 8}, at::kByte, dev);
  if (fo_packbits(static_cast<const uint8_t*>(x->data_ptr()), x->numel(), code, static_cast<uint8_t*>(y.data_ptr()),
                  stream_of(dev)))
    return raise_last();
  return THPVariable_Wrap(std::move(y));
  TORCH_GUARD_END
}

// Words of pinned memory that kernels leave a length in.  A call takes one and puts it back; there are
// as many as calls have ever waited at the same time (guarded by the interpreter's lock).
std::vector<uint64_t*> g_words;
uint32_t g_ticket = 0;

// (x, indptr, bit order code) -> (y, indptr of y)
PyObject* segment_packbits(PyObject*, PyObject* const* args, Py_ssize_t n) {
  TORCH_GUARD_BEGIN
  const Tensor *x, *ip;
  int64_t code;
  int dev;
  FALL_BACK_UNLESS(n == 3 && opt_tensor(args[0], &x) && bool_bytes(x, &dev) && opt_tensor(args[1], &ip) && ip &&
                   on(*ip, dev) && ip->dim() == 1 && ip->is_contiguous() && ip->numel() >= 2 && ip->numel() <= 1025 &&
                   (ip->scalar_type() == at::kInt || ip->scalar_type() == at::kLong) && whole(args[2], &code));
  hipStream_t stream = static_cast<hipStream_t>(stream_of(dev));
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  FALL_BACK_UNLESS(hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone);
  const int64_t segments = ip->numel() - 1, capacity = (x->numel() + 7 * segments) / 8;
  FALL_BACK_UNLESS(capacity < (int64_t(1) << 31));
  if (g_words.empty()) {
    void* w = nullptr;
    if (hipHostMalloc(&w, 64, hipHostMallocCoherent) != hipSuccess) {
      PyErr_SetString(PyExc_RuntimeError, "hipHostMalloc failed");
      return nullptr;
    }
    g_words.push_back(static_cast<uint64_t*>(w));
  }
  Tensor y = new_tensor({capacity}, at::kByte, dev), out_ip = new_tensor({segments + 1}, at::kInt, dev);
  uint64_t* word = g_words.back();
  g_words.pop_back();
  const uint32_t ticket = ++g_ticket;
  *static_cast<volatile uint64_t*>(word) = static_cast<uint64_t>(~ticket) << 32;
  const int rc = fo_segment_packbits_scan(static_cast<const uint8_t*>(x->data_ptr()), x->numel(), ip->data_ptr(),
                                          ip->scalar_type() == at::kLong, segments, code,
                                          static_cast<uint8_t*>(y.data_ptr()), capacity, out_ip.data_ptr<int32_t>(), word,
                                          ticket, stream);
  uint64_t got = 0;
  bool arrived = false;
  hipError_t err = hipSuccess;
  if (!rc) {
    // The word arrives 8-11 us after the call where nothing else is queued: looked at for 50 us, then the stream
    // is waited for (the kernel may be behind other work; that wait takes 12 us by itself.  A limit of 20000
    // looks was about 10 us long: calls fell on either side of it, 11 or 23 us, with the code around the loop.)
    Py_BEGIN_ALLOW_THREADS
    const auto limit = std::chrono::steady_clock::now() + std::chrono::microseconds(50);
    do {
      for (int look = 0; look < 64 && !arrived; ++look) {
        got = *static_cast<volatile uint64_t*>(word);
        arrived = got >> 32 == ticket;
      }
    } while (!arrived && std::chrono::steady_clock::now() < limit);
    if (!arrived) {
      err = hipStreamSynchronize(stream);
      got = *static_cast<volatile uint64_t*>(word);
      arrived = got >> 32 == ticket;
    }
    Py_END_ALLOW_THREADS
  }
  g_words.push_back(word);
  if (rc) return raise_last();
  if (err != hipSuccess || !arrived) {
    PyErr_SetString(PyExc_RuntimeError, hipGetErrorString(err));
    return nullptr;
  }
  const int32_t total = static_cast<int32_t>(static_cast<uint32_t>(got));
  FALL_BACK_UNLESS(total >= 0);
  if (total != capacity) y = y.narrow(0, 0, total);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(y)), THPVariable_Wrap(std::move(out_ip)));
  TORCH_GUARD_END
}

#define FASTCALL(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef g_methods[] = {
    {"gemm_q", FASTCALL(gemm_q), nullptr},
    {"gemm_o", FASTCALL(gemm_o), nullptr},
    {"plan", FASTCALL(plan), nullptr},
    {"host_plan", FASTCALL(host_plan), nullptr},
    {"new_ring", new_ring, METH_NOARGS, nullptr},
    {"attention", FASTCALL(attention), nullptr},
    {"enter_plan", FASTCALL(enter_plan), nullptr},
    {"follow_run", follow_run, METH_O, nullptr},
    {"note_list", FASTCALL(note_list), nullptr},
    {"list_source", FASTCALL(list_source), nullptr},
    {"capture", capture, METH_O, nullptr},
    {"kept_symbols", kept_symbols, METH_O, nullptr},
    {"packbits", FASTCALL(packbits), nullptr},
    {"segment_packbits", FASTCALL(segment_packbits), nullptr},
    {"set_gemm_scratch", set_gemm_scratch, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

PyMemberDef g_plan_members[] = {{"state", T_INT, offsetof(Plan, state), 0, nullptr},
                                {"recorded_in", T_ULONGLONG, offsetof(Plan, recorded_in), 0, nullptr},
                                {"recording", T_INT, offsetof(Plan, recording), READONLY, nullptr},
                                {"recorded_full", T_INT, offsetof(Plan, recorded_full), READONLY, nullptr},
                                {"from_zero", T_BOOL, offsetof(Plan, from_zero), READONLY, nullptr},
                                {"sched_at", T_LONGLONG, offsetof(Plan, z.sched), READONLY, nullptr},
                                {nullptr, 0, 0, 0, nullptr}};
PyType_Slot g_ring_slots[] = {{Py_tp_dealloc, reinterpret_cast<void*>(ring_dealloc)}, {0, nullptr}};
PyType_Spec g_ring_spec = {"flashomni_amd._native.Ring", sizeof(Ring), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_DISALLOW_INSTANTIATION,
                           g_ring_slots};
PyType_Slot g_plan_slots[] = {{Py_tp_dealloc, reinterpret_cast<void*>(plan_dealloc)},
                              {Py_tp_members, g_plan_members},
                              {0, nullptr}};
PyType_Spec g_plan_spec = {"flashomni_amd._native.Plan", sizeof(Plan), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_DISALLOW_INSTANTIATION,
                           g_plan_slots};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  g_ring_type = reinterpret_cast<PyTypeObject*>(PyType_FromSpec(&g_ring_spec));
  if (!g_ring_type) return nullptr;
  g_plan_type = reinterpret_cast<PyTypeObject*>(PyType_FromSpec(&g_plan_spec));
  if (!g_plan_type) return nullptr;
  return PyModule_Create(&g_module);
}
