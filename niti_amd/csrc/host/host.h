// Helpers of the tensor front end (host.cpp, conv.cpp, linear.cpp): argument access, allocation, error reporting.
//
// The front end is the part of niti_amd/ops.py that runs on every call - argument checks, output allocation, sync words,
// the call into the C ABI - as native code.  A launch takes the GPU 5 - 20 us at the sizes of a layer; the same steps in
// Python took 12 - 20 us per launch, so an eager step waited for its host.
#pragma once
#include <Python.h>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <initializer_list>
#include <stdexcept>
#include <string>

#include "niti_gfx950.h"

namespace niti_host {

// A refused call: RuntimeError, or niti_amd._lib.NitiError where the C ABI refused it.
struct Refused : std::runtime_error {
  bool niti;
  Refused(const std::string& what, bool niti_error) : std::runtime_error(what), niti(niti_error) {}
};
[[noreturn]] inline void refuse(const std::string& what) { throw Refused(what, false); }
[[noreturn]] inline void refuse_niti(const std::string& what) { throw Refused(what, true); }

inline void check(int status, const char* who) {
  if (status != NITI_OK)
    refuse_niti(std::string(who) + ": " + niti_status_string(status) + " (" + niti_last_error() + ")");
}
// true when the call was refused because its grid does not fit the device (the caller then takes the separate steps)
inline bool check_fits(int status, const char* who) {
  if (status == NITI_ERR_UNSUPPORTED && std::string(niti_last_error()).find("do not fit") != std::string::npos) return false;
  check(status, who);
  return true;
}

using Opt = const at::Tensor*;   // nullptr for None

// Positional arguments of a METH_FASTCALL function, taken in order.
class Args {
 public:
  Args(PyObject* const* args, Py_ssize_t n, Py_ssize_t want, const char* who) : a_(args) {
    if (n != want) refuse(std::string(who) + ": " + std::to_string(want) + " arguments expected, got " + std::to_string(n));
  }
  const at::Tensor& tensor() {
    PyObject* o = a_[i_++];
    if (!THPVariable_Check(o)) refuse("niti_amd: tensor expected");
    return use(THPVariable_Unpack(o));
  }
  Opt opt() {
    PyObject* o = a_[i_++];
    if (o == Py_None) return nullptr;
    if (!THPVariable_Check(o)) refuse("niti_amd: tensor or None expected");
    return &use(THPVariable_Unpack(o));
  }
  Opt exponent() {   // one value, as a layer hands it on
    Opt t = opt();
    if (t != nullptr && (t->numel() != 1 || t->scalar_type() != at::kInt)) refuse("niti_amd: an exponent is one int32 value");
    return t;
  }
  long integer() {
    const long v = PyLong_AsLong(a_[i_++]);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
  }
  int i() { return static_cast<int>(integer()); }
  bool flag() { return PyObject_IsTrue(a_[i_++]) == 1; }

 private:
  static const at::Tensor& use(const at::Tensor& t) {
    if (!t.is_cuda()) refuse("niti_amd: tensor must live on the GPU");
    if (!t.is_contiguous()) refuse("niti_amd: tensor must be contiguous");
    return t;
  }
  PyObject* const* a_;
  int i_ = 0;
};

template <typename T = void>
inline T* ptr(const at::Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}
template <typename T = void>
inline T* ptr(Opt t) {
  return t == nullptr ? nullptr : static_cast<T*>(t->data_ptr());
}

inline at::Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt));
}
inline at::Tensor empty8(at::IntArrayRef shape, const at::Tensor& like) { return empty(shape, at::kChar, like); }
inline at::Tensor empty32(at::IntArrayRef shape, const at::Tensor& like) { return empty(shape, at::kInt, like); }
// An uninitialised int32 tensor of one element: exponents and shifts, of which a layer returns several per call.  They are cut
// from blocks of 128 (an allocation takes longer than everything else about such a tensor); no element is handed out twice.
at::Tensor scalar32(const at::Tensor& like);

inline void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

inline bool has_shape(const at::Tensor& t, at::IntArrayRef shape) { return t.sizes() == shape; }
// a launch reads or writes `bytes` of t: a tensor of other extents than the rest of the call's must not be smaller
inline void want_bytes(const at::Tensor& t, int64_t bytes, const char* who, const char* what) {
  if (static_cast<int64_t>(t.nbytes()) < bytes)
    refuse(std::string(who) + ": " + what + " of " + std::to_string(bytes) + " bytes expected, got " + std::to_string(t.nbytes()));
}
inline void want_i8(const at::Tensor& t, const char* who) {
  if (t.scalar_type() != at::kChar) refuse(std::string(who) + ": int8 tensor expected");
}

// ---- zeroed sync words -------------------------------------------------------------------------------------------
// `words` zeroed 32-bit words of the device's arena; `view` receives a tensor over them where the caller hands them out.
uint32_t* arena_take(long words, const at::Tensor& like, at::Tensor* view);
// the sync words of a call: the caller's tensor, or a slice of the arena
inline uint32_t* sync_words(Opt sync, size_t words, const at::Tensor& like, at::Tensor* view, size_t* have, const char* who) {
  if (sync == nullptr) {
    *have = words;
    return arena_take(static_cast<long>(words), like, view);
  }
  if (sync->scalar_type() != at::kInt || sync->numel() < static_cast<int64_t>(words))
    refuse(std::string(who) + ": sync must be a zeroed int32 tensor of at least " + std::to_string(words) + " words");
  if (view != nullptr) *view = *sync;
  *have = static_cast<size_t>(sync->numel());
  return static_cast<uint32_t*>(sync->data_ptr());
}

// `bytes` of scratch memory that the caller may use until its next call on this stream
at::Tensor scratch(size_t bytes, const at::Tensor& like);
// int32 product op(a) @ op(b); absmax (zeroed word) receives max|c|
at::Tensor gemm(const at::Tensor& a, const at::Tensor& b, bool ta, bool tb, uint32_t* absmax);

// ---- results -----------------------------------------------------------------------------------------------------
inline PyObject* wrap(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
inline PyObject* tuple_of(std::initializer_list<at::Tensor> ts) {
  PyObject* out = PyTuple_New(static_cast<Py_ssize_t>(ts.size()));
  if (out == nullptr) throw python_error();
  Py_ssize_t i = 0;
  for (const at::Tensor& t : ts) PyTuple_SET_ITEM(out, i++, wrap(t));
  return out;
}

PyObject* raise(const Refused& e);
template <typename F>
inline PyObject* guarded(F f) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const Refused& e) {
    return raise(e);
  }
  END_HANDLE_TH_ERRORS
}

// tables of the other translation units
extern PyMethodDef kConvMethods[];
extern PyMethodDef kLinearMethods[];

}  // namespace niti_host
