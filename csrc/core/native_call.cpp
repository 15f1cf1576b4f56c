#include "native_call.hpp"

#include <algorithm>
#include <memory>

namespace lc {
namespace {

constexpr const char* kCapsule = "lc.native_fn";

// The System V calling convention of x86-64 hands integers and pointers on in one sequence (six registers, then 8-byte stack slots) and up to
// eight floats in another (vector registers), whatever their order among each other. A function whose arguments are
// ints, 64-bit ints, pointers and at most eight floats therefore finds them where a prototype of all its integers followed by
// all its floats puts them; integers past its own are stack slots that it does not look at.
#if defined(__x86_64__) && !defined(_WIN32)
constexpr bool kKnownConvention = true;
#else
constexpr bool kKnownConvention = false;
#endif

#define LC_W8(b) w[b], w[b + 1], w[b + 2], w[b + 3], w[b + 4], w[b + 5], w[b + 6], w[b + 7]
#define LC_U8 uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t
#define LC_F8 float, float, float, float, float, float, float, float

int invoke(void* address, int words, const uint64_t* w, const float* f) {
  if (words <= 16)
    return reinterpret_cast<int (*)(LC_U8, LC_U8, LC_F8)>(address)(LC_W8(0), LC_W8(8), f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
  if (words <= 32)
    return reinterpret_cast<int (*)(LC_U8, LC_U8, LC_U8, LC_U8, LC_F8)>(address)(LC_W8(0), LC_W8(8), LC_W8(16), LC_W8(24), f[0], f[1], f[2],
                                                                                 f[3], f[4], f[5], f[6], f[7]);
  return reinterpret_cast<int (*)(LC_U8, LC_U8, LC_U8, LC_U8, LC_U8, LC_U8, LC_F8)>(address)(
      LC_W8(0), LC_W8(8), LC_W8(16), LC_W8(24), LC_W8(32), LC_W8(40), f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
}

PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  auto* fn = static_cast<NativeFn*>(PyCapsule_GetPointer(self, kCapsule));
  if (fn == nullptr) return nullptr;
  if (n != static_cast<Py_ssize_t>(fn->kinds.size())) Py_RETURN_NOTIMPLEMENTED;
  uint64_t w[NativeFn::kMaxWords] = {};
  float f[NativeFn::kMaxFloats] = {};
  int words = 0, floats = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* a = args[i];
    if (fn->kinds[i] == 'F') {
      if (!PyFloat_Check(a)) Py_RETURN_NOTIMPLEMENTED;
      f[floats++] = static_cast<float>(PyFloat_AS_DOUBLE(a));
    } else if (PyLong_Check(a)) {
      w[words++] = PyLong_AsUnsignedLongLongMask(a);      // (an int argument reads the low half, as a C conversion would leave it)
    } else if (a == Py_None && fn->kinds[i] == 'P') {
      w[words++] = 0;
    } else {
      Py_RETURN_NOTIMPLEMENTED;
    }
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = invoke(fn->address, words, w, f);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

void destroy(PyObject* capsule) { delete static_cast<NativeFn*>(PyCapsule_GetPointer(capsule, kCapsule)); }

}  // namespace

PyObject* make_native_call(uint64_t address, const std::string& kinds, const std::string& name) {
  const auto floats = std::count(kinds.begin(), kinds.end(), 'F');
  if (!kKnownConvention || address == 0 || kinds.find_first_not_of("PILF") != std::string::npos || floats > NativeFn::kMaxFloats ||
      static_cast<int>(kinds.size()) - floats > NativeFn::kMaxWords) {
    PyErr_SetString(PyExc_ValueError, "native call: a null address, or argument kinds that it does not take");
    return nullptr;
  }
  auto fn = std::make_unique<NativeFn>();
  fn->address = reinterpret_cast<void*>(address);
  fn->kinds = kinds;
  fn->name = name;
  fn->def = {fn->name.c_str(), reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call)), METH_FASTCALL, nullptr};
  PyMethodDef* def = &fn->def;
  PyObject* self = PyCapsule_New(fn.get(), kCapsule, destroy);
  if (self == nullptr) return nullptr;
  fn.release();                                            // (the capsule's from here on)
  PyObject* f = PyCFunction_New(def, self);
  Py_DECREF(self);
  return f;
}

}  // namespace lc
