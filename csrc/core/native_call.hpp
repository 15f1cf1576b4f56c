// Calls of C functions by address from Python: what ctypes does for a launcher of some thirty arguments takes 2 - 3 us of
// conversions (each through an object of its argument's type), this about 0.2.
#pragma once

#include <Python.h>

#include <cstdint>
#include <string>

namespace lc {

// A C function that returns int, and the kinds of its arguments: 'P' pointer (int or None), 'I' int, 'L' 64-bit int, 'F' float.
struct NativeFn {
  static constexpr int kMaxWords = 48, kMaxFloats = 8;
  void* address;
  std::string kinds, name;
  PyMethodDef def;
};

// Python callable over ``address``. It returns the function's int, or NotImplemented, without calling it, for arguments of another
// number or of other types than Python's int, float and None (the caller then takes the general way). The GIL is released
// around the call. Returns nullptr with an exception set for kinds that it does not know or too many of them.
PyObject* make_native_call(uint64_t address, const std::string& kinds, const std::string& name);

}  // namespace lc
