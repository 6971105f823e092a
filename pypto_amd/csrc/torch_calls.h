// The operators' native call path (torch_calls.cpp): functions added to the extension module.
#pragma once
#include <Python.h>

namespace pto {
// 0, or -1 with a Python error set
int add_torch_calls(PyObject *module);
}  // namespace pto
