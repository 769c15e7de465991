#pragma once

#include <Python.h>

namespace mccl {

/// Adds the `_fast_*` functions (FastCalls.cpp) to the extension module.
void add_fast_calls(PyObject* module);

}  // namespace mccl
