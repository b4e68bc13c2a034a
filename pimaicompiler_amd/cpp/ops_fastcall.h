// Adds the native per-call functions of pimaicompiler_amd.ops (ops_fastcall.cpp) to the extension module.
#pragma once

#include <Python.h>

void addFastcalls(PyObject* module);
