// call.hpp - how a function of the binding runs: its answer to Python and the
// library call without the GIL.
#pragma once

#include <Python.h>

#include <exception>

namespace sqa_py {

struct General {};  // leave the call to the Python wrapper

// Runs f (descriptors, then the library call) and returns its status, or None for
// the general path. Only C++ exceptions are caught, by type: a daemon thread that
// asks for the GIL once the interpreter has begun to end is ended by pthread_exit
// there, and that unwinding passes through here; a catch (...) without a rethrow
// (or a destructor on its way) would turn it into an abort of the process.
template <class F>
PyObject *answer(F f) {
    int rc;
    try {
        rc = f();
    } catch (const General &) {
        PyErr_Clear();
        Py_RETURN_NONE;
    } catch (const std::exception &) {  // torch refusing (the wrapper meets the same and reports it)
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    return PyLong_FromLong(rc);
}

template <class F>
int without_gil(F f) {
    PyThreadState *s = PyEval_SaveThread();
    int rc;
    try {
        rc = f();
    } catch (...) {
        PyEval_RestoreThread(s);
        throw;
    }
    PyEval_RestoreThread(s);
    return rc;
}

}  // namespace sqa_py
