"""A daemon thread inside a native call when the interpreter ends: it is ended at the
GIL, and the process exits as with a ctypes call (no GPU: the call is a sleep)."""
import os
import subprocess
import sys
import sysconfig

SOURCE = r"""
#include <Python.h>
#include <unistd.h>
#include "call.hpp"
static PyObject *nap(PyObject *, PyObject *const *, Py_ssize_t) {
    return sqa_py::answer([] { return sqa_py::without_gil([] { usleep(300000); return 0; }); });
}
static PyMethodDef methods[] = {{"nap", (PyCFunction)(void (*)(void))nap, METH_FASTCALL, nullptr},
                                {nullptr, nullptr, 0, nullptr}};
static PyModuleDef module = {PyModuleDef_HEAD_INIT, "napping", nullptr, -1, methods};
PyMODINIT_FUNC PyInit_napping() { return PyModule_Create(&module); }
"""

# sys.keep outlives the start of finalization and holds it up until the thread wakes
PROGRAM = """
import sys, threading, time
import napping
assert napping.nap() == 0
threading.Thread(target=lambda: napping.nap(), daemon=True).start()
time.sleep(0.05)
class Keep:
    def __del__(self, sleep=time.sleep):
        sleep(0.6)
sys.keep = Keep()
"""


def test_daemon_thread_in_a_call_at_exit(tmp_path):
    import __graft_entry__ as ge

    src = tmp_path / "napping.cpp"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", f"-I{sysconfig.get_paths()['include']}",
                    f"-I{os.path.join(ge.PKG_DIR, 'binding')}", str(src), "-o", str(tmp_path / "napping.so")], check=True)
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=tmp_path, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
