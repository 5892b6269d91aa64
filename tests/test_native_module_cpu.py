"""The native module's ways out of a call and into a process, which need no GPU: small modules and libraries built here stand in for
what it meets."""
import importlib.machinery
import importlib.util
import os
import subprocess
import sys
import sysconfig

import pytest

from flashlight_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _module(tmp_path, name, source):
    src, lib = tmp_path / (name + ".cpp"), str(tmp_path / (name + ".so"))
    src.write_text(source)
    subprocess.check_call([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-fPIC", "-shared", "-I" + os.path.join(ROOT, "flashlight_amd", "bind"),
                           "-isystem", sysconfig.get_paths()["include"], "-o", lib, str(src)])
    loader = importlib.machinery.ExtensionFileLoader(name, lib)
    module = importlib.util.module_from_spec(importlib.util.spec_from_loader(name, loader))
    loader.exec_module(module)
    return module


def test_an_exception_out_of_a_launch_finds_the_interpreter_held(tmp_path):
    m = _module(tmp_path, "launches", r"""
#include "unlocked.h"
#include <new>
static PyObject* run(PyObject*, PyObject* fails) {
  const bool f = PyObject_IsTrue(fails);
  int inside = -1, held = -1, rc = -1;
  try {
    rc = launched([&]() -> int {
      inside = PyGILState_Check();
      if (f) throw std::bad_alloc();
      return 7;
    });
  } catch (const std::bad_alloc&) {
    rc = 8;
  }
  held = PyGILState_Check();
  if (!held) PyGILState_Ensure();
  return Py_BuildValue("iii", inside, held, rc);
}
static PyMethodDef methods[] = {{"run", run, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
static PyModuleDef module = {PyModuleDef_HEAD_INIT, "launches", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
PyMODINIT_FUNC PyInit_launches() { return PyModule_Create(&module); }
""")
    assert m.run(False) == (0, 1, 7)
    assert m.run(True) == (0, 1, 8)


_LOAD = """
import ctypes, sys
sys.path.insert(0, sys.argv[1])
if sys.argv[2]:
    ctypes.CDLL(sys.argv[2], ctypes.RTLD_GLOBAL)      # (in front of libflhip.so's)
import torch
from flashlight_amd import capi
try:
    capi.native()
    print("loaded")
except ImportError as e:
    print("refused:", e)
"""


def test_the_module_is_refused_beside_a_library_of_another_layout(tmp_path):
    def load(version):
        lib = ""
        if version:
            src, lib = tmp_path / "v.c", str(tmp_path / ("v%d.so" % version))
            src.write_text("int flhip_version(void) { return %d; }" % version)
            subprocess.check_call([os.environ.get("CC", "gcc"), "-fPIC", "-shared", "-o", lib, str(src)])
        return subprocess.run([sys.executable, "-c", _LOAD, ROOT, lib], capture_output=True, text=True, check=True).stdout.strip()

    with open(os.path.join(ROOT, "include", "flhip.h")) as f:
        own = int(next(line.split()[2] for line in f if line.startswith("#define FLHIP_VERSION")))
    assert own == capi.VERSION
    assert load(0) == load(own) == load(own // 100 * 100 + 99) == "loaded"
    for other in (own + 100, own - 100):
        assert load(other) == "refused: flhip_torch: libflhip version %d, compiled against %d" % (other, own)


def test_a_library_of_another_layout_is_refused(monkeypatch):
    for version, refused in ((capi.VERSION + 100, True), (capi.VERSION - 100, True), (capi.VERSION // 100 * 100, False)):
        monkeypatch.setattr(capi, "_lib", None)
        monkeypatch.setattr(capi, "VERSION", version)
        if refused:
            with pytest.raises(RuntimeError, match="version"):
                capi.lib()
        else:
            assert capi.lib().flhip_version() // 100 == version // 100
