// A call during which other threads run Python.
#pragma once
#include <Python.h>

// f's result, the interpreter's lock given up meanwhile and held again however f ends: an exception's handler makes a Python error of it
template <typename F>
int launched(F f) {
  struct Unlocked {
    PyThreadState* const state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
  } unlocked;
  return f();
}
