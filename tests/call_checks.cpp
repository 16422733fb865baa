// _call.so's own helpers behind a C name, for tests/test_native_call.py.
#include "../ffn_kernel_amd/csrc/call.cpp"

// Whether the GIL is held where an exception out of a foreign call arrives (it is held again on return, either way).
extern "C" __attribute__((visibility("default"))) int cc_gil_held_after_throw() {
  PyThreadState* const state = PyThreadState_Get();
  int held = -1;
  try {
    run("a call that throws", []() -> int { throw std::runtime_error("no data pointer"); });
  } catch (const std::runtime_error&) {
    held = PyGILState_Check();
    if (!held) PyEval_RestoreThread(state);
  }
  return held;
}
