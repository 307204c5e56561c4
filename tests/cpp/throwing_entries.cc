// Entry points that throw, called through the binding's own conversion: a module for test_native_call.py.
#include "../../hotspa-ae_amd/pybind/hk_call.cc"

#include <stdexcept>

namespace {

int throws(int what, const int64_t* list) {
  if (PyGILState_Check()) return -1;   // an entry point runs without the interpreter's lock
  if (what == 1) throw std::bad_alloc();
  if (what == 2) throw std::length_error("a list too long");
  if (what == 3) throw 3;
  return list == nullptr ? 0 : int(list[0]);
}

PyMethodDef throwing_methods[] = {ENTRY(throws), {nullptr, nullptr, 0, nullptr}};
PyModuleDef throwing_module = {PyModuleDef_HEAD_INIT, "throwing_entries", nullptr, -1, throwing_methods,
                               nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit_throwing_entries(void) { return PyModule_Create(&throwing_module); }
