// Python module maltos_amd._torch_ops.
#include "common.hpp"

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "torch operators and autograd nodes over libmaltos_hip.so";
  maltos::bind_ops(m);
  maltos::bind_llama(m);
}
