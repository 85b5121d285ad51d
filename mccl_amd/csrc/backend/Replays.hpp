// Replays.hpp -- the allreduce replays of mccl_amd/harness.py over Python lists of tensors.
#pragma once

#include <pybind11/pybind11.h>

namespace mccl {
// Adds _allreduce_replay and _allreduce_replay_many to the extension module.
void bind_replays(pybind11::module_& m);
}  // namespace mccl
