// lbm_tiled.hpp -- host-side interface to the several-steps-per-launch kernels in lbm_tiled.hip.
#pragma once

#include "lbm_kernels.hpp"

namespace cfd_hip {

// Whether tiled_steps can advance a lattice of `nx` x `ny` cells (population array of `bytes` bytes) by `k`
// (2 or 4) steps a launch, faster than single steps.
bool tiled_pays(int q, int storage, size_t nx, size_t ny, size_t bytes, int k, bool bounded, bool forced);

// `k` steps (2 or 4) of a D2Q9 lattice from src (even parity) into dst, another array of the same
// layout, asynchronously on st.stream.
void tiled_steps(int storage, const LaunchState& st, int k, bool bounded, bool forced, const void* src, void* dst);

}  // namespace cfd_hip
