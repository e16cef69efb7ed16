// lbm_tiled.hpp -- host-side interface to the several-steps-per-launch kernels in lbm_tiled.hip.
#pragma once

#include "lbm_kernels.hpp"

namespace cfd_hip {

// Whether a lattice of `nx` x `ny` D2Q9 cells can be advanced by tiled_steps.
bool tiled_supported(int q, int storage, size_t nx, size_t ny);

// `k` steps (2 or 4) of a D2Q9 lattice from src (even parity) into dst, another array of the same
// layout, asynchronously on st.stream.
void tiled_steps(int storage, const LaunchState& st, int k, bool bounded, bool forced, const void* src, void* dst);

}  // namespace cfd_hip
