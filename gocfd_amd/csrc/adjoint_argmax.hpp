// Ranking of the face points whose speeds bound the time step, shared by the
// kernels that form the speeds and the one that closes the maximum.
#pragma once

#include <hip/hip_runtime.h>

#include "dual.hpp"

namespace gocfd {
namespace dev {

__device__ __forceinline__ double val_of(double a) { return a; }
__device__ __forceinline__ double val_of(const ad::Dual &a) { return a.v; }

// The largest speed, ties to the smallest index (a deterministic choice of the
// point the dt follows); bi < 0: none yet
__device__ __forceinline__ bool ranks_before(double v, int i, double bv, int bi) {
  return v > bv || (v == bv && i >= 0 && (bi < 0 || i < bi));
}

}  // namespace dev
}  // namespace gocfd
