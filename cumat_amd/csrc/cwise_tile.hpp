// cwise_tile.hpp -- component-wise programs with transposed leaves
// (cwise_tile.hip).
#pragma once
#include "cwise_core.hpp"
#include "jit.hpp"

namespace cm {

// Returned by the generators for a program that another path has to run.
constexpr int JIT_DECLINED = 1;

// Launches the tiled kernel generated for P if it reads leaves across the
// destination's order; JIT_DECLINED otherwise.
int jit_cwise_tile(cm_ctx_t ctx, const CwProgram& P, bool wide);

}  // namespace cm
