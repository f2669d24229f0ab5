// Launches of the solvers' element passes (elem_kernel.h, W_SOLVER modes).
#pragma once

#include "elem_kernel.h"

namespace apl {

// WHAT: W_E | W_G | W_H | W_TRIAL, W_HQ | W_DIR (x unused: the solver's own
// iterate), W_HP | W_VQ | W_CGD, W_HP | W_ACT (x the caller's displacements, p
// the direction of W_ACT); the first three also with W_FUSED.  Every law of a model mesh, each over its own blocks.
template <unsigned WHAT, class R>
int launch_solve_pass(apl_mesh* m, int material, const void* mu, const void* lam, const void* x, const void* p,
                      const SolveArgs<R>& S, int grid_override, hipStream_t s);
// query (and cache) the pass's persistent grid, outside any capture
template <unsigned WHAT, class R>
void solve_pass_grid(apl_mesh* m, int material);

}  // namespace apl
