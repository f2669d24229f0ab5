// Definitions of elem_solve.h, instantiated pass by pass in elem_pncg*.hip and
// elem_cg.hip (separate files so that they compile in parallel).
#pragma once

#include "elem_solve.h"

namespace apl {

// the solver's iterate is FP64; the CG reads the caller's displacements
template <unsigned WHAT, class R>
using pass_x = std::conditional_t<(WHAT & (W_TRIAL | W_DIR)) != 0, double, R>;

template <class Go>
static int for_laws(const apl_mesh* m, int material, Go go) {
  auto one = [&](int law) {
    if (law == MAT_SNH) return go(std::integral_constant<int, MAT_SNH>{});
    if (law == MAT_ARAP) return go(std::integral_constant<int, MAT_ARAP>{});
    return go(std::integral_constant<int, MAT_MUSCLE>{});
  };
  if (material != MAT_MODEL) return one(material);
  for (int law = 0; law < N_MAT; ++law)
    if (m->law_nblk[law] > 0 && one(law)) return -1;
  return 0;
}

template <unsigned WHAT, class R>
int launch_solve_pass(apl_mesh* m, int material, const void* mu, const void* lam, const void* x, const void* p,
                      const SolveArgs<R>& S0, int grid_override, hipStream_t s) {
  using X = pass_x<WHAT, R>;
  SolveArgs<R> S = S0;
  if (m->activation == nullptr && launch_blocks(m, MAT_MUSCLE) > 0 && (material == MAT_MUSCLE || material == MAT_MODEL)) {
    set_error("the muscle law needs the activation: call apl_mesh_set_activation first");
    return -1;
  }
  auto go = [&](auto mat_c) -> int {
    constexpr int MAT = decltype(mat_c)::value;
    if (launch_blocks(m, MAT) == 0 && S.n_iso == 0) return 0;
    const ElemArgs<R, X> A = make_args<R, X>(m, mu, lam, x, p, nullptr, nullptr, 0, nullptr, nullptr);
    if (launch_pass<MAT, WHAT, R, X>(m, A, S.filter != 0, grid_override, s, S)) return -1;
    S.n_iso = 0;  // the first launch has stepped the vertices without tets
    return 0;
  };
  if (m->L.nblocks == 0) return go(std::integral_constant<int, MAT_SNH>{});
  return for_laws(m, material, go);
}

template <unsigned WHAT, class R>
void solve_pass_grid(apl_mesh* m, int material) {
  using X = pass_x<WHAT, R>;
  (void)for_laws(m, m->L.nblocks == 0 ? (int)MAT_SNH : material, [&](auto mat_c) {
    (void)grid_for<decltype(mat_c)::value, WHAT, R, X>(m, m->L.n_inst > 1);
    return 0;
  });
}

#define APL_SOLVE_PASS(W, R)                                                                                        \
  template int launch_solve_pass<W, R>(apl_mesh*, int, const void*, const void*, const void*, const void*,          \
                                       const SolveArgs<R>&, int, hipStream_t);                                      \
  template void solve_pass_grid<W, R>(apl_mesh*, int);

}  // namespace apl
