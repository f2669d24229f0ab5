// The CG's Hessian-vector passes (elem_kernel.h, W_CGD and W_ACT).
#include "elem_solve_impl.h"

namespace apl {
APL_SOLVE_PASS(W_HP | W_VQ | W_CGD, float)
APL_SOLVE_PASS(W_HP | W_VQ | W_CGD, double)
APL_SOLVE_PASS(W_HP | W_VQ | W_CGD | W_FUSED, float)
APL_SOLVE_PASS(W_HP | W_VQ | W_CGD | W_FUSED, double)
APL_SOLVE_PASS(W_HP | W_ACT, float)
APL_SOLVE_PASS(W_HP | W_ACT, double)
}  // namespace apl
