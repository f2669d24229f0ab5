// The PNCG's step and quadratic-form pass (elem_kernel.h, W_DIR).
#include "elem_solve_impl.h"

namespace apl {
APL_SOLVE_PASS(W_HQ | W_DIR, float)
APL_SOLVE_PASS(W_HQ | W_DIR, double)
APL_SOLVE_PASS(W_HQ | W_DIR | W_ONE, float)
APL_SOLVE_PASS(W_HQ | W_DIR | W_ONE, double)
APL_SOLVE_PASS(W_HQ | W_DIR | W_FUSED, float)
APL_SOLVE_PASS(W_HQ | W_DIR | W_FUSED, double)
}  // namespace apl
