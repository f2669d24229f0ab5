// The PNCG's trial pass (elem_kernel.h, W_TRIAL).
#include "elem_solve_impl.h"

namespace apl {
APL_SOLVE_PASS(W_E | W_G | W_H | W_TRIAL, float)
APL_SOLVE_PASS(W_E | W_G | W_H | W_TRIAL, double)
APL_SOLVE_PASS(W_E | W_G | W_H | W_TRIAL | W_ONE, float)
APL_SOLVE_PASS(W_E | W_G | W_H | W_TRIAL | W_ONE, double)
APL_SOLVE_PASS(W_E | W_G | W_H | W_TRIAL | W_FUSED, float)
APL_SOLVE_PASS(W_E | W_G | W_H | W_TRIAL | W_FUSED, double)
}  // namespace apl
