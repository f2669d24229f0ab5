// Per-instance state of the device solvers and the scalar decisions taken on
// it, shared by the solver's scalar kernels and its element passes.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "../../include/apple_amd.h"
#include "internal.h"

namespace apl {

enum : int { D_G2 = 0, D_GPG, D_GPG0, D_GPGC, D_GPGC0, D_GCPGC, D_GCPGC0, D_GTP, D_GCP, D_HSUM, D_HCNT, D_EXT, D_PP, D_E };
static_assert(D_E < N_DOTS, "dot table too small");
static_assert(D_PP < N_DOTS, "dot slots");

// One instance's solver state, one record per instance.  `cur` names the
// buffer of the pair (iterate, direction) that holds the committed point: an
// accepted step flips it, and the direction pass that follows writes the new
// point there from the other one, so blocks that share a vertex all read the
// old values whatever order they run in.
struct alignas(16) InstState {
  double f, gd, alpha, alpha_commit, beta, gnorm0, gnorm, pmean, f_first, pHp, gbest, f_mark, f0;
  int32_t status, act_eval, act_dir, commit, n_steps, n_evals, ls_step, n_backtracks, phase, restarts, best_step,
      ls_last, cur;
};

constexpr int STATE_DOUBLES = sizeof(InstState) / 8;

// threads whose order the sums over whole tables follow (the scalar kernels
// run with as many: each sums whole tables of per-block values, so more
// loads in flight shorten them)
constexpr int SCAL_TH = 1024;

// A single instance's scalar steps ride in the element pass that follows
// them up to these table sizes: FUSE_BLOCKS element blocks for the step length
// (and for d.Hd in the CG's update), FUSE_VBLOCKS vertex blocks of 16 columns for
// the decision, FUSE_CG_VBLOCKS of two columns for the CG's beta.  Every
// workgroup reads the whole table and the pass takes more registers, so the gain
// falls with size.  Whole iterations of SNH in FP32, us, in the pass / as a launch:
//   step length  20 blocks 19.7 / 21.3, 640 25.8 / 27.2, 2,028 42.1 / 44.0, 2,160
//                45.1 / 46.9, 4,012 64.8 / 65.2 (about the end of the short tables)
//   decision     6 vertex blocks 19.7 / 20.9, 141 25.8 / 26.9, 198 29.3 / 30.2
//   CG's beta    6 13.0 / 14.2, 141 15.9 / 17.0, 270 20.5 / 22.2, 290 23.1 / 23.1,
//                356 25.5 / 24.6, 844 37.8 / 37.1
// The first two lines keep a margin to where the gain ends.  The CG's is generous:
// from 290 vertex blocks on the launch is up to 5 % faster in FP32 (SNH FP64: the
// pass, to 460), for ARAP from about 200, and for ARAP and muscle in FP64 from
// about 100 (141: 25.8 / 23.2 and 24.6 / 22.2).
constexpr int FUSE_BLOCKS = 2048, FUSE_VBLOCKS = 192, FUSE_CG_VBLOCKS = 1024;
static_assert(FUSE_BLOCKS <= 4 * SCAL_TH && FUSE_VBLOCKS * N_DOTS <= 4 * SCAL_TH && FUSE_CG_VBLOCKS * 2 <= 4 * SCAL_TH,
              "short tables (flatsum.h)");

struct Params {
  double rtol, atol, overstep, c1, wolfe_delta, wolfe_eps, beta_max;
  int max_steps, max_backtracking, stall_steps;
};

// per-instance decision from the instance's dot totals
__device__ inline void pncg_scalar_step(InstState& s, const Params& P, const double* tot) {
  const double fE = tot[D_E];
  const double ft = fE + tot[D_EXT];
  const double gn = sqrt(tot[D_G2]);
  const int phase = s.phase;
  s.n_evals += 1;
  bool accept;
  if (phase != 1) {
    accept = true;
  } else {
    const double f0 = s.f, a = s.alpha, gd = s.gd;
    const bool fin = isfinite(ft);
    const bool armijo = fin && ft <= f0 + P.c1 * a * gd;
    const bool wolfe = P.wolfe_delta > 0.0 && fin && ft <= f0 + P.wolfe_eps * fabs(f0) &&
                       tot[D_GTP] <= (2.0 * P.wolfe_delta - 1.0) * gd;
    accept = armijo || wolfe;
  }
  if (accept) {
    s.alpha_commit = phase == 1 ? s.alpha : 0.0;
    s.f0 = phase == 0 ? ft : s.f;  // the line search's start and end energies
    s.ls_last = s.ls_step;
    s.f = ft;
    s.gnorm = gn;
    s.commit = 1;
    s.cur ^= 1;
    if (phase == 0) {
      s.gnorm0 = gn;
      s.f_first = ft;
    }
    if (phase == 1) {
      s.n_steps += 1;
      s.restarts = 0;
    }
    // progress marker: the last step that lowered the best gradient norm by
    // 10% or the energy, since the previous marker, by more than the energy
    // noise the approximate-Wolfe test tolerates (10 wolfe_eps relative)
    const bool g_prog = gn < 0.9 * s.gbest;
    const double f_tol = fmax(10.0 * P.wolfe_eps, 1e-12) * fabs(ft);
    const bool f_prog = !(s.f_mark - ft <= f_tol);
    if (g_prog) s.gbest = gn;
    if (g_prog || f_prog) {
      s.best_step = s.n_steps;
      s.f_mark = ft;
    }
    int status = APL_RUNNING;
    if (!isfinite(gn) || !isfinite(ft))
      status = APL_NON_FINITE;
    else if (gn <= P.rtol * s.gnorm0 || gn <= P.atol)
      status = APL_PRIMARY_SUCCESS;
    else if (s.n_steps >= P.max_steps)
      status = APL_MAX_STEPS_REACHED;
    else if (P.stall_steps > 0 && s.n_steps - s.best_step >= P.stall_steps && s.gbest <= 1e3 * P.rtol * s.gnorm0)
      status = APL_STAGNATION;  // within 3 decades of the target: the rounding floor of the gradient
    s.status = status;
    if (status == APL_RUNNING) {
      const double pm = tot[D_HCNT] > 0.0 ? tot[D_HSUM] / tot[D_HCNT] : 1.0;
      s.pmean = pm;
      const double gPg = tot[D_GPG] + tot[D_GPG0] / pm;
      double beta = 0.0;
      if (phase == 1) {
        const double gPgc = tot[D_GPGC] + tot[D_GPGC0] / pm;
        const double gcPgc = tot[D_GCPGC] + tot[D_GCPGC0] / pm;
        const double yp = tot[D_GTP] - tot[D_GCP];
        if (fabs(yp) > 1e-300) {
          const double gPy = gPg - gPgc;
          const double yPy = gPg - 2.0 * gPgc + gcPgc;
          beta = gPy / yp - (yPy / yp) * (tot[D_GTP] / yp);
        } else {
          beta = INFINITY;
        }
        if (!isfinite(beta) || fabs(beta) > P.beta_max) beta = 0.0;
      }
      double gd = -gPg + beta * tot[D_GTP];
      if (!(isfinite(gd) && gd < 0.0)) {
        beta = 0.0;
        gd = -gPg;
      }
      s.beta = beta;
      s.gd = gd;
      s.act_dir = 1;
    } else {
      s.act_dir = 0;
      s.act_eval = 0;
    }
    s.ls_step = 0;
    s.phase = 1;
  } else {
    s.commit = 0;
    s.act_dir = 0;
    s.ls_step += 1;
    s.n_backtracks += 1;
    const double a = s.alpha * 0.5;
    if (s.ls_step > P.max_backtracking || !(a > 0.0)) {
      if (s.restarts >= 1) {
        s.status = APL_STAGNATION;
        s.act_eval = 0;
      } else {
        // restart from x with steepest descent: re-evaluate at alpha = 0
        s.restarts += 1;
        s.phase = 2;
        s.alpha = 0.0;
        s.ls_step = 0;
      }
    } else {
      s.alpha = a;
    }
  }
}

// step length of a new direction from its quadratic form; the iteration's
// flags are cleared
__device__ inline void pncg_alpha_step(InstState& s, const Params& P, double pHp) {
  if (s.act_dir != 0) {
    s.pHp = pHp;
    double a = -s.gd / pHp;
    if (isnan(a)) a = 0.0;
    else if (a == -INFINITY) a = 0.0;
    else if (a == INFINITY) a = 1.0;
    if (!(a > 0.0 && isfinite(a))) a = 1.0;
    s.alpha = a * P.overstep;
  }
  s.commit = 0;
  s.act_dir = 0;
}

// ---- PCG (adjoint).  State reuse: gd = r.z, gnorm0 = ||b||, gnorm = ||r||,
// alpha = a, pHp = d.Hd, pmean = mean positive diagonal, f = ||r|| / ||b||,
// phase = 1 once an update has run.

// before an iteration: from the last update's r.r and r.z the residual, the
// stop tests and beta
__device__ inline void cg_beta_step(InstState& s, double rtol, int max_iters, double rr, double rz) {
  if (s.act_eval == 0) return;
  if (s.phase == 0) {
    s.phase = 1;  // the first direction is z (beta 0)
    return;
  }
  const double rn = sqrt(rr);
  s.gnorm = rn;
  s.n_steps += 1;
  s.f = s.gnorm0 > 0.0 ? rn / s.gnorm0 : 0.0;
  if (rn <= rtol * s.gnorm0) {
    s.status = APL_PRIMARY_SUCCESS;
    s.act_eval = 0;
  } else if (!isfinite(rn)) {
    s.status = APL_NON_FINITE;
    s.act_eval = 0;
  } else if (s.n_steps >= max_iters) {
    s.status = APL_MAX_STEPS_REACHED;
    s.act_eval = 0;
  } else {
    s.beta = rz / s.gd;
    s.gd = rz;
    s.cur ^= 1;  // the next direction is formed in the other buffer
  }
}

// after the Hessian-vector pass: the step from d.Hd
__device__ inline void cg_alpha_step(InstState& s, double dq) {
  if (s.act_eval == 0) return;
  s.pHp = dq;
  if (!(dq > 0.0) || !isfinite(dq)) {
    s.status = APL_NON_FINITE;
    s.act_eval = 0;
    s.alpha = 0.0;
  } else {
    s.alpha = s.gd / dq;
  }
}

}  // namespace apl
