// Device-resident PNCG static solver and PCG adjoint solver.
//
// PNCG restates the loop of liblaf-peach as apple states it in
// benches/bench_pncg_branching_backends.py:254-330,393-456,606-679 (the
// external peach package itself is not vendored): Jacobi preconditioner
// P = 1/|diag H| with the mean of the positive entries for zeros, Dai-Kou
// beta reset when non-finite or |beta| > beta_max, steepest-descent fallback
// when g.p >= 0, alpha = -g.p / p^T H p (x overstep), halving backtracking,
// stop at ||g|| <= rtol ||g_0|| (or atol).  The sufficient-decrease test is
// Armijo OR the approximate Wolfe conditions of Hager & Zhang (2005): energy
// differences stop resolving the decrease long before ||g|| reaches 1e-6
// relative in FP32, the directional-derivative test does not.
//
// One iteration, all with device-side control (no host sync):
//   S2 per-instance: alpha = -gd / pHp
//   A  element pass at the trial point x + alpha p: energy, gradient, Hdiag
//   R  vertex pass: sums of shared-vertex partials, masks, FP64 partial dots
//   S  per-instance scalar step: energy/dot totals, accept/reject, beta, gd
//   B  element pass: the step x += alpha p, p = -P g + beta p formed while the
//      blocks stage their vertices, and p^T H p (clamped per tet)
// S2 and S are taken by A's and B's own workgroups for a single instance
// whose tables are small (FUSE_BLOCKS, FUSE_VBLOCKS), else they are launches.
// A rejected trial skips B/S2 work (flags) and the next A re-evaluates at
// the halved step.  K iterations are captured in one HIP graph; the host
// checks the per-instance status once per graph launch.  Every instance of a
// batch runs in the same launches; finished instances drop out via flags.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../../include/apple_amd.h"
#include "elem_solve.h"
#include "internal.h"
#include "flatsum.h"
#include "lanes.h"
#include "solve_state.h"
#include "persist.h"
#include "vsum.h"
#include "tetmath.h"

namespace apl {

// Workgroup sums of the 16 per-thread dots, in a fixed order, to out[0..16).
// Recursive halving across the wave (offsets 32, 16, 8, 4: each lane keeps
// half of its entries and adds its partner's copy of them) leaves dot
// lane / 4 in lanes 4j..4j+3; two more exchanges complete those sums, and
// the waves are added in order.  17 exchanges instead of 16 x 6.
__device__ inline void block_dots(double (&v)[N_DOTS], double* sm, double* out) {
  static_assert(N_DOTS == 16, "halving tree is written for 16 dots");
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = swap_add<32>(v[k], v[k + 8]);
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = swap_add<16>(v[k], v[k + 4]);
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const bool up = (lane & 8) != 0;
    v[k] = (up ? v[k + 2] : v[k]) + xor_lane<8>(up ? v[k] : v[k + 2]);
  }
  {
    const bool up = (lane & 4) != 0;
    v[0] = (up ? v[1] : v[0]) + xor_lane<4>(up ? v[0] : v[1]);
  }
  v[0] = add_xor<1>(add_xor<2>(v[0]));
  if ((lane & 3) == 0) sm[w * N_DOTS + (lane >> 2)] = v[0];
  __syncthreads();
  if ((int)threadIdx.x < N_DOTS) {
    double s = 0.0;
#pragma unroll
    for (int ww = 0; ww < NTH / 64; ++ww) s += sm[ww * N_DOTS + threadIdx.x];
    out[threadIdx.x] = s;
  }
}

// This vertex block's share of its instance's element-block energies: the
// instance's blocks split into equal consecutive runs, one per vertex block
// (both counted from the instance's start, so a batch sums the same way as
// the instance alone).
__device__ inline double energy_share(const double* blk_red, long long b0, long long nb, long long nvb, long long vb) {
  const long long per = (nb + nvb - 1) / nvb;
  const long long lo = b0 + vb * per;
  const long long hi = lo + per < b0 + nb ? lo + per : b0 + nb;
  double acc = 0.0;
  for (long long b = lo + threadIdx.x; b < hi; b += NTH) acc += blk_red[RED_STRIDE * b];
  return acc;
}

// Persistent loop of a vector kernel over its vertex blocks blockIdx.x +
// j gridDim.x (compacted to the active ones in a batch).
template <class IsActive, class Body>
__device__ inline void vertex_blocks(int nvblk, bool filter, int* list, IsActive is_active, Body body) {
  const int b0 = blockIdx.x, G = gridDim.x;
  const int n_cand = b0 < nvblk ? (nvblk - b0 + G - 1) / G : 0;
  for_active<NTH>(n_cand, filter, list, [&](int j) { return b0 + j * G; }, is_active, body);
}

template <class R>
struct VecArgs {
  const int32_t* vblk_off;
  const int32_t* vblk_inst;
  const int32_t* vtx_slot_off;
  const R* partial;
  const uint8_t* mask;
  const R* fext;
  // padded records of the vertices, as in SolveArgs
  const Vec4<double>* x;
  const Vec4<R>* p;
  Vec4<R>* g;
  Vec4<R>* P;
  double* vblk_dots;
  const double* blk_red;          // per element block: energy, quadratic form
  const int64_t* inst_blk_off;
  const int64_t* inst_vblk_off;
  const InstState* st;
  size_t V;  // vertices: the pairs' second buffers start here
  int nvblk;   // vertex blocks of the mesh
  int nblocks;  // element blocks of the mesh
};

template <class R>
__global__ __launch_bounds__(NTH) void fill_kernel(R* a, long long n, R v) {
  for (long long i = (long long)blockIdx.x * NTH + threadIdx.x; i < n; i += (long long)gridDim.x * NTH) a[i] = v;
}

// both copies of the states
__global__ void solve_init_kernel(InstState* st, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 2 * n) return;
  InstState s{};
  s.pmean = 1.0;
  s.gbest = INFINITY;
  s.f_mark = INFINITY;
  s.status = APL_RUNNING;
  s.act_eval = 1;
  st[i] = s;
}

// the committed iterate of every instance (the current buffer) into out
template <class R>
__global__ __launch_bounds__(NTH) void iterate_kernel(const InstState* st, const int32_t* vblk_off,
                                                      const int32_t* vblk_inst, const Vec4<double>* x, size_t V,
                                                      R* out) {
  const int vb = blockIdx.x;
  const Vec4<double>* src = x + (st[vblk_inst[vb]].cur ? V : (size_t)0);
  for (int i = 3 * vblk_off[vb] + (int)threadIdx.x; i < 3 * vblk_off[vb + 1]; i += NTH) out[i] = (R)src[i / 3].v[i % 3];
}

// the caller's start into the first iterate buffer
template <class R>
__global__ __launch_bounds__(NTH) void start_kernel(const R* src, Vec4<double>* x, long long n) {
  for (long long i = (long long)blockIdx.x * NTH + threadIdx.x; i < n; i += (long long)gridDim.x * NTH)
    x[i] = Vec4<double>{{(double)src[3 * i], (double)src[3 * i + 1], (double)src[3 * i + 2], 0.0}};
}

// per slot: its vertex, with OWNER_BIT where it is the first of the vertex's partials
__global__ __launch_bounds__(NTH) void owner_kernel(const int32_t* loc_gid, const int32_t* loc_dst,
                                                    const int32_t* vtx_slot_off, long long n, uint32_t* own) {
  for (long long k = (long long)blockIdx.x * NTH + threadIdx.x; k < n; k += (long long)gridDim.x * NTH) {
    const int v = loc_gid[k];
    own[k] = (uint32_t)v | (loc_dst[k] == vtx_slot_off[v] ? OWNER_BIT : 0u);
  }
}

// vertices without a slot (no tet touches them): counted, and listed when
// there is a list (its order does not matter: each is stepped by itself)
__global__ __launch_bounds__(NTH) void isolated_kernel(const int32_t* vblk_off, const int32_t* vblk_inst,
                                                       const int32_t* vtx_slot_off, int* count, int32_t* list,
                                                       int32_t* inst) {
  const int vb = blockIdx.x;
  for (int v = vblk_off[vb] + (int)threadIdx.x; v < vblk_off[vb + 1]; v += NTH)
    if (vtx_slot_off[v] == vtx_slot_off[v + 1]) {
      const int k = atomicAdd(count, 1);
      if (list != nullptr) {
        list[k] = v;
        inst[k] = vblk_inst[vb];
      }
    }
}

// R: vertex sums of the slot partials + FP64 partial dots of one vertex
// block (one DOF per thread and stride, coalesced), plus the block's share of
// the instance's element-block energies.  What bounds it is the chain of
// dependent loads: offsets -> partials -> sums -> dots, with the states and
// the vertex records beside it; every load is started before the first wait
// of that chain, and the lane exchanges of the dots stay in the VALU.  Per
// launch 7.4 -> 5.9 us at 10^3 cubes, 8.2 -> 6.5 us at 32^3; at 64^3 (49 MB)
// 13.3 us as before.  SINGLE (one instance): the block's vertices, its
// instance and its share of the energies follow from its number, so the chain
// has no table look-ups before the offsets.  Five waves per SIMD (96 VGPRs)
// keep the 64^3 mesh's 1,073 workgroups in one round.
template <class R, bool SINGLE>
__device__ inline void pncg_reduce_block(const VecArgs<R>& A, const int vb, double* sm, R* win) {
  const int inst = SINGLE ? 0 : A.vblk_inst[vb];
  const InstState& st = A.st[inst];
  const int v0 = SINGLE ? vb * NTH : A.vblk_off[vb];
  const int v1 = SINGLE ? min(v0 + NTH, (int)A.V) : A.vblk_off[vb + 1];
  const int i0 = 3 * v0, i1 = 3 * v1;
  // the partials' window first (its loads start a chain), then the energies
  // and the records, which are needed last
  VertexSums<R, 6, NTH> vs{A.vtx_slot_off, A.partial, win};
  typename VertexSums<R, 6, NTH>::template Window<12> w;
  vs.fetch(v0, v1, VSUM_LDS_BYTES / (int)sizeof(R), w);
  int k0[DOF_PER_THREAD], k1[DOF_PER_THREAD];
#pragma unroll
  for (int j = 0; j < DOF_PER_THREAD; ++j) {
    const int i = i0 + (int)threadIdx.x + j * NTH;
    k0[j] = k1[j] = 0;
    if (i < i1) {
      k0[j] = A.vtx_slot_off[i / 3];
      k1[j] = A.vtx_slot_off[i / 3 + 1];
    }
  }
  double e_share;
  if constexpr (SINGLE) {
    e_share = energy_share(A.blk_red, 0, A.nblocks, A.nvblk, vb);
  } else {
    const long long b0 = A.inst_blk_off[inst], vb0 = A.inst_vblk_off[inst];
    e_share = energy_share(A.blk_red, b0, A.inst_blk_off[inst + 1] - b0, A.inst_vblk_off[inst + 1] - vb0, vb - vb0);
  }
  if (SINGLE && st.act_eval == 0) return;  // (batches visit active instances only)
  const double alpha = st.alpha;
  // the committed point's buffers, and where the trial's gradient goes
  const Vec4<double>* x = A.x + (st.cur ? A.V : (size_t)0);
  const Vec4<R>* p = A.p + (st.cur ? A.V : (size_t)0);
  const Vec4<R>* gc0 = A.g + (st.cur ? A.V : (size_t)0);
  Vec4<R>* gt1 = A.g + (st.cur ? (size_t)0 : A.V);
  double xv[DOF_PER_THREAD];
  R pv[DOF_PER_THREAD], gcv[DOF_PER_THREAD], fv[DOF_PER_THREAD];
  unsigned mv[DOF_PER_THREAD];
#pragma unroll
  for (int j = 0; j < DOF_PER_THREAD; ++j) {
    const int i = i0 + (int)threadIdx.x + j * NTH;
    xv[j] = 0.0;
    pv[j] = gcv[j] = fv[j] = R(0);
    mv[j] = 0u;
    if (i < i1) {
      const int v = i / 3, c = i - 3 * v;
      xv[j] = x[v].v[c];
      pv[j] = p[v].v[c];
      gcv[j] = gc0[v].v[c];
      if (A.fext != nullptr) fv[j] = A.fext[i];
      if (A.mask != nullptr) mv[j] = A.mask[v];
    }
  }
  vs.store(w);
  double d[N_DOTS];
#pragma unroll
  for (int k = 0; k < N_DOTS; ++k) d[k] = 0.0;
#pragma unroll
  for (int j = 0; j < DOF_PER_THREAD; ++j) {
    const int i = i0 + (int)threadIdx.x + j * NTH;
    if (i >= i1) continue;
    R gh[2];
    const int v = i / 3, c = i - 3 * v;
    vs.sum_dof(k0[j], k1[j], c, gh);
    const double pc = (double)pv[j];
    d[D_EXT] -= (double)fv[j] * (xv[j] + alpha * pc);
    const bool fixed = ((mv[j] >> c) & 1u) != 0;
    const R h = gh[1], gf = fixed ? R(0) : gh[0] - fv[j];
    const R P1 = fixed ? R(0) : (h > R(0) ? R(1) / h : R(-1));
    gt1[v].v[c] = gf;
    A.P[v].v[c] = P1;
    if (fixed) continue;
    const double gt = (double)gf;
    const double gc = (double)gcv[j];
    d[D_G2] += gt * gt;
    if (h > R(0)) {
      const double P = (double)P1;  // the preconditioner the direction update uses
      d[D_GPG] += gt * gt * P;
      d[D_GPGC] += gt * gc * P;
      d[D_GCPGC] += gc * gc * P;
      d[D_HSUM] += (double)h;
      d[D_HCNT] += 1.0;
    } else {
      d[D_GPG0] += gt * gt;
      d[D_GPGC0] += gt * gc;
      d[D_GCPGC0] += gc * gc;
    }
    d[D_GTP] += gt * pc;
    d[D_GCP] += gc * pc;
    d[D_PP] += pc * pc;
  }
  d[D_E] = e_share;
  block_dots(d, sm, A.vblk_dots + (long long)vb * N_DOTS);
}

template <class R, bool SINGLE>
__global__ __launch_bounds__(NTH, sizeof(R) == 4 ? 5 : 4) void pncg_reduce_kernel(VecArgs<R> A) {
  __shared__ double sm[(NTH / 64) * N_DOTS];
  __shared__ R win[VSUM_LDS_BYTES / sizeof(R)];
  __shared__ int list[SINGLE ? 1 : NTH];
  vertex_blocks(A.nvblk, !SINGLE, list, [&](int vb) { return A.st[A.vblk_inst[vb]].act_eval != 0; },
                [&](int vb) { pncg_reduce_block<R, SINGLE>(A, vb, sm, win); });
}

// S: per-instance decision, one workgroup per instance, from the states `in`
// to `out`
__global__ __launch_bounds__(SCAL_TH) void pncg_scalar_kernel(const InstState* in, InstState* out, Params P,
                                                          const double* vblk_dots, const int64_t* inst_vblk_off) {
  __shared__ double tot[(SCAL_TH / 64 + 1) * N_DOTS];
  const int i = blockIdx.x;
  // the active flag, the table bounds and the state are independent: all are
  // loaded before the first wait (an inactive instance sums an empty table)
  const bool act = in[i].act_eval != 0;
  const long long vb0 = inst_vblk_off[i], vb1 = inst_vblk_off[i + 1];
  InstState s;
  if (threadIdx.x == 0) s = in[i];
  flat_column_sums<N_DOTS, SCAL_TH>(vblk_dots + vb0 * N_DOTS, act ? (vb1 - vb0) * N_DOTS : 0, tot);
  if (threadIdx.x != 0) return;
  if (act) pncg_scalar_step(s, P, tot);
  out[i] = s;
}

// An instance's state on its way through a scalar kernel: into LDS (one double
// per thread, stored before the sums, whose barriers publish it), and out again
// after thread 0's step.  As a local of thread 0 that only the step touches it
// was given to every thread, in scratch and 49 KB of LDS: the alpha kernel of
// 256 instances took 17 us instead of 4.5.
__device__ __forceinline__ void state_in(const InstState* in, InstState* lds) {
  const int t = threadIdx.x;
  if (t < STATE_DOUBLES) reinterpret_cast<double*>(lds)[t] = reinterpret_cast<const double*>(in)[t];
}
template <class Step>
__device__ __forceinline__ void state_out(InstState* lds, InstState* out, Step step) {
  const int t = threadIdx.x;
  if (t == 0) step(*lds);
  __syncthreads();
  if (t < STATE_DOUBLES) reinterpret_cast<double*>(out)[t] = reinterpret_cast<const double*>(lds)[t];
}

// S2: alpha from the quadratic form; clears the per-iteration flags
__global__ __launch_bounds__(SCAL_TH) void pncg_alpha_kernel(const InstState* in, InstState* out, Params P,
                                                         const double* hq, const int64_t* inst_blk_off) {
  __shared__ double red[SCAL_TH / 64];
  const int i = blockIdx.x;
  // all loads issued before the first wait, as in pncg_scalar_kernel
  __shared__ InstState s;
  const bool dir = in[i].act_dir != 0;
  const long long b0 = inst_blk_off[i], b1 = inst_blk_off[i + 1];
  state_in(in + i, &s);
  const double q = flat_sum_odd<SCAL_TH>(hq + b0, dir ? b1 - b0 : 0, red);
  state_out(&s, out + i, [&](InstState& st) { pncg_alpha_step(st, P, q); });
}

// ------------------------------------------------------------------ PCG (adjoint)
//
// One iteration is two launches (four for batches and meshes with long
// tables, whose scalar steps are launches of their own):
//   H  element pass: beta from the last update's dots (cg_beta_step), the
//      direction d = z + beta d formed while the blocks stage their vertices,
//      H d into the slot partials, and d.Hd per block
//   U  vertex pass: the step from d.Hd (cg_alpha_step), q = H d summed from
//      the partials, y += a d, r -= a q, z = r / diag, the dots r.r and r.z
// d.Hd is summed over the tets (products and sums in FP64, as over the DOFs)
// rather than from q, which would need a vertex pass and a launch of its own
// between H and U.  An iteration of
// a 32^3 cube takes 15.8 us (H 9.6, U 5.6; launches 1.6 us each), in five
// launches it took 28.

template <class R>
struct CgArgs {
  const int32_t* vblk_off;
  const int32_t* vblk_inst;
  const int32_t* vtx_slot_off;
  const R* partial;
  const uint8_t* mask;
  const R* rhs;
  R* y;
  R* r;
  Vec4<R>* z;  // padded records, as in SolveArgs
  Vec4<R>* d;  // two buffers (InstState::cur)
  R* hd;
  R* t;     // normal equations: H d (or the masked right-hand side while it is formed)
  R* tout;  // CG_T / CG_MASKCOPY output
  double* vblk_dots;  // the initial stages' table, then the update's (2 columns)
  double* t_dots;     // normal equations: t.t per vertex block
  const InstState* in;  // the states a stage reads (U with FUSED: before its scalar step)
  InstState* out;       // U with FUSED: where workgroup 0 keeps those after it
  const double* hq;     // U with FUSED: d.Hd per element block
  size_t V;
  int nvblk;    // vertex blocks of the mesh
  int nblocks;  // element blocks of the mesh
  int normal;   // CG on the normal equations H^2 y = H b, Jacobi with diag(H)^2
};

// Sums over the workgroup of N per-thread values, to out[0..N): a DPP tree per
// wave, the waves in order.  sm: NTH / 64 * N doubles.
template <int N>
__device__ inline void block_sums(const double (&v)[N], double* sm, double* out) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const double s = wave_sum(v[k]);
    if (lane == 63) sm[w * N + k] = s;
  }
  __syncthreads();
  if ((int)threadIdx.x < N) {
    double s = 0.0;
#pragma unroll
    for (int ww = 0; ww < NTH / 64; ++ww) s += sm[ww * N + threadIdx.x];
    out[threadIdx.x] = s;
  }
}

// Stages before the iterations, and of the normal equations:
// CG_DIAG: diag H from its partials, r = b, y = 0, both direction buffers 0
// CG_PRECOND: z = r / diag
// CG_T: tout = H v summed from the partials, fixed DOFs 0, and tout.tout
// CG_MASKCOPY: tout = rhs with fixed DOFs 0
enum CgStage : int { CG_DIAG = 0, CG_PRECOND = 1, CG_T = 2, CG_MASKCOPY = 3 };

template <class R, int STAGE>
__device__ inline void cg_vec_block(const CgArgs<R>& A, const int vb, double* sm, R* win) {
  constexpr bool SUMS = STAGE == CG_DIAG || STAGE == CG_T;
  const InstState& st = A.in[A.vblk_inst[vb]];
  if (STAGE == CG_T && st.act_eval == 0) return;
  const int v0 = A.vblk_off[vb], v1 = A.vblk_off[vb + 1];
  const int i0 = 3 * v0, i1 = 3 * v1;
  VertexSums<R, 3, NTH> vs{A.vtx_slot_off, A.partial, win};
  if constexpr (SUMS) vs.stage(v0, v1, VSUM_LDS_BYTES / (int)sizeof(R));
  double d3[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < DOF_PER_THREAD; ++j) {
    const int i = i0 + (int)threadIdx.x + j * NTH;
    if (i >= i1) continue;
    const int v = i / 3, c = i - 3 * v;
    const bool fixed = A.mask != nullptr && ((A.mask[v] >> c) & 1u) != 0;
    R s1[1];
    if constexpr (SUMS) vs.sum_dof(A.vtx_slot_off[v], A.vtx_slot_off[v + 1], c, s1);
    if constexpr (STAGE == CG_DIAG) {
      A.hd[i] = s1[0];
      const R b = fixed ? R(0) : A.rhs[i];
      A.r[i] = b;
      A.y[i] = R(0);
      A.d[v].v[c] = R(0);
      A.d[A.V + v].v[c] = R(0);
      if (!fixed) {
        d3[0] += (double)b * (double)b;
        if (s1[0] > R(0)) {
          d3[1] += (double)s1[0];
          d3[2] += 1.0;
        }
      }
    } else if constexpr (STAGE == CG_T) {
      const R t = fixed ? R(0) : s1[0];
      A.tout[i] = t;
      d3[0] += (double)t * (double)t;
    } else if constexpr (STAGE == CG_MASKCOPY) {
      A.tout[i] = fixed ? R(0) : A.rhs[i];
    } else {
      const R rv = A.r[i], h = A.hd[i];
      const R hh = h > R(0) ? h : (R)st.pmean;
      const R zv = fixed ? R(0) : (A.normal ? rv / (hh * hh) : rv / hh);
      A.z[v].v[c] = zv;
      d3[0] += (double)rv * (double)zv;
    }
  }
  if constexpr (STAGE == CG_T) {
    const double one[1] = {d3[0]};
    block_sums<1>(one, sm, A.t_dots + vb);
  } else if constexpr (STAGE != CG_MASKCOPY) {
    // (rows of 16 columns, summed by cg_scalar_kernel)
    block_sums<3>(d3, sm, A.vblk_dots + (long long)vb * N_DOTS);
  }
  __syncthreads();
}

template <class R, int STAGE>
__global__ __launch_bounds__(NTH) void cg_vec_kernel(CgArgs<R> A) {
  __shared__ double sm[(NTH / 64) * 3];
  constexpr bool SUMS = STAGE == CG_DIAG || STAGE == CG_T;
  __shared__ R win[SUMS ? VSUM_LDS_BYTES / sizeof(R) : 1];
  for (int vb = blockIdx.x; vb < A.nvblk; vb += gridDim.x) cg_vec_block<R, STAGE>(A, vb, sm, win);
}

// the scalars of the initial stages, one workgroup per instance: 0 after
// CG_DIAG, 1 after CG_PRECOND
__global__ __launch_bounds__(SCAL_TH) void cg_scalar_kernel(InstState* st, int stage, const double* vblk_dots,
                                                        const int64_t* inst_vblk_off) {
  __shared__ double tot[(SCAL_TH / 64 + 1) * N_DOTS];
  const int i = blockIdx.x;
  const long long vb0 = inst_vblk_off[i], vb1 = inst_vblk_off[i + 1];
  flat_column_sums<N_DOTS, SCAL_TH>(vblk_dots + vb0 * N_DOTS, (vb1 - vb0) * N_DOTS, tot);
  if (threadIdx.x != 0) return;
  InstState s = st[i];
  if (stage == 0) {
    s.pmean = tot[2] > 0.0 ? tot[1] / tot[2] : 1.0;
    const double bn = sqrt(tot[0]);
    s.gnorm0 = bn;
    s.gnorm = bn;
    s.n_steps = 0;
    s.f = bn > 0.0 ? 1.0 : 0.0;
    s.status = bn > 0.0 ? APL_RUNNING : APL_PRIMARY_SUCCESS;
    s.act_eval = bn > 0.0 ? 1 : 0;
    s.alpha = 0.0;
    s.beta = 0.0;
  } else {
    s.gd = tot[0];
  }
  st[i] = s;
}

// the iteration's scalar steps as launches, one workgroup per instance
__global__ __launch_bounds__(SCAL_TH) void cg_beta_kernel(const InstState* in, InstState* out, double rtol, int max_iters,
                                                      const double* dots, const int64_t* inst_vblk_off) {
  __shared__ double tot[(SCAL_TH / 64 + 1) * 2];
  const int i = blockIdx.x;
  // all loads issued before the first wait, as in pncg_scalar_kernel
  const bool act = in[i].act_eval != 0;
  const long long vb0 = inst_vblk_off[i], vb1 = inst_vblk_off[i + 1];
  __shared__ InstState s;
  state_in(in + i, &s);
  flat_column_sums<2, SCAL_TH>(dots + 2 * vb0, act ? 2 * (vb1 - vb0) : 0, tot);
  state_out(&s, out + i, [&](InstState& st) { cg_beta_step(st, rtol, max_iters, tot[0], tot[1]); });
}

__global__ __launch_bounds__(SCAL_TH) void cg_alpha_kernel(const InstState* in, InstState* out, const double* table,
                                                       const int64_t* inst_off) {
  __shared__ double red[SCAL_TH / 64];
  const int i = blockIdx.x;
  const bool act = in[i].act_eval != 0;
  const long long b0 = inst_off[i], b1 = inst_off[i + 1];
  __shared__ InstState s;
  state_in(in + i, &s);
  const double dq = flat_sum_odd<SCAL_TH>(table + b0, act ? b1 - b0 : 0, red);
  state_out(&s, out + i, [&](InstState& st) { cg_alpha_step(st, dq); });
}

// U of one vertex block, with the instance's step a and buffer
template <class R, bool SINGLE>
__device__ inline void cg_update_block(const CgArgs<R>& A, const int vb, double* sm, R* win, const R a, const R pm,
                                       const int cur) {
  const int v0 = SINGLE ? vb * NTH : A.vblk_off[vb];
  const int v1 = SINGLE ? min(v0 + NTH, (int)A.V) : A.vblk_off[vb + 1];
  const int i0 = 3 * v0, i1 = 3 * v1;
  const Vec4<R>* d = A.d + (cur ? A.V : (size_t)0);
  // as in pncg_reduce_block: every load before the first wait
  VertexSums<R, 3, NTH> vs{A.vtx_slot_off, A.partial, win};
  typename VertexSums<R, 3, NTH>::template Window<8> w;
  vs.fetch(v0, v1, VSUM_LDS_BYTES / (int)sizeof(R), w);
  int k0[DOF_PER_THREAD], k1[DOF_PER_THREAD];
  R dv[DOF_PER_THREAD], yv[DOF_PER_THREAD], rv[DOF_PER_THREAD], hv[DOF_PER_THREAD];
  unsigned mv[DOF_PER_THREAD];
#pragma unroll
  for (int j = 0; j < DOF_PER_THREAD; ++j) {
    const int i = i0 + (int)threadIdx.x + j * NTH;
    k0[j] = k1[j] = 0;
    dv[j] = yv[j] = rv[j] = hv[j] = R(0);
    mv[j] = 0u;
    if (i < i1) {
      const int v = i / 3, c = i - 3 * v;
      k0[j] = A.vtx_slot_off[v];
      k1[j] = A.vtx_slot_off[v + 1];
      dv[j] = d[v].v[c];
      yv[j] = A.y[i];
      rv[j] = A.r[i];
      hv[j] = A.hd[i];
      if (A.mask != nullptr) mv[j] = A.mask[v];
    }
  }
  vs.store(w);
  double dots[2] = {0.0, 0.0};
#pragma unroll
  for (int j = 0; j < DOF_PER_THREAD; ++j) {
    const int i = i0 + (int)threadIdx.x + j * NTH;
    if (i >= i1) continue;
    const int v = i / 3, c = i - 3 * v;
    const bool fixed = ((mv[j] >> c) & 1u) != 0;
    R s1[1];
    vs.sum_dof(k0[j], k1[j], c, s1);
    A.y[i] = yv[j] + a * dv[j];
    const R r = rv[j] - a * (fixed ? R(0) : s1[0]);
    A.r[i] = r;
    // Jacobi: 1/diag(H), or 1/diag(H)^2 for the normal equations (diag(H^2) >= diag(H)^2)
    const R hh = hv[j] > R(0) ? hv[j] : pm;
    const R z = fixed ? R(0) : (A.normal ? r / (hh * hh) : r / hh);
    A.z[v].v[c] = z;
    dots[0] += (double)r * (double)r;
    dots[1] += (double)r * (double)z;
  }
  block_sums<2>(dots, sm, A.vblk_dots + 2 * (long long)vb);
}

// MODE: a batch, a single instance whose scalar step was a launch, or one
// whose workgroups take the step themselves (FUSE_BLOCKS)
enum UpdateMode : int { U_BATCH = 0, U_SINGLE = 1, U_FUSED = 2 };

template <class R, int MODE>
__global__ __launch_bounds__(NTH) void cg_update_kernel(CgArgs<R> A) {
  __shared__ double sm[(NTH / 64) * 2];
  __shared__ R win[VSUM_LDS_BYTES / sizeof(R)];
  if constexpr (MODE == U_BATCH) {
    __shared__ int list[NTH];
    vertex_blocks(A.nvblk, true, list, [&](int vb) { return A.in[A.vblk_inst[vb]].act_eval != 0; }, [&](int vb) {
      const InstState& st = A.in[A.vblk_inst[vb]];
      cg_update_block<R, false>(A, vb, sm, win, (R)st.alpha, (R)st.pmean, st.cur);
      __syncthreads();
    });
  } else {
    __shared__ InstState st;
    const int t = threadIdx.x;
    if (t < STATE_DOUBLES) reinterpret_cast<double*>(&st)[t] = reinterpret_cast<const double*>(A.in)[t];
    if constexpr (MODE == U_FUSED) {
      __shared__ double red[SCAL_TH / 64];
      const double dq = flat_sum_odd_short<SCAL_TH, NTH>(A.hq, A.nblocks, red);
      if (t == 0) {
        InstState s = st;
        cg_alpha_step(s, dq);
        st = s;
      }
    }
    __syncthreads();
    if (MODE == U_FUSED && blockIdx.x == 0 && t < STATE_DOUBLES)
      reinterpret_cast<double*>(A.out)[t] = reinterpret_cast<double*>(&st)[t];
    if (st.act_eval == 0) return;
    for (int vb = blockIdx.x; vb < A.nvblk; vb += gridDim.x) {
      cg_update_block<R, true>(A, vb, sm, win, (R)st.alpha, (R)st.pmean, st.cur);
      __syncthreads();
    }
  }
}

}  // namespace apl

using namespace apl;

struct apl_solver {
  apl_mesh* mesh = nullptr;  // holds one reference of the mesh
  int device = 0;
  int material = 0;
  void* mem = nullptr;     // one allocation for everything on the device
  Vec4<double>* x = nullptr;  // PNCG iterate: two buffers of V
  void* p = nullptr;       // PNCG direction: two buffers of V records of the mesh dtype
  void* g = nullptr;       // gradient: two buffers of V records, then the preconditioner (V records)
  void* cg = nullptr;      // CG: z (V records), d (two buffers of V records)
  void* vecs = nullptr;    // CG: r, hd, t, b (N_VECS x V x 3)
  uint32_t* own = nullptr;  // per slot: vertex and OWNER_BIT
  int32_t* iso = nullptr;  // vertices without tets, then their instances
  int n_iso = 0;
  // PNCG: per element block the quadratic form of the direction, and the states
  // after the step length (n), then after the decision (n); kept from one
  // apl_pncg_advance to the next
  double* hq = nullptr;
  InstState* st = nullptr;
  // the same of the CG (d.Hd; after the beta step, after the alpha step): its
  // own, so that a CG between two steps of a PNCG run leaves the run as it is
  double* cg_hq = nullptr;
  InstState* cg_st = nullptr;
  hipStream_t cap = nullptr;
  hipGraphExec_t gexec = nullptr;
  hipGraph_t graph = nullptr;
  std::vector<char> gkey;
  hipGraphExec_t cg_gexec = nullptr;  // K PCG iterations
  hipGraph_t cg_graph = nullptr;
  std::vector<char> cg_gkey;
  InstState* host_st = nullptr;  // pinned copy of the states
  struct apl_solver_run* run = nullptr;  // the step-wise solve in progress
};

namespace apl {

constexpr int N_VECS = 4;

template <class R>
static VecArgs<R> vec_args(apl_solver* s, const void* fext, const uint8_t* mask) {
  apl_mesh* m = s->mesh;
  VecArgs<R> A;
  A.vblk_off = m->d.vblk_off;
  A.vblk_inst = m->d.vblk_inst;
  A.vtx_slot_off = m->d.vtx_slot_off;
  A.partial = (const R*)m->d.partial;
  A.mask = mask;
  A.fext = (const R*)fext;
  A.x = s->x;
  A.p = (const Vec4<R>*)s->p;
  A.g = (Vec4<R>*)s->g;
  A.P = A.g + 2 * (size_t)m->L.V;
  A.vblk_dots = m->d.vblk_dots;
  A.blk_red = m->d.blk_red;
  A.inst_blk_off = m->d.inst_blk_off;
  A.inst_vblk_off = m->d.inst_vblk_off;
  A.st = s->st;
  A.V = (size_t)m->L.V;
  A.nvblk = (int)m->L.vblk_inst.size();
  A.nblocks = (int)m->L.nblocks;
  return A;
}

// the solver's buffers as its element passes see them (PNCG, or CG)
template <class R>
static SolveArgs<R> solve_args(apl_solver* s, bool cg) {
  apl_mesh* m = s->mesh;
  SolveArgs<R> S;
  S.st = cg ? s->cg_st : s->st;
  S.out = nullptr;
  S.table = nullptr;
  S.n_table = 0;
  S.x = s->x;
  S.V = (size_t)m->L.V;
  S.z = (const Vec4<R>*)s->cg;
  S.p = cg ? (Vec4<R>*)s->cg + S.V : (Vec4<R>*)s->p;
  S.g = (const Vec4<R>*)s->g;
  S.P = S.g + 2 * S.V;
  S.own = s->own;
  S.iso = s->iso;
  S.iso_inst = s->iso + s->n_iso;
  S.hq = cg ? s->cg_hq : s->hq;
  S.n_iso = s->n_iso;
  S.filter = m->L.n_inst > 1 ? 1 : 0;
  return S;
}

static Params to_params(const apl_pncg_params* p) {
  Params P;
  std::memset(&P, 0, sizeof P);  // the bytes (padding included) key the cached graph
  P.rtol = p->rtol;
  P.atol = p->atol;
  P.overstep = p->overstep;
  P.c1 = p->c1;
  P.wolfe_delta = p->wolfe_delta;
  P.wolfe_eps = p->wolfe_eps;
  P.beta_max = p->beta_max;
  P.max_steps = p->max_steps;
  P.max_backtracking = p->max_backtracking;
  P.stall_steps = p->stall_steps;
  return P;
}

// Persistent grid of the vector kernels: every vertex block its own
// workgroup up to sixteen per CU, beyond that a grid-stride loop.
static unsigned vec_grid(const apl_mesh* m) {
  const long long nvb = (long long)m->L.vblk_inst.size();
  const long long cap = 16LL * m->n_cu;
  return (unsigned)(nvb < cap ? nvb : cap);
}

constexpr unsigned PASS_TRIAL = W_E | W_G | W_H | W_TRIAL, PASS_DIR = W_HQ | W_DIR;
constexpr unsigned PASS_CGD = W_HP | W_VQ | W_CGD, PASS_ACT = W_HP | W_ACT;

template <class R>
static int pncg_iteration(apl_solver* s, const void* mu, const void* lam, const void* fext, const uint8_t* mask,
                          const Params& P, int grid, hipStream_t st) {
  apl_mesh* m = s->mesh;
  const VecArgs<R> A = vec_args<R>(s, fext, mask);
  SolveArgs<R> S = solve_args<R>(s, false);
  S.prm = P;
  const unsigned nvb = (unsigned)m->L.vblk_inst.size();
  const unsigned ni = (unsigned)m->L.n_inst;
  InstState *sa = s->st, *sb = s->st + ni;  // after the step length, after the decision
  const bool single = ni == 1 && m->L.nblocks > 0;
  // step length, trial pass
  int rc = 0;
  if (single && m->L.nblocks <= FUSE_BLOCKS) {
    S.st = sb, S.out = sa;
    S.table = s->hq, S.n_table = (int)m->L.nblocks;
    rc = launch_solve_pass<PASS_TRIAL | W_FUSED, R>(m, s->material, mu, lam, nullptr, nullptr, S, grid, st);
  } else {
    hipLaunchKernelGGL(pncg_alpha_kernel, dim3(ni), dim3(SCAL_TH), 0, st, sb, sa, P, s->hq, m->d.inst_blk_off);
    S.st = sa;
    rc = ni == 1 ? launch_solve_pass<PASS_TRIAL | W_ONE, R>(m, s->material, mu, lam, nullptr, nullptr, S, grid, st)
                 : launch_solve_pass<PASS_TRIAL, R>(m, s->material, mu, lam, nullptr, nullptr, S, grid, st);
  }
  if (rc) return -1;
  if (nvb && ni == 1)
    hipLaunchKernelGGL((pncg_reduce_kernel<R, true>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
  else if (nvb)
    hipLaunchKernelGGL((pncg_reduce_kernel<R, false>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
  // decision, direction pass
  if (single && nvb <= FUSE_VBLOCKS) {
    S.st = sa, S.out = sb;
    S.table = m->d.vblk_dots, S.n_table = (int)nvb * N_DOTS;
    rc = launch_solve_pass<PASS_DIR | W_FUSED, R>(m, s->material, mu, lam, nullptr, nullptr, S, grid, st);
  } else {
    hipLaunchKernelGGL(pncg_scalar_kernel, dim3(ni), dim3(SCAL_TH), 0, st, sa, sb, P, m->d.vblk_dots, m->d.inst_vblk_off);
    S.st = sb;
    rc = ni == 1 ? launch_solve_pass<PASS_DIR | W_ONE, R>(m, s->material, mu, lam, nullptr, nullptr, S, grid, st)
                 : launch_solve_pass<PASS_DIR, R>(m, s->material, mu, lam, nullptr, nullptr, S, grid, st);
  }
  if (rc) return -1;
  APL_CHECK_HIP(hipGetLastError());
  return 0;
}

template <class R>
static int fill(R* a, long long n, R v, hipStream_t st) {
  if (n <= 0) return 0;
  long long g = (n + NTH - 1) / NTH;
  if (g > 4096) g = 4096;
  hipLaunchKernelGGL((fill_kernel<R>), dim3((unsigned)g), dim3(NTH), 0, st, a, n, v);
  APL_CHECK_HIP(hipGetLastError());
  return 0;
}

// A solve in progress: what apl_pncg_begin bound, for the following
// advance / end calls.
struct PncgRun {
  bool open = false;
  const void* mu = nullptr;
  const void* lam = nullptr;
  void* x = nullptr;  // the caller's iterate (mesh dtype)
  const void* fext = nullptr;
  const uint8_t* mask = nullptr;
  Params P{};
  int K = 16, grid = 0;
  bool use_graph = true;
  long long done = 0, guard = 0;
};

template <class R>
static int pncg_begin_t(apl_solver* s, const void* mu, const void* lam, void* x, const void* fext,
                        const uint8_t* mask, const apl_pncg_params* prm, hipStream_t st);
template <class R>
static int pncg_advance_t(apl_solver* s, long long max_iters, int steps, hipStream_t st);
template <class R>
static int pncg_end_t(apl_solver* s, apl_pncg_stats* stats, hipStream_t st);

}  // namespace apl

struct apl_solver_run {
  apl::PncgRun r;
};

namespace apl {

template <class R>
static int pncg_begin_t(apl_solver* s, const void* mu, const void* lam, void* x, const void* fext,
                        const uint8_t* mask, const apl_pncg_params* prm, hipStream_t st) {
  apl_mesh* m = s->mesh;
  PncgRun& run = s->run->r;
  run.open = false;
  const int n = (int)m->L.n_inst;
  const Params P = to_params(prm);
  const int K = prm->iters_per_launch > 0 ? prm->iters_per_launch : 16;
  // reset state and work vectors (p and g_cur must start at zero)
  hipLaunchKernelGGL(solve_init_kernel, dim3((2 * n + 255) / 256), dim3(256), 0, st, s->st, n);
  const long long nv = m->L.V;
  if (fill<R>((R*)s->p, 4 * nv, R(0), st) || fill<R>((R*)s->g, 4 * nv, R(0), st)) return -1;
  APL_CHECK_HIP(hipGetLastError());
  // the iterate lives in FP64, in the solver's own pair of buffers
  if (nv > 0) {
    hipLaunchKernelGGL((start_kernel<R>), dim3((unsigned)std::min<long long>((nv + NTH - 1) / NTH, 4096)), dim3(NTH), 0, st,
                       (const R*)x, s->x, nv);
    APL_CHECK_HIP(hipGetLastError());
  }
  const int grid = prm->grid_override;
  // occupancy-derived grids are queried (and cached) outside any capture
  solve_pass_grid<PASS_TRIAL, R>(m, s->material);
  solve_pass_grid<PASS_DIR, R>(m, s->material);
  solve_pass_grid<PASS_TRIAL | W_ONE, R>(m, s->material);
  solve_pass_grid<PASS_DIR | W_ONE, R>(m, s->material);
  solve_pass_grid<PASS_TRIAL | W_FUSED, R>(m, s->material);
  solve_pass_grid<PASS_DIR | W_FUSED, R>(m, s->material);
  // cached graph of K iterations for these pointers and parameters
  bool use_graph = prm->use_graph != 0;
  if (use_graph) {
    std::vector<char> key(sizeof(void*) * 5 + sizeof(Params) + 3 * sizeof(int));
    char* k = key.data();
    const void* ptrs[5] = {mu, lam, fext, mask, m->activation};
    std::memcpy(k, ptrs, sizeof ptrs);
    k += sizeof ptrs;
    std::memcpy(k, &P, sizeof P);
    k += sizeof P;
    std::memcpy(k, &K, sizeof K);
    k += sizeof K;
    std::memcpy(k, &grid, sizeof grid);
    k += sizeof grid;
    std::memcpy(k, &m->grid_pct, sizeof m->grid_pct);
    if (s->gexec == nullptr || key != s->gkey) {
      if (s->gexec) {
        drop_hip_error(hipGraphExecDestroy(s->gexec));
        s->gexec = nullptr;
      }
      if (s->graph) {
        drop_hip_error(hipGraphDestroy(s->graph));
        s->graph = nullptr;
      }
      if (s->cap == nullptr) APL_CHECK_HIP(hipStreamCreateWithFlags(&s->cap, hipStreamNonBlocking));
      APL_CHECK_HIP(hipStreamBeginCapture(s->cap, hipStreamCaptureModeThreadLocal));
      int rc = 0;
      for (int it = 0; it < K && rc == 0; ++it) rc = pncg_iteration<R>(s, mu, lam, fext, mask, P, grid, s->cap);
      hipGraph_t g = nullptr;
      hipError_t e = hipStreamEndCapture(s->cap, &g);
      if (rc != 0 || e != hipSuccess) {
        if (g) drop_hip_error(hipGraphDestroy(g));
        if (rc == 0) set_error(std::string("graph capture failed: ") + hipGetErrorString(e));
        return -1;
      }
      s->graph = g;
      APL_CHECK_HIP(hipGraphInstantiate(&s->gexec, g, nullptr, nullptr, 0));
      s->gkey = key;
    }
  }
  run.mu = mu;
  run.lam = lam;
  run.x = x;
  run.fext = fext;
  run.mask = mask;
  run.P = P;
  run.K = K;
  run.grid = grid;
  run.use_graph = use_graph;
  run.done = 0;
  run.guard = ((long long)prm->max_steps + 2) * ((long long)prm->max_backtracking + 2) * 2 + 8;
  run.open = true;
  return 0;
}

// the instances' states after an iteration on the host (waits for the stream)
static int read_states(apl_solver* s, const InstState* states, hipStream_t st) {
  const size_t n = (size_t)s->mesh->L.n_inst;
  APL_CHECK_HIP(hipMemcpyAsync(s->host_st, states + n, n * sizeof(InstState), hipMemcpyDeviceToHost, st));
  APL_CHECK_HIP(hipStreamSynchronize(st));
  return 0;
}

// the committed iterate into a caller's (V,3) array
template <class R>
static int copy_iterate(apl_solver* s, void* out, hipStream_t st) {
  apl_mesh* m = s->mesh;
  const unsigned nvb = (unsigned)m->L.vblk_inst.size();
  if (nvb == 0) return 0;
  hipLaunchKernelGGL((iterate_kernel<R>), dim3(nvb), dim3(NTH), 0, st, s->st + m->L.n_inst, m->d.vblk_off, m->d.vblk_inst, s->x,
                     (size_t)m->L.V, (R*)out);
  APL_CHECK_HIP(hipGetLastError());
  return 0;
}

// Run device iterations (trial evaluations) until no instance is running,
// the guard is reached, max_iters more have run (max_iters > 0) or, when
// steps > 0, every running instance has taken that many more accepted steps
// (one trial per launch, with a status read after each).
template <class R>
static int pncg_advance_t(apl_solver* s, long long max_iters, int steps, hipStream_t st) {
  apl_mesh* m = s->mesh;
  PncgRun& run = s->run->r;
  const int n = (int)m->L.n_inst;
  std::vector<int32_t> target;
  if (steps > 0) {
    if (read_states(s, s->st, st)) return -1;
    for (int i = 0; i < n; ++i) target.push_back(s->host_st[i].n_steps + steps);
  }
  long long ran = 0;
  while (true) {
    // one trial per launch when counting steps; eager launches for a
    // remainder shorter than the captured graph
    const long long left = max_iters > 0 ? max_iters - ran : run.K;
    const bool graph = run.use_graph && steps <= 0 && left >= run.K;
    const int K = steps > 0 ? 1 : (graph ? run.K : (int)std::min<long long>(run.K, left));
    if (graph) {
      APL_CHECK_HIP(hipGraphLaunch(s->gexec, st));
    } else {
      for (int it = 0; it < K; ++it)
        if (pncg_iteration<R>(s, run.mu, run.lam, run.fext, run.mask, run.P, run.grid, st)) return -1;
    }
    run.done += K;
    ran += K;
    if (read_states(s, s->st, st)) return -1;
    bool running = false, pending = false;
    for (int i = 0; i < n; ++i) {
      const bool r = s->host_st[i].status == APL_RUNNING;
      running = running || r;
      if (steps > 0 && r && s->host_st[i].n_steps < target[i]) pending = true;
    }
    if (!running || run.done > run.guard || (max_iters > 0 && ran >= max_iters) || (steps > 0 && !pending)) break;
  }
  return 0;
}

// Copy the iterate into the caller's x and read the stats.
template <class R>
static int pncg_end_t(apl_solver* s, apl_pncg_stats* stats, hipStream_t st) {
  PncgRun& run = s->run->r;
  if (copy_iterate<R>(s, run.x, st)) return -1;
  if (stats != nullptr) {
    if (read_states(s, s->st, st)) return -1;
    for (int i = 0; i < (int)s->mesh->L.n_inst; ++i) {
      const InstState& h = s->host_st[i];
      apl_pncg_stats& o = stats[i];
      o.f = h.f;
      o.alpha = h.alpha_commit;
      o.beta = h.beta;
      o.grad_norm_first = h.gnorm0;
      o.grad_norm = h.gnorm;
      o.f_first = h.f_first;
      o.status = h.status;
      o.n_steps = h.n_steps;
      o.n_evals = h.n_evals;
      o.n_backtracks = h.n_backtracks;
      if (o.status == APL_RUNNING) o.status = APL_MAX_STEPS_REACHED;
    }
  }
  return 0;
}

template <class R>
static int pncg_solve_t(apl_solver* s, const void* mu, const void* lam, void* x, const void* fext,
                        const uint8_t* mask, const apl_pncg_params* prm, apl_pncg_stats* stats, hipStream_t st) {
  if (pncg_begin_t<R>(s, mu, lam, x, fext, mask, prm, st)) return -1;
  if (pncg_advance_t<R>(s, 0, 0, st)) return -1;
  const int rc = pncg_end_t<R>(s, stats, st);
  s->run->r.open = false;
  return rc;
}

template <class R>
static CgArgs<R> cg_args(apl_solver* s, const void* rhs, void* y, const uint8_t* mask) {
  apl_mesh* m = s->mesh;
  const size_t nv = 3 * (size_t)m->L.V;
  R* base = (R*)s->vecs;
  CgArgs<R> A;
  A.vblk_off = m->d.vblk_off;
  A.vblk_inst = m->d.vblk_inst;
  A.vtx_slot_off = m->d.vtx_slot_off;
  A.partial = (const R*)m->d.partial;
  A.mask = mask;
  A.rhs = (const R*)rhs;
  A.y = (R*)y;
  A.r = base;
  A.z = (Vec4<R>*)s->cg;
  A.d = (Vec4<R>*)s->cg + (size_t)m->L.V;
  A.hd = base + nv;
  A.t = base + 2 * nv;
  A.tout = A.t;
  A.nvblk = (int)m->L.vblk_inst.size();
  A.nblocks = (int)m->L.nblocks;
  A.vblk_dots = m->d.vblk_dots;
  A.t_dots = m->d.vblk_dots + 2 * (size_t)A.nvblk;
  A.in = s->cg_st + m->L.n_inst;
  A.out = nullptr;
  A.hq = s->cg_hq;
  A.V = (size_t)m->L.V;
  A.normal = 0;
  return A;
}

template <class R>
static int cg_iteration(apl_solver* s, const void* mu, const void* lam, const void* x, CgArgs<R> A, double rtol,
                        int max_iters, hipStream_t st) {
  apl_mesh* m = s->mesh;
  const unsigned nvb = (unsigned)m->L.vblk_inst.size();
  const unsigned ni = (unsigned)m->L.n_inst;
  InstState *sa = s->cg_st, *sb = s->cg_st + ni;  // after the beta step, after the alpha step
  const bool single = ni == 1 && m->L.nblocks > 0;
  SolveArgs<R> S = solve_args<R>(s, true);
  S.prm.rtol = rtol;
  S.prm.max_steps = max_iters;
  int rc = 0;
  if (single && nvb <= FUSE_CG_VBLOCKS) {
    S.st = sb, S.out = sa;
    S.table = m->d.vblk_dots, S.n_table = 2 * (int)nvb;
    rc = launch_solve_pass<PASS_CGD | W_FUSED, R>(m, s->material, mu, lam, x, nullptr, S, 0, st);
  } else {
    hipLaunchKernelGGL(cg_beta_kernel, dim3(ni), dim3(SCAL_TH), 0, st, sb, sa, rtol, max_iters, m->d.vblk_dots,
                       m->d.inst_vblk_off);
    S.st = sa;
    rc = launch_solve_pass<PASS_CGD, R>(m, s->material, mu, lam, x, nullptr, S, 0, st);
  }
  if (rc) return -1;
  if (A.normal) {
    // q = H (H d): t = H d with fixed DOFs zeroed, whose square is d.H^2 d, then the pass on t
    A.in = sa;
    if (nvb) hipLaunchKernelGGL((cg_vec_kernel<R, CG_T>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
    S.st = sa;
    if (launch_solve_pass<PASS_ACT, R>(m, s->material, mu, lam, x, A.t, S, 0, st)) return -1;
  }
  if (single && !A.normal && m->L.nblocks <= FUSE_BLOCKS) {
    A.in = sa, A.out = sb;
    if (nvb) hipLaunchKernelGGL((cg_update_kernel<R, U_FUSED>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
  } else {
    hipLaunchKernelGGL(cg_alpha_kernel, dim3(ni), dim3(SCAL_TH), 0, st, sa, sb, A.normal ? A.t_dots : s->cg_hq,
                       A.normal ? m->d.inst_vblk_off : m->d.inst_blk_off);
    A.in = sb;
    if (nvb && ni == 1)
      hipLaunchKernelGGL((cg_update_kernel<R, U_SINGLE>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
    else if (nvb)
      hipLaunchKernelGGL((cg_update_kernel<R, U_BATCH>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
  }
  APL_CHECK_HIP(hipGetLastError());
  return 0;
}

template <class R>
static int cg_solve_t(apl_solver* s, const void* mu, const void* lam, const void* x, const void* rhs, void* y,
                      const uint8_t* mask, double rtol, int max_iters, apl_pncg_stats* stats, hipStream_t st,
                      int normal) {
  apl_mesh* m = s->mesh;
  const int n = (int)m->L.n_inst;
  const unsigned nvb = (unsigned)m->L.vblk_inst.size();
  CgArgs<R> A = cg_args<R>(s, rhs, y, mask);
  hipLaunchKernelGGL(solve_init_kernel, dim3((2 * n + 255) / 256), dim3(256), 0, st, s->cg_st, n);
  if (normal) {
    // the normal equations' right-hand side H b (b with fixed DOFs zeroed),
    // kept by the solver; the CG then runs on it
    A.normal = 1;
    R* b2 = (R*)s->vecs + 3 * 3 * (size_t)m->L.V;
    CgArgs<R> Ab = A;
    Ab.tout = A.t;
    if (nvb) hipLaunchKernelGGL((cg_vec_kernel<R, CG_MASKCOPY>), dim3(vec_grid(m)), dim3(NTH), 0, st, Ab);
    if (launch_elem(m, s->material, W_HP, mu, lam, x, A.t, nullptr, nullptr, 0, st)) return -1;
    Ab.tout = b2;
    if (nvb) hipLaunchKernelGGL((cg_vec_kernel<R, CG_T>), dim3(vec_grid(m)), dim3(NTH), 0, st, Ab);
    A.rhs = b2;
  }
  // zero the diagonal buffer (vertices with no tet keep 0) and run the Hdiag pass at x
  if (fill<R>(A.hd, 3 * (long long)m->L.V, R(0), st)) return -1;
  if (launch_elem(m, s->material, W_H, mu, lam, x, nullptr, nullptr, A.hd, 0, st)) return -1;
  if (nvb) hipLaunchKernelGGL((cg_vec_kernel<R, CG_DIAG>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
  InstState* sb = s->cg_st + n;
  hipLaunchKernelGGL(cg_scalar_kernel, dim3(n), dim3(SCAL_TH), 0, st, sb, 0, m->d.vblk_dots, m->d.inst_vblk_off);
  if (nvb) hipLaunchKernelGGL((cg_vec_kernel<R, CG_PRECOND>), dim3(vec_grid(m)), dim3(NTH), 0, st, A);
  hipLaunchKernelGGL(cg_scalar_kernel, dim3(n), dim3(SCAL_TH), 0, st, sb, 1, m->d.vblk_dots, m->d.inst_vblk_off);
  APL_CHECK_HIP(hipGetLastError());
  solve_pass_grid<PASS_CGD, R>(m, s->material);
  solve_pass_grid<PASS_CGD | W_FUSED, R>(m, s->material);
  if (normal) solve_pass_grid<PASS_ACT, R>(m, s->material);
  const int K = 16;
  // K iterations captured once per set of pointers and parameters
  {
    std::vector<char> key(sizeof(void*) * 7 + sizeof(double) + 3 * sizeof(int));
    char* k = key.data();
    const void* ptrs[7] = {mu, lam, x, rhs, y, mask, m->activation};
    std::memcpy(k, ptrs, sizeof ptrs);
    k += sizeof ptrs;
    std::memcpy(k, &rtol, sizeof rtol);
    k += sizeof rtol;
    std::memcpy(k, &max_iters, sizeof max_iters);
    k += sizeof max_iters;
    std::memcpy(k, &normal, sizeof normal);
    k += sizeof normal;
    std::memcpy(k, &m->grid_pct, sizeof m->grid_pct);
    if (s->cg_gexec == nullptr || key != s->cg_gkey) {
      if (s->cg_gexec) {
        drop_hip_error(hipGraphExecDestroy(s->cg_gexec));
        s->cg_gexec = nullptr;
      }
      if (s->cg_graph) {
        drop_hip_error(hipGraphDestroy(s->cg_graph));
        s->cg_graph = nullptr;
      }
      if (s->cap == nullptr) APL_CHECK_HIP(hipStreamCreateWithFlags(&s->cap, hipStreamNonBlocking));
      APL_CHECK_HIP(hipStreamBeginCapture(s->cap, hipStreamCaptureModeThreadLocal));
      int rc = 0;
      for (int it = 0; it < K && rc == 0; ++it) rc = cg_iteration<R>(s, mu, lam, x, A, rtol, max_iters, s->cap);
      hipGraph_t g = nullptr;
      hipError_t e = hipStreamEndCapture(s->cap, &g);
      if (rc != 0 || e != hipSuccess) {
        if (g) drop_hip_error(hipGraphDestroy(g));
        if (rc == 0) set_error(std::string("graph capture failed: ") + hipGetErrorString(e));
        return -1;
      }
      s->cg_graph = g;
      APL_CHECK_HIP(hipGraphInstantiate(&s->cg_gexec, g, nullptr, nullptr, 0));
      s->cg_gkey = key;
    }
  }
  // (an update's residual is tested at the start of the next iteration, so an
  // instance that ends with a launch's last update is seen to after the next launch)
  long long done = 0;
  while (true) {
    APL_CHECK_HIP(hipGraphLaunch(s->cg_gexec, st));
    done += K;
    if (read_states(s, s->cg_st, st)) return -1;
    bool running = false;
    for (int i = 0; i < n; ++i) running = running || s->host_st[i].status == APL_RUNNING;
    if (!running || done > (long long)max_iters + K) break;
  }
  if (stats != nullptr) {
    for (int i = 0; i < n; ++i) {
      const InstState& h = s->host_st[i];  // as read after the last iterations
      apl_pncg_stats& o = stats[i];
      o.f = h.f;
      o.alpha = h.alpha;
      o.beta = h.beta;
      o.grad_norm_first = h.gnorm0;
      o.grad_norm = h.gnorm;
      o.f_first = 1.0;
      o.status = h.status == APL_RUNNING ? APL_MAX_STEPS_REACHED : h.status;
      o.n_steps = h.n_steps;
      o.n_evals = h.n_steps;
      o.n_backtracks = 0;
    }
  }
  return 0;
}

}  // namespace apl

extern "C" {

int apl_solver_create(apl_mesh* m, int material, apl_solver** out) {
  if (m == nullptr || out == nullptr) {
    set_error("NULL argument");
    return -1;
  }
  if (!material_ok(m, material)) {
    set_error(m->model ? "a model mesh takes material APL_MODEL"
                       : "material must be APL_SNH, APL_ARAP or APL_SNH_MUSCLE");
    return -1;
  }
  *out = nullptr;
  APL_CHECK_HIP(hipSetDevice(m->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  apl_solver* s = new apl_solver();
  s->run = new apl_solver_run();
  s->mesh = m;
  ++m->refs;
  s->device = m->device;
  s->material = material;
  const int n = (int)m->L.n_inst;
  // one allocation, cut into 256-byte aligned parts
  const size_t nv = (size_t)std::max<int64_t>(m->L.V, 1), rs = real_size(m);
  size_t total = 0;
  auto part = [&](size_t bytes) {
    const size_t off = total;
    total += (bytes + 255) / 256 * 256;
    return off;
  };
  const size_t o_st = part(2 * (size_t)n * sizeof(InstState)), o_cg_st = part(2 * (size_t)n * sizeof(InstState)),
               o_iso = part(sizeof(int)), o_x = part(2 * nv * 4 * sizeof(double)), o_p = part(2 * nv * 4 * rs),
               o_g = part(3 * nv * 4 * rs), o_cg = part(3 * nv * 4 * rs),
               o_vecs = part(N_VECS * nv * 3 * rs),
               o_own = part((size_t)std::max<int64_t>(m->L.n_slots, 1) * sizeof(uint32_t)),
               o_hq = part((size_t)std::max<int64_t>(m->L.nblocks, 1) * sizeof(double)),
               o_cg_hq = part((size_t)std::max<int64_t>(m->L.nblocks, 1) * sizeof(double));
  auto fail = [&](const char* what) {
    set_error(what);
    (void)hipGetLastError();
    apl_solver_destroy(s);
    return -1;
  };
  if (hipMalloc(&s->mem, total) != hipSuccess ||
      hipHostMalloc((void**)&s->host_st, (size_t)n * sizeof(InstState), 0) != hipSuccess)
    return fail("out of memory creating the solver");
  char* base = (char*)s->mem;
  s->st = (InstState*)(base + o_st);
  int* iso_count = (int*)(base + o_iso);
  s->x = (Vec4<double>*)(base + o_x);
  s->p = base + o_p;
  s->g = base + o_g;
  s->cg = base + o_cg;
  s->vecs = base + o_vecs;
  s->own = (uint32_t*)(base + o_own);
  s->hq = (double*)(base + o_hq);
  s->cg_st = (InstState*)(base + o_cg_st);
  s->cg_hq = (double*)(base + o_cg_hq);
  // zeroed once: a solve overwrites what it reads
  if (hipMemset(s->mem, 0, o_own) != hipSuccess) return fail("hipMemset failed creating the solver");
  // owner slots, and the vertices that no tet touches
  const unsigned nvb = (unsigned)m->L.vblk_inst.size();
  if (m->L.n_slots > 0)
    hipLaunchKernelGGL(owner_kernel, dim3((unsigned)std::min<int64_t>((m->L.n_slots + NTH - 1) / NTH, 8192)), dim3(NTH), 0,
                       nullptr, m->d.loc_gid, m->d.loc_dst, m->d.vtx_slot_off, (long long)m->L.n_slots, s->own);
  if (nvb > 0)
    hipLaunchKernelGGL(isolated_kernel, dim3(nvb), dim3(NTH), 0, nullptr, m->d.vblk_off, m->d.vblk_inst, m->d.vtx_slot_off,
                       iso_count, (int32_t*)nullptr, (int32_t*)nullptr);
  if (hipGetLastError() != hipSuccess ||
      hipMemcpy(&s->n_iso, iso_count, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess)
    return fail("setup kernels failed creating the solver");
  if (s->n_iso > 0) {
    if (hipMalloc((void**)&s->iso, 2 * (size_t)s->n_iso * sizeof(int32_t)) != hipSuccess)
      return fail("out of device memory creating the solver");
    if (hipMemset(iso_count, 0, sizeof(int)) != hipSuccess) return fail("hipMemset failed creating the solver");
    hipLaunchKernelGGL(isolated_kernel, dim3(nvb), dim3(NTH), 0, nullptr, m->d.vblk_off, m->d.vblk_inst, m->d.vtx_slot_off,
                       iso_count, s->iso, s->iso + s->n_iso);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess)
      return fail("setup kernels failed creating the solver");
  }
  *out = s;
  return 0;
}

int apl_solver_destroy(apl_solver* s) {
  if (s == nullptr) return 0;
  drop_hip_error(hipSetDevice(s->device));
  if (s->gexec) drop_hip_error(hipGraphExecDestroy(s->gexec));
  if (s->graph) drop_hip_error(hipGraphDestroy(s->graph));
  if (s->cg_gexec) drop_hip_error(hipGraphExecDestroy(s->cg_gexec));
  if (s->cg_graph) drop_hip_error(hipGraphDestroy(s->cg_graph));
  if (s->cap) drop_hip_error(hipStreamDestroy(s->cap));
  if (s->mem) drop_hip_error(hipFree(s->mem));
  if (s->iso) drop_hip_error(hipFree(s->iso));
  if (s->host_st) drop_hip_error(hipHostFree(s->host_st));
  delete s->run;
  if (s->mesh) mesh_release(s->mesh);
  delete s;
  return 0;
}

int apl_pncg_solve(apl_solver* s, const void* mu, const void* lam, void* x, const void* f_ext,
                   const uint8_t* fixed_mask, const apl_pncg_params* params, apl_pncg_stats* stats, void* stream) {
  if (s == nullptr || params == nullptr || (s->mesh->L.V > 0 && x == nullptr) ||
      (s->mesh->L.T > 0 && (mu == nullptr || (needs_lambda(s->mesh, s->material) && lam == nullptr)))) {
    set_error("NULL argument");
    return -1;
  }
  if (params->max_steps < 0 || params->max_backtracking < 0 || !(params->rtol >= 0) || !(params->atol >= 0)) {
    set_error("invalid PNCG parameters");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(s->mesh->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  if (s->mesh->dtype == DT_F32)
    return pncg_solve_t<float>(s, mu, lam, x, f_ext, fixed_mask, params, stats, (hipStream_t)stream);
  return pncg_solve_t<double>(s, mu, lam, x, f_ext, fixed_mask, params, stats, (hipStream_t)stream);
}

int apl_pncg_begin(apl_solver* s, const void* mu, const void* lam, void* x, const void* f_ext,
                   const uint8_t* fixed_mask, const apl_pncg_params* params, void* stream) {
  if (s == nullptr || params == nullptr || (s->mesh->L.V > 0 && x == nullptr) ||
      (s->mesh->L.T > 0 && (mu == nullptr || (needs_lambda(s->mesh, s->material) && lam == nullptr)))) {
    set_error("NULL argument");
    return -1;
  }
  if (params->max_steps < 0 || params->max_backtracking < 0 || !(params->rtol >= 0) || !(params->atol >= 0)) {
    set_error("invalid PNCG parameters");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(s->mesh->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  if (s->mesh->dtype == DT_F32) return pncg_begin_t<float>(s, mu, lam, x, f_ext, fixed_mask, params, (hipStream_t)stream);
  return pncg_begin_t<double>(s, mu, lam, x, f_ext, fixed_mask, params, (hipStream_t)stream);
}

int apl_pncg_advance(apl_solver* s, int32_t steps, int64_t max_iters, void* x_out, apl_pncg_state* state,
                     void* stream) {
  if (s == nullptr || !s->run->r.open) {
    set_error("no PNCG run in progress: call apl_pncg_begin first");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(s->mesh->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  hipStream_t st = (hipStream_t)stream;
  apl_mesh* m = s->mesh;
  const bool f32 = m->dtype == DT_F32;
  if ((f32 ? pncg_advance_t<float>(s, max_iters, steps, st) : pncg_advance_t<double>(s, max_iters, steps, st)))
    return -1;
  const long long nx = 3 * (long long)m->L.V;
  if (x_out != nullptr && nx > 0 && (f32 ? copy_iterate<float>(s, x_out, st) : copy_iterate<double>(s, x_out, st)))
    return -1;
  if (state != nullptr) {
    if (read_states(s, s->st, st)) return -1;
    for (int i = 0; i < (int)m->L.n_inst; ++i) {
      const InstState& h = s->host_st[i];
      apl_pncg_state& o = state[i];
      o.status = h.status;
      o.n_steps = h.n_steps;
      o.n_evals = h.n_evals;
      o.ls_steps = h.ls_last;
      o.ok = h.restarts == 0 ? 1 : 0;
      o.alpha = h.alpha_commit;
      o.f0 = h.f0;
      o.f_alpha = h.f;
      o.grad_norm = h.gnorm;
      o.grad_norm_first = h.gnorm0;
      o.hess_diag_mean = h.pmean;
      o.beta = h.beta;
    }
  }
  return 0;
}

int apl_pncg_end(apl_solver* s, apl_pncg_stats* stats, void* stream) {
  if (s == nullptr || !s->run->r.open) {
    set_error("no PNCG run in progress: call apl_pncg_begin first");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(s->mesh->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  hipStream_t st = (hipStream_t)stream;
  const int rc = s->mesh->dtype == DT_F32 ? pncg_end_t<float>(s, stats, st) : pncg_end_t<double>(s, stats, st);
  s->run->r.open = false;
  return rc;
}

int apl_cg_solve(apl_solver* s, const void* mu, const void* lam, const void* x, const void* rhs, void* y,
                 const uint8_t* fixed_mask, double rtol, int max_iters, apl_pncg_stats* stats, void* stream) {
  if (s == nullptr || (s->mesh->L.V > 0 && (x == nullptr || rhs == nullptr || y == nullptr)) ||
      (s->mesh->L.T > 0 && (mu == nullptr || (needs_lambda(s->mesh, s->material) && lam == nullptr)))) {
    set_error("NULL argument");
    return -1;
  }
  if (!(rtol >= 0) || max_iters < 0) {
    set_error("invalid CG parameters");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(s->mesh->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  if (s->mesh->dtype == DT_F32)
    return cg_solve_t<float>(s, mu, lam, x, rhs, y, fixed_mask, rtol, max_iters, stats, (hipStream_t)stream, 0);
  return cg_solve_t<double>(s, mu, lam, x, rhs, y, fixed_mask, rtol, max_iters, stats, (hipStream_t)stream, 0);
}

int apl_cg_solve_normal(apl_solver* s, const void* mu, const void* lam, const void* x, const void* rhs, void* y,
                        const uint8_t* fixed_mask, double rtol, int max_iters, apl_pncg_stats* stats, void* stream) {
  if (s == nullptr || (s->mesh->L.V > 0 && (x == nullptr || rhs == nullptr || y == nullptr)) ||
      (s->mesh->L.T > 0 && (mu == nullptr || (needs_lambda(s->mesh, s->material) && lam == nullptr)))) {
    set_error("NULL argument");
    return -1;
  }
  if (!(rtol >= 0) || max_iters < 0) {
    set_error("invalid CG parameters");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(s->mesh->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  if (s->mesh->dtype == DT_F32)
    return cg_solve_t<float>(s, mu, lam, x, rhs, y, fixed_mask, rtol, max_iters, stats, (hipStream_t)stream, 1);
  return cg_solve_t<double>(s, mu, lam, x, rhs, y, fixed_mask, rtol, max_iters, stats, (hipStream_t)stream, 1);
}

}  // extern "C"
