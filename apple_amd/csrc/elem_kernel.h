// Element kernel template: one pass over the tets of every block computes any of
// energy, gradient, clamped Hessian diagonal, Hessian-vector product,
// clamped quadratic form and mixed parameter derivatives, and reduces the
// per-vertex quantities deterministically.
//
// Replaces the fun/grad/hess_diag/hess_prod/hess_quad kernel templates of
// warp/fem/_base.py:243-383 (one launch and one re-gather of u per quantity,
// float atomics for every reduction) by one fused launch per pass:
//
//  * each workgroup (256 threads) owns a run of consecutive tets (a block) and
//    stages the displacement of every vertex the block touches into LDS once
//    (padded to 4 lanes, one wide LDS read per corner);
//  * per-tet element data are SoA in HBM (9 x T inverse rest shapes, dV, mu,
//    lambda, and one 16-byte record of 4 local corner slots and 4 corner
//    positions), addressed by 32-bit offsets from per-block uniform base
//    pointers: every load is coalesced;
//  * each corner's contribution goes to LDS at its position (corners ranked
//    by slot, then tet, then corner; channels packed into 16/8-byte records),
//    so the corners of a local vertex form a contiguous run; one to four lanes sum each run in a fixed order
//    (bitwise reproducible) and one partial per slot goes into a
//    vertex-major buffer (a vertex's partials contiguous, in block order);
//    the vertex pass adds each vertex's contiguous run;
//  * energies and quadratic forms are summed per thread, then in FP64 by a
//    fixed DPP tree per wave and over the block's four waves in order (behind
//    the barrier of the slot sums where a pass has them); a per-instance pass
//    adds the blocks' values in a fixed order;
//  * the grid is persistent and XCD-aware: workgroup i runs on XCD i % 8, and
//    XCD x walks every eighth chunk of up to 16 consecutive blocks, so
//    neighbouring blocks (which share vertices) mostly hit the same L2 while
//    any instance of more than 8 chunks spreads over all XCDs.
#pragma once

#include "internal.h"
#include "tetmath.h"
#include "flatsum.h"
#include "lanes.h"
#include "persist.h"
#include "solve_state.h"

#include <algorithm>
#include <type_traits>

namespace apl {

constexpr int XCD_CHUNK = 16;  // consecutive blocks per XCD chunk
constexpr size_t ELEM_LDS_MAX = 65536;  // LDS one element workgroup may use

template <class R, class X>
struct ElemArgs {
  const R* dminv;
  const R* dV;
  const uint4* corner;  // per tet: 4 x u16 local slots, 4 x u16 chunk positions
  const int32_t* blk_tet_off;
  const int32_t* blk_loc_off;
  const int32_t* blk_inst;
  const int32_t* loc_gid;
  const int32_t* loc_dst;
  const int32_t* blk_co_off;
  const uint16_t* chunk_off;
  const R* mu;
  const R* lam;
  const R* act;  // (T, 6) activation of the muscle law
  const X* x;  // displacements (X = R, or the solver's FP64 iterate)
  const R* p;
  R* out_a;  // per-tet outputs of the mixed pass
  R* out_b;
  R* out_c;  // (T, 6) activation derivatives of the mixed pass
  R* partial;  // vertex-major partial sums (scatter passes)
  double* blk_red;
  const int32_t* blk_list;  // model meshes: this law's blocks (else NULL: every block)
  int T;
  int nblocks;  // blocks this launch visits (the list's length with a list)
  int nloc_max;
  int accumulate;
};

// 4-lane padded vector (one 16/32-byte access)
template <class T>
struct alignas(4 * sizeof(T)) Vec4 {
  T v[4];
};

// The solver's element passes.  WHAT carries one of these staging modes
// beside the outputs:
//   W_TRIAL  the PNCG trial point x + alpha p of the instance's committed
//            buffers, alpha from its state
//   W_DIR    the accepted step: the block forms the new iterate and direction
//            of its vertices while it stages them, and the slot that comes
//            first in a vertex's partial run (the owner) writes them to the
//            other buffer.  As a launch of its own the step took 8.2 us at
//            64^3 cubes and 3.8 us (the launch) at 10^3; here it adds 4.5 us
//            to a 20 us pass at 64^3 (the records of a vertex are read once
//            per block that touches it, 2.3 times) and nothing at 10^3.
//   W_CGD    the CG direction d = z + beta d, formed and written the same way;
//            with W_VQ its d.Hd, so that the update needs no pass of its own
//            for the step length
//   W_ACT    the caller's direction, blocks of running instances only
// W_ONE with W_TRIAL or W_DIR: the mesh has one instance, whose scalars each
// workgroup reads once, by scalar loads (64^3: trial pass 31.0 -> 30.3 us,
// direction pass 24.2 -> 23.7, against one variant for both; a batch's
// direction pass grows from 24.6 to 26.6 us if it reads its states that way).
// W_FUSED with one of them: a single instance's pass that takes the scalar
// step before it (scalar_step).  A variant of its own: the batches' passes
// lose 8-15 % to the registers and scalar traffic of that code.
constexpr unsigned W_TRIAL = 256u, W_DIR = 512u, W_CGD = 1024u, W_ACT = 2048u, W_FUSED = 4096u,
                   W_ONE = 8192u;
constexpr unsigned W_SOLVER = W_TRIAL | W_DIR | W_CGD | W_ACT;
constexpr unsigned W_OUT = 255u;  // the bits tet_eval knows
constexpr unsigned OWNER_BIT = 0x80000000u;

struct NoSolve {};

// The solver's vertex data, one padded record per vertex: a staged slot reads
// a few 16-byte words (the runs of 3 scalars that a (V,3) array gives cost
// three loads each, and the staging loads are what bounds the direction pass).
template <class R>
struct SolveArgs {
  const InstState* st;  // the states this pass acts on; W_FUSED: those before its scalar step,
  InstState* out;       // where workgroup 0 keeps those after it,
  const double* table;  // and the table that the pass before left for it
  int n_table;
  Params prm;
  Vec4<double>* x;  // PNCG iterate: two buffers of V (InstState::cur)
  Vec4<R>* p;       // PNCG / CG direction: two buffers of V
  const Vec4<R>* g;   // two buffers of V: g - f, 0 on fixed DOFs
  const Vec4<R>* P;   // 1 / diag H: 0 on fixed DOFs, -1 where the diagonal is not positive
  const Vec4<R>* z;   // CG: preconditioned residual
  const uint32_t* own;   // per slot: vertex, OWNER_BIT on the vertex's first slot
  const int32_t* iso;    // vertices no tet touches, and their instances
  const int32_t* iso_inst;
  double* hq;     // per block quadratic form
  size_t V;
  int n_iso;      // (first launch of a pass only)
  int filter;     // visit only blocks of active instances (batches)
};

// The scalars of an instance that a pass needs, in scalar registers.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}

// Entry i of a table that the kernel does not write, i uniform: a scalar load
// whatever the compiler knows of the kernel's stores.
#define APL_CONSTANT __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ const APL_CONSTANT T& constant_at(const T* t, int i) {
  return ((const APL_CONSTANT T*)(uintptr_t)t)[i];
}

struct InstScalars {
  double alpha, alpha_commit, beta, pmean;
  int act_eval, commit, act_dir, cur;
  InstScalars() = default;
  __device__ explicit InstScalars(const InstState& s)
      : alpha(uni(s.alpha)), alpha_commit(uni(s.alpha_commit)), beta(uni(s.beta)), pmean(uni(s.pmean)),
        act_eval(uni(s.act_eval)), commit(uni(s.commit)), act_dir(uni(s.act_dir)), cur(uni(s.cur)) {}
  __device__ explicit InstScalars(const APL_CONSTANT InstState& s)
      : alpha(s.alpha), alpha_commit(s.alpha_commit), beta(s.beta), pmean(s.pmean), act_eval(s.act_eval),
        commit(s.commit), act_dir(s.act_dir), cur(s.cur) {}
};

// An accepted step: x += alpha_commit p, p = -P g + beta p with the Jacobi
// preconditioner P = 1/diag H (the mean of the positive entries where the
// diagonal is not positive).
template <class R>
struct Step {
  double a;
  R beta, ipm;
  bool dir;
  const Vec4<double>* x0;
  const Vec4<R>* p0;
  const Vec4<R>* g;
  const Vec4<R>* P;
  Vec4<double>* x1;
  Vec4<R>* p1;
  template <class State>
  __device__ Step(const SolveArgs<R>& S, const State& st, int cur)
      : a(st.alpha_commit), beta((R)st.beta), ipm(R(1) / (R)st.pmean), dir(st.act_dir != 0),
        x0(S.x + (cur ? (size_t)0 : S.V)), p0(S.p + (cur ? (size_t)0 : S.V)),
        g(S.g + (cur ? S.V : (size_t)0)), P(S.P), x1(S.x + (cur ? S.V : (size_t)0)),
        p1(S.p + (cur ? S.V : (size_t)0)) {}
};

// Element i of a uniform base pointer through a 32-bit byte offset: maps to
// the scalar-base + vector-offset load/store form (no per-lane 64-bit
// address arithmetic).  Mesh sizes are limited so that offsets fit 32 bits.
template <class T>
__device__ __forceinline__ const T& at(const T* base, unsigned i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * (unsigned)sizeof(T));
}
template <class T>
__device__ __forceinline__ T& at(T* base, unsigned i) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + i * (unsigned)sizeof(T));
}

// 3 i: one full-rate instruction (a product with 12 or 24 compiles to a
// 32-bit multiply, which takes four times as long).
__device__ __forceinline__ unsigned three_times(unsigned i) {
  unsigned t;
  asm("v_lshl_add_u32 %0, %1, 1, %1" : "=v"(t) : "v"(i));
  return t;
}
// Elements [N i, N i + N) of a uniform base pointer, N = 3 or 6, moved by the
// widest accesses (dword alignment is enough for them).
template <class T, int N>
struct Run {
  T v[N];
};
template <int N, class T>
__device__ __forceinline__ const Run<T, N>& run_at(const T* base, unsigned i) {
  static_assert(N == 3 || N == 6, "runs of three or six");
  return *reinterpret_cast<const Run<T, N>*>(reinterpret_cast<const char*>(base) +
                                            three_times(i) * (unsigned)(N / 3 * sizeof(T)));
}
template <int N, class T>
__device__ __forceinline__ Run<T, N>& run_at(T* base, unsigned i) {
  return const_cast<Run<T, N>&>(run_at<N>((const T*)base, i));
}

// LDS by byte address: base + SIZE * (the low or high half of w) in one
// instruction each (as shifts, masks and adds two to three).
#define APL_LDS __attribute__((address_space(3)))
template <class T, int N>
using Vx = T __attribute__((ext_vector_type(N)));
__device__ __forceinline__ unsigned lds_address(const void* p) {
  return (unsigned)(uintptr_t)(APL_LDS const char*)p;
}
template <class V>
__device__ __forceinline__ V lds_get(unsigned a) {
  return *(APL_LDS const V*)(uintptr_t)a;
}
// the first three of a padded vector
template <class T>
__device__ __forceinline__ V3<T> lds_get3(unsigned a) {
  if constexpr (sizeof(T) == 8) {
    const Vx<T, 2> w = lds_get<Vx<T, 2>>(a);  // (as one vector all 32 bytes are read)
    return v3(w[0], w[1], lds_get<T>(a + 16));
  } else {
    const Vx<T, 3> w = lds_get<Vx<T, 3>>(a);
    return v3(w[0], w[1], w[2]);
  }
}
template <class V>
__device__ __forceinline__ void lds_put(unsigned a, V v) {
  *(APL_LDS V*)(uintptr_t)a = v;
}
template <int SIZE, bool HIGH>
__device__ __forceinline__ unsigned lds_entry(unsigned w, unsigned base) {
  static_assert(SIZE >= 4 && SIZE <= 64, "inline constants");
  unsigned a;
  if constexpr (HIGH)
    asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(a) : "v"(w), "n"(SIZE), "s"(base));
  else
    asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(a) : "v"(w), "n"(SIZE), "s"(base));
  return a;
}

// Raw buffer loads: a scalar resource (base address) plus a per-lane and a
// uniform byte offset.  Used for the per-tet record so that no lane does
// 64-bit address arithmetic.  The resource's fourth word is the gfx9 raw
// buffer format; the record count is left unbounded (indices are exact).
using rsrc_t = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, -1, 0x00020000);
}
template <class R>
__device__ __forceinline__ R bload(rsrc_t r, unsigned voff, unsigned soff);
template <>
__device__ __forceinline__ float bload<float>(rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
template <>
__device__ __forceinline__ double bload<double>(rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ uint4 bload_u4(rsrc_t r, unsigned voff, unsigned soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// Per-tet record, loaded into registers ahead of the block's LDS staging.
template <class R>
struct TetRec {
  R B[9];
  R dV, mu, lam;
  R act[6];  // muscle activation
  uint4 cr;  // local slots (x, y), positions (z, w): two u16 per word
};

// Resources of one block's tet data.  dminv is SoA (row kk at kk * T), so its
// base moves with the block and the row offset kk * T * sizeof(R) stays
// below 2^32 bytes (mesh creation limits T accordingly).
struct BlockRes {
  rsrc_t dm, dv, mu, lam, act, cr;
  unsigned row, t0b;  // row stride and block start, in bytes of R
};

template <int MAT, class R, class X>
__device__ inline BlockRes block_res(const ElemArgs<R, X>& A, int t0) {
  BlockRes br;
  br.dm = make_rsrc(A.dminv + t0);
  br.dv = make_rsrc(A.dV);
  br.mu = make_rsrc(A.mu);
  br.lam = make_rsrc(MAT != MAT_ARAP ? A.lam : A.mu);
  br.act = make_rsrc(MAT == MAT_MUSCLE ? A.act + 6 * (size_t)t0 : A.mu);  // block-relative (T x 24 B may pass 2^32)
  br.cr = make_rsrc(A.corner);
  br.row = (unsigned)A.T * (unsigned)sizeof(R);
  br.t0b = (unsigned)t0 * (unsigned)sizeof(R);
  return br;
}

template <int MAT, class R>
__device__ inline void load_rec(const BlockRes& br, unsigned tl, TetRec<R>& r) {
  const unsigned vo = tl * (unsigned)sizeof(R);
#pragma unroll
  for (int kk = 0; kk < 9; ++kk) r.B[kk] = bload<R>(br.dm, vo, (unsigned)kk * br.row);
  r.dV = bload<R>(br.dv, vo, br.t0b);
  r.mu = bload<R>(br.mu, vo, br.t0b);
  r.lam = (MAT != MAT_ARAP) ? bload<R>(br.lam, vo, br.t0b) : R(0);
  if constexpr (MAT == MAT_MUSCLE) {
#pragma unroll
    for (int k = 0; k < 6; ++k) r.act[k] = bload<R>(br.act, 6u * vo + (unsigned)k * (unsigned)sizeof(R), 0u);
  }
  r.cr = bload_u4(br.cr, tl * 16u, br.t0b / (unsigned)sizeof(R) * 16u);
}

// Channel packing of the contribution buffer: one region per group of 4
// channels ([position][4]: one 16/32-byte LDS access per corner and per
// position), then a region for the remainder (a pair, a single channel, or
// 3 channels padded to 4).  Pass A's 6 channels take a 16-byte and an 8-byte
// access instead of six 4-byte ones.
template <int NCH>
struct Pack {
  static constexpr int G4 = NCH / 4;
  static constexpr int REM = NCH % 4;
  static constexpr int REMW = REM == 3 ? 4 : REM;  // stored width of the remainder
  static constexpr int NCHP = 4 * G4 + REMW;       // stored channels per position
};

// The accepted step at vertex v into u (new iterate) and d (new direction);
// the owner also writes them to the other buffer.  Every caller of a vertex
// gets the same values.
template <class R>
__device__ __forceinline__ void step_vertex(const Step<R>& t, unsigned v, bool owner, Vec4<double>& u, Vec4<R>& d) {
  const Vec4<double> xo = t.x0[v];
  const Vec4<R> pc = t.p0[v], g = t.g[v], P = t.P[v];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    u.v[c] = xo.v[c] + t.a * (double)pc.v[c];
    const R Pc = P.v[c] < R(0) ? t.ipm : P.v[c];
    d.v[c] = -Pc * g.v[c] + t.beta * pc.v[c];
  }
  u.v[3] = 0.0;
  d.v[3] = R(0);
  if (owner) {
    t.x1[v] = u;
    if (t.dir) t.p1[v] = d;
  }
}

// ... at the vertices no tet touches (no block stages them)
template <class R>
__device__ __forceinline__ void step_isolated(const SolveArgs<R>& S, const InstState* st) {
  for (int k = (int)blockIdx.x * NTH + (int)threadIdx.x; k < S.n_iso; k += (int)gridDim.x * NTH) {
    const InstState& s = st[S.iso_inst[k]];
    if (s.commit == 0) continue;
    Vec4<double> u;
    Vec4<R> d;
    step_vertex(Step<R>(S, s, s.cur), (unsigned)S.iso[k], true, u, d);
  }
}

// The CG direction of the iteration, likewise: d = z + beta d from the
// instance's other buffer into the current one.
template <class R>
struct Direction {
  R beta;
  const Vec4<R>* z;
  const Vec4<R>* d0;
  Vec4<R>* d1;
  template <class State>
  __device__ Direction(const SolveArgs<R>& S, const State& st, int cur)
      : beta((R)st.beta), z(S.z), d0(S.p + (cur ? (size_t)0 : S.V)), d1(S.p + (cur ? S.V : (size_t)0)) {}
};

template <class R>
__device__ __forceinline__ void direction_vertex(const Direction<R>& t, unsigned v, bool owner, Vec4<R>& d) {
  const Vec4<R> z = t.z[v], o = t.d0[v];
#pragma unroll
  for (int c = 0; c < 3; ++c) d.v[c] = z.v[c] + t.beta * o.v[c];
  d.v[3] = R(0);
  if (owner) t.d1[v] = d;
}

template <class R>
__device__ __forceinline__ void direction_isolated(const SolveArgs<R>& S, const InstState* st) {
  for (int k = (int)blockIdx.x * NTH + (int)threadIdx.x; k < S.n_iso; k += (int)gridDim.x * NTH) {
    const InstState& s = st[S.iso_inst[k]];
    if (s.act_eval == 0) continue;
    Vec4<R> d;
    direction_vertex(Direction<R>(S, s, s.cur), (unsigned)S.iso[k], true, d);
  }
}

// The scalar step before a pass, taken by every workgroup of a single
// instance's pass for itself.  A kernel of its own for one thread's decision
// costs a launch and a walk over the table by one CU (4.4 us each in a
// captured graph); here the pass grows by 1.5-2.3 us.  A PNCG iteration of a
// 10^3 cube went from 19.7 to 17.9 us, of a 32^3 ARAP cube from 35.5 to 31 us.
template <unsigned WHAT, class R>
__device__ __forceinline__ void scalar_step(const SolveArgs<R>& S, InstState* st, double* sm) {
  static_assert(sizeof(InstState) == 8 * STATE_DOUBLES, "state record");
  // every load before the first wait: the state (one double per thread) and the table
  const int t = threadIdx.x;
  double s_in = 0.0;
  if (t < STATE_DOUBLES) s_in = reinterpret_cast<const double*>(S.st)[t];
  if constexpr ((WHAT & W_TRIAL) != 0) {
    if (t < STATE_DOUBLES) reinterpret_cast<double*>(st)[t] = s_in;
    const double q = flat_sum_odd_short<SCAL_TH, NTH>(S.table, S.n_table, sm);
    if (t == 0) {
      InstState s = *st;
      pncg_alpha_step(s, S.prm, q);
      *st = s;
    }
  } else if constexpr ((WHAT & W_DIR) != 0) {
    if (t < STATE_DOUBLES) reinterpret_cast<double*>(st)[t] = s_in;
    flat_column_sums_short<N_DOTS, SCAL_TH, NTH>(S.table, S.n_table, sm);
    if (t == 0) {
      InstState s = *st;
      double tot[N_DOTS];
#pragma unroll
      for (int k = 0; k < N_DOTS; ++k) tot[k] = sm[k];
      if (s.act_eval != 0) pncg_scalar_step(s, S.prm, tot);
      *st = s;
    }
  } else {
    if (t < STATE_DOUBLES) reinterpret_cast<double*>(st)[t] = s_in;
    flat_column_sums_short<2, SCAL_TH, NTH>(S.table, S.n_table, sm);
    if (t == 0) {
      InstState s = *st;
      cg_beta_step(s, S.prm.rtol, S.prm.max_steps, sm[0], sm[1]);
      *st = s;
    }
  }
  __syncthreads();
  if (blockIdx.x == 0 && t < STATE_DOUBLES) reinterpret_cast<double*>(S.out)[t] = reinterpret_cast<double*>(st)[t];
}

// SPT: slot items per thread.  A block with nloc slots splits each slot's
// position range over tps = 4, 2 or 1 adjacent lanes (the most that fit
// SPT * NTH items), so all four waves share the sums; the lanes' interleaved
// partial sums are combined by a fixed xor-shuffle tree.
// LIST: the launch visits a list of blocks (a model mesh's law), else every
// block.  A separate instantiation: the list's lane-varying load in the
// block gather otherwise costs the scatter-free passes their next-block
// prefetch (the compiler's conservative memory waits, measured 17.5 ->
// 20.2 us for pass B).
template <int MAT, unsigned WHAT, class R, class X, int SPT, bool LIST, class SOLVE>
__device__ __forceinline__ void elem_body(const ElemArgs<R, X>& A, const SOLVE& S) {
  constexpr bool TRIAL = (WHAT & W_TRIAL) != 0;
  constexpr bool DIR = (WHAT & W_DIR) != 0;
  constexpr bool CGD = (WHAT & W_CGD) != 0;
  constexpr bool SOLVER = (WHAT & W_SOLVER) != 0;
  constexpr bool FUSED = (WHAT & W_FUSED) != 0;
  constexpr bool ONE = FUSED || (WHAT & W_ONE) != 0;  // the mesh has one instance
  static_assert(SOLVER == !std::is_same_v<SOLVE, NoSolve>, "solver passes take SolveArgs");
  constexpr bool HAS_G = (WHAT & W_G) != 0;
  constexpr bool HAS_H = (WHAT & W_H) != 0;
  constexpr bool HAS_HP = (WHAT & W_HP) != 0;
  constexpr int NCH = (HAS_G ? 3 : 0) + (HAS_H ? 3 : 0) + (HAS_HP ? 3 : 0);
  constexpr bool SCATTER = NCH > 0;
  constexpr int NCHA = NCH > 0 ? NCH : 1;
  constexpr bool NEEDV = (WHAT & (W_HP | W_HQ | W_MIX | W_MIXA)) != 0;
  constexpr bool RED_Q = (WHAT & (W_HQ | W_VQ)) != 0;
  constexpr bool RED = (WHAT & W_E) != 0 || RED_Q;
  constexpr int CS = 4 * NTH;  // channel stride of the contribution buffer
  static_assert(NCH <= MAX_CH, "too many channels");

  extern __shared__ double smem_d[];
  double* red = smem_d;  // wave partials of the block sums
  // the fused scalar step's state and, before the first block, its table sums
  InstState* st_lds = reinterpret_cast<InstState*>(smem_d + 8);
  constexpr int HEAD = 8 + (FUSED ? STATE_DOUBLES : 0);
  X* u_lds = reinterpret_cast<X*>(smem_d + HEAD);  // 4 per slot (padded)
  R* v_lds = reinterpret_cast<R*>(u_lds + 4 * A.nloc_max);
  R* contrib = v_lds + (NEEDV ? 4 * A.nloc_max : 0);  // [channel group][position][channel in group]
  using PK = Pack<NCHA>;

  // the same by LDS address: window slots and the two regions of the buffer
  // (groups of four channels, the remainder)
  const unsigned u_at = lds_address(u_lds), v_at = lds_address(v_lds), c_at = lds_address(contrib);
  constexpr int GB = 4 * sizeof(R), RB = PK::REMW * sizeof(R);  // bytes per position
  static_assert(PK::G4 <= 1, "one group of four channels");
  const unsigned r_at = c_at + PK::G4 * GB * CS;

  const int tid = threadIdx.x;
  const int pid = blockIdx.x;
  const int xcd = pid & 7, k0 = pid >> 3, K = gridDim.x >> 3;
  // XCD x owns the chunks x, x + 8, x + 16, ... of C consecutive blocks
  // (C up to XCD_CHUNK, smaller for small meshes so that every XCD gets
  // work): neighbouring blocks (which share vertices) mostly meet in one L2,
  // and every instance larger than 8 chunks spreads over all XCDs (a batch
  // whose few unconverged instances sat in one XCD's range would idle the
  // others).  The XCD's j-th block is xcd_block(j).
  const int nb = A.nblocks;
  const int C = nb / 64 < 1 ? 1 : (nb / 64 > XCD_CHUNK ? XCD_CHUNK : nb / 64);  // >= 8 chunks per XCD if possible
  const int nchunk = (nb + C - 1) / C;
  const int my_chunks = xcd < nchunk ? (nchunk - 1 - xcd) / 8 + 1 : 0;
  const bool owns_last = my_chunks > 0 && (nchunk - 1) % 8 == xcd;
  const int nb_x = my_chunks * C - (owns_last ? nchunk * C - nb : 0);
  auto xcd_block = [&](int j) {
    const int k = ((j / C) * 8 + xcd) * C + j % C;
    if constexpr (LIST)
      return constant_at(A.blk_list, k);
    else
      return k;
  };

  // This workgroup's blocks are xcd_block(k0 + j K), j < n_cand; in a solve
  // only those of still-active instances.
  const int n_cand = k0 < nb_x ? (nb_x - k0 + K - 1) / K : 0;
  bool filter = false;
  InstScalars single;  // the instance's scalars (ONE)
  // the vertex of slot s of the block whose slots start at sb (with OWNER_BIT
  // where the pass needs it)
  auto slot_vertex = [&](int sb, int s) -> uint32_t {
    if constexpr (DIR || CGD)
      return at(S.own + sb, (unsigned)s);
    else
      return (uint32_t)at(A.loc_gid + sb, (unsigned)s);
  };
  // FUSED: the first block's tables, records and slot vertices are loaded
  // before the scalar step, whose sums and barriers hide their latency
  int pre_b = -1;
  uint32_t pre_o = 0u;
  TetRec<R> pre_rec;
  if constexpr (FUSED) {
    if (n_cand > 0) {
      pre_b = xcd_block(k0);
      const int t0 = constant_at(A.blk_tet_off, pre_b), t1 = constant_at(A.blk_tet_off, pre_b + 1);
      const int sb = constant_at(A.blk_loc_off, pre_b), sb1 = constant_at(A.blk_loc_off, pre_b + 1);
      pre_o = slot_vertex(sb, min(tid, sb1 - sb - 1));
      load_rec<MAT>(block_res<MAT>(A, t0), (unsigned)min(tid, t1 - t0 - 1), pre_rec);
    }
    scalar_step<WHAT>(S, st_lds, smem_d + HEAD);
    if constexpr (DIR) step_isolated(S, st_lds);
    if constexpr (CGD) direction_isolated(S, st_lds);
    single = InstScalars(*st_lds);
    if ((DIR ? single.commit : single.act_eval) == 0) return;
  } else if constexpr (SOLVER) {
    if constexpr (DIR) step_isolated(S, S.st);
    if constexpr (CGD) direction_isolated(S, S.st);
    if constexpr (ONE) {
      single = InstScalars(constant_at(S.st, 0));
      if ((DIR ? single.commit : single.act_eval) == 0) return;
    } else {
      filter = S.filter != 0;
      if (!filter && (DIR ? S.st[0].commit : S.st[0].act_eval) == 0) return;
    }
  }
  // the active-block list (solves only) sits after the contribution buffer
  int* act_list = reinterpret_cast<int*>(contrib + (SCATTER ? PK::NCHP * CS : 0));
  // Passes without a scatter phase have registers to spare: each thread
  // loads the next block's staging inputs (its slot tid) while the current
  // block finishes, so that block's staging waits on no global load.  Not in
  // the scatter passes, where the registers cost a wave per SIMD and the gain
  // disappears (measured), nor in the solver's, which stage other records.
  constexpr bool PREFETCH = !SCATTER && !SOLVER;
  int pf_b = -1;
  X pf_x[3] = {X(0), X(0), X(0)};
  R pf_p[3] = {R(0), R(0), R(0)};
  for_active<NTH>(
      n_cand, filter, act_list, [&](int j) { return xcd_block(k0 + j * K); },
      [&](int bb) {
        if constexpr (SOLVER) {
          const InstState& st = S.st[A.blk_inst[bb]];  // (bb differs by lane)
          return (DIR ? st.commit : st.act_eval) != 0;
        }
        return true;
      },
      [&](const int b, const int bn) {
      // the scalars of the block's instance
      const auto& inst = [&]() -> const auto& {
        if constexpr (ONE)
          return single;
        else if constexpr (SOLVER)
          return S.st[A.blk_inst[b]];
        else
          return S;
      }();
      // Everything a block reads that does not depend on another load of it is
      // started here, without a branch between: the tables by scalar loads, then
      // the thread's slot vertex, its tet record and the destinations of its
      // slot partials (idle threads read the block's last entries), so the
      // staging waits for the slot vertex alone.  With the destinations first
      // and each load under its own branch a block took five memory latencies
      // in turn, now three: 51^3 H v 27.6 -> 25.9 us, FP64 pass at 37^3 25.9 ->
      // 24.4 us, 64^3 solve 55.6 -> 53.1 ms.  The positions of the slots come
      // along (looked up after the staging they were a latency of their own);
      // with that, fewer address instructions and one barrier less per block
      // 51^3 H v 25.8 -> 22.6 us, 45^3 muscle 22.0 -> 20.1, 64^3 SNH 40.7 -> 39.1,
      // ARAP 52.3 -> 50.5 (whole evaluations).
      const int t0 = constant_at(A.blk_tet_off, b), t1 = constant_at(A.blk_tet_off, b + 1);
      const int sb = constant_at(A.blk_loc_off, b), sb1 = constant_at(A.blk_loc_off, b + 1);
      const int co_off = SCATTER ? constant_at(A.blk_co_off, b) : 0;
      const int nt = t1 - t0, nloc = sb1 - sb;
      const int lg = (4 * nloc <= SPT * NTH) ? 2 : ((2 * nloc <= SPT * NTH) ? 1 : 0);
      const int tps = 1 << lg;
      // which of its two buffers the instance is in: the staging's addresses wait for it
      int cur = 0;
      if constexpr (TRIAL || DIR || CGD) cur = inst.cur;
      const BlockRes br = block_res<MAT>(A, t0);
      uint32_t o0 = pre_o;
      TetRec<R> rec;
      if (FUSED && b == pre_b) {
        rec = pre_rec;
      } else {
        o0 = slot_vertex(sb, min(tid, nloc - 1));
        __builtin_amdgcn_sched_barrier(0);  // this load first: the staging waits for it alone
        load_rec<MAT>(br, (unsigned)min(tid, nt - 1), rec);
      }
      int dst_pre[SPT];
      uint32_t run_pre[SPT];  // the first chunk's positions of the slot item: [low half, high half)
      const uint16_t* co = A.chunk_off + co_off;
      auto slot_run = [&](const uint16_t* cc, int s) {
        uint32_t w;
        __builtin_memcpy(&w, &at(cc, (unsigned)s), sizeof(w));  // entries s and s + 1
        return w;
      };
      if constexpr (SCATTER) {
#pragma unroll
        for (int k = 0; k < SPT; ++k) {
          const int s = min((tid + k * NTH) >> lg, nloc - 1);
          dst_pre[k] = at(A.loc_dst + sb, (unsigned)s);
          run_pre[k] = slot_run(co, s);
        }
      }
      // (a lane's own value from here: made uniform where it is loaded, it is waited for there)
      if constexpr (SOLVER && !ONE) asm("" : "+v"(cur));

      // stage the block's vertex window (u = x + alpha p for a trial point; the
      // new iterate and direction for an accepted step): stage(slot, o), o its
      // vertex as slot_vertex gives it
      auto put_u = [&](int s, const Vec4<X>& u4) { *reinterpret_cast<Vec4<X>*>(u_lds + 4 * s) = u4; };
      auto put_v = [&](int s, const Vec4<R>& v4) { *reinterpret_cast<Vec4<R>*>(v_lds + 4 * s) = v4; };
      auto window = [&](auto stage) {
        // the thread's first slot apart from the others, or the wait at the
        // loop's head would be for the tet records too; and neither a vertex
        // nor cur is ever all ones: asked here, so that their loads are not
        // moved down into this branch, behind the others
        if ((tid < nloc) & (o0 != ~0u) & (cur != -1)) {
          stage(tid, o0);
          for (int s = tid + NTH; s < nloc; s += NTH) stage(s, slot_vertex(sb, s));
        }
      };
      if constexpr (DIR) {
        const Step<R> step(S, inst, cur);
        window([&](int s, uint32_t o) {
          Vec4<X> u4;
          Vec4<R> v4;
          step_vertex(step, o & ~OWNER_BIT, (o & OWNER_BIT) != 0, u4, v4);
          put_u(s, u4);
          put_v(s, v4);
        });
        if (!step.dir) return;  // converged at this step: no new direction
      } else if constexpr (CGD) {
        const Direction<R> dir(S, inst, cur);
        window([&](int s, uint32_t o) {
          const unsigned v = o & ~OWNER_BIT;
          const auto xv = run_at<3>(A.x, v);
          const Vec4<X> u4 = {{xv.v[0], xv.v[1], xv.v[2], X(0)}};
          Vec4<R> v4;
          direction_vertex(dir, v, (o & OWNER_BIT) != 0, v4);
          put_u(s, u4);
          put_v(s, v4);
        });
      } else if constexpr (TRIAL) {
        const double alpha = inst.alpha;
        const Vec4<double>* xb = S.x + (cur ? S.V : (size_t)0);
        const Vec4<R>* pb = S.p + (cur ? S.V : (size_t)0);
        window([&](int s, uint32_t o) {
          const size_t v = o;
          Vec4<double> u4 = xb[v];
          const Vec4<R> p4 = pb[v];
#pragma unroll
          for (int c = 0; c < 3; ++c) u4.v[c] += alpha * (double)p4.v[c];
          put_u(s, u4);
        });
      } else {
        window([&](int s, uint32_t o) {
          X ux, uy, uz;
          R px = R(0), py = R(0), pz = R(0);
          if (PREFETCH && s == tid && pf_b == b) {
            ux = pf_x[0];
            uy = pf_x[1];
            uz = pf_x[2];
            px = pf_p[0];
            py = pf_p[1];
            pz = pf_p[2];
          } else if constexpr (PREFETCH) {
            // (a load per component, as the prefetch: one for all three lands in
            // registers of its own, and the prefetched values would be waited
            // for where they are loaded, to be moved there: 64^3 v.Hv 22.1 ->
            // 26.3 us)
            const unsigned g3 = 3u * o;
            ux = at(A.x, g3);
            uy = at(A.x, g3 + 1);
            uz = at(A.x, g3 + 2);
            if constexpr (NEEDV) {
              px = at(A.p, g3);
              py = at(A.p, g3 + 1);
              pz = at(A.p, g3 + 2);
            }
          } else {
            const auto xv = run_at<3>(A.x, o);
            ux = xv.v[0];
            uy = xv.v[1];
            uz = xv.v[2];
            if constexpr (NEEDV) {
              const auto pv = run_at<3>(A.p, o);
              px = pv.v[0];
              py = pv.v[1];
              pz = pv.v[2];
            }
          }
          put_u(s, Vec4<X>{{ux, uy, uz, X(0)}});
          if constexpr (NEEDV) put_v(s, Vec4<R>{{px, py, pz, R(0)}});
        });
      }
      __syncthreads();

      R acc[SPT][NCHA];
#pragma unroll
      for (int k = 0; k < SPT; ++k)
#pragma unroll
        for (int ch = 0; ch < NCHA; ++ch) acc[k][ch] = R(0);
      R e_acc = R(0);
      // (v.Hv of the CG comes in FP64 and is added up in it: the step length
      // hangs on it, and the unclamped forms of the tets cancel)
      std::conditional_t<(WHAT & W_VQ) != 0, double, R> q_acc = 0;
      // one FP64 partial per wave and column into LDS, added in a fixed order
      // by one thread after the next barrier
      auto wave_partials = [&]() {
        const int lane = tid & 63, w = tid >> 6;
        if constexpr ((WHAT & W_E) != 0) {
          const double e = wave_sum((double)e_acc);
          if (lane == 63) red[2 * w] = e;
        }
        if constexpr (RED_Q) {
          const double q = wave_sum((double)q_acc);
          if (lane == 63) red[2 * w + 1] = q;
        }
      };
      // before the sums of the slots, where its chain overlaps the LDS writes
      // (64^3 SNH 39.75 -> 39.4 us), but not when the waves come to that
      // barrier at different times (ARAP: 50.3 us after them, 51.2 before)
      constexpr bool EARLY_RED = RED && SCATTER && MAT != MAT_ARAP;
      const int nchunks = (nt + NTH - 1) / NTH;
      for (int c = 0; c < nchunks; ++c) {
        const int tl = c * NTH + tid;
        // this chunk's position ranges of the thread's slot items
        uint32_t runs[SPT];
        if constexpr (SCATTER) {
#pragma unroll
          for (int k = 0; k < SPT; ++k)
            runs[k] = c == 0 ? run_pre[k] : slot_run(co + c * (nloc + 1), min((tid + k * NTH) >> lg, nloc - 1));
        }
        if (tl < nt) {
          if (c > 0) load_rec<MAT>(br, (unsigned)tl, rec);
          const TetGeom<R> g = make_geom(rec.B, rec.dV);
          // edge differences u_a - u_0 in the storage precision X, then R: F - I
          // depends only on them, and forming them before rounding keeps F
          // accurate relative to the strain rather than to |u|.
          constexpr int XB = 4 * sizeof(X), VB = 4 * sizeof(R);  // bytes per window slot
          const unsigned ua[4] = {lds_entry<XB, false>(rec.cr.x, u_at), lds_entry<XB, true>(rec.cr.x, u_at),
                                  lds_entry<XB, false>(rec.cr.y, u_at), lds_entry<XB, true>(rec.cr.y, u_at)};
          V3<X> uc[4];
#pragma unroll
          for (int a = 0; a < 4; ++a) uc[a] = lds_get3<X>(ua[a]);
          V3<R> u[4], v[4];
#pragma unroll
          for (int a = 0; a < 4; ++a) {
            u[a] = v3((R)(uc[a].x - uc[0].x), (R)(uc[a].y - uc[0].y), (R)(uc[a].z - uc[0].z));
            if constexpr (NEEDV) {
              const uint32_t w = a < 2 ? rec.cr.x : rec.cr.y;
              v[a] = lds_get3<R>(a % 2 ? lds_entry<VB, true>(w, v_at) : lds_entry<VB, false>(w, v_at));
            } else {
              v[a] = v3(R(0), R(0), R(0));
            }
          }
          TetOut<R> o;
          tet_eval<MAT, WHAT & W_OUT, R>(g, rec.mu, rec.lam, rec.act, u, v, o);
          if constexpr ((WHAT & W_E) != 0) e_acc += o.e;
          if constexpr ((WHAT & W_HQ) != 0) q_acc += o.hq;
          if constexpr ((WHAT & W_VQ) != 0) q_acc += o.vq;
          if constexpr ((WHAT & W_MIX) != 0) {
            R* oa = A.out_a + t0;
            R* ob = A.out_b + t0;
            if (A.accumulate) {
              at(oa, (unsigned)tl) += o.dmu;
              if (MAT != MAT_ARAP) at(ob, (unsigned)tl) += o.dlam;
            } else {
              at(oa, (unsigned)tl) = o.dmu;
              if (MAT != MAT_ARAP) at(ob, (unsigned)tl) = o.dlam;
            }
          }
          if constexpr ((WHAT & W_MIXA) != 0) {
            R* oc = A.out_c + 6 * (size_t)t0;
#pragma unroll
            for (int k = 0; k < 6; ++k) {
              if (A.accumulate)
                at(oc, 6u * (unsigned)tl + (unsigned)k) += o.dact[k];
              else
                at(oc, 6u * (unsigned)tl + (unsigned)k) = o.dact[k];
            }
          }
          if constexpr (SCATTER) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
              R vals[NCHA];
              int ch = 0;
              if constexpr (HAS_G) {
                vals[ch + 0] = o.g[a].x;
                vals[ch + 1] = o.g[a].y;
                vals[ch + 2] = o.g[a].z;
                ch += 3;
              }
              if constexpr (HAS_H) {
                vals[ch + 0] = o.h[a].x;
                vals[ch + 1] = o.h[a].y;
                vals[ch + 2] = o.h[a].z;
                ch += 3;
              }
              if constexpr (HAS_HP) {
                vals[ch + 0] = o.hp[a].x;
                vals[ch + 1] = o.hp[a].y;
                vals[ch + 2] = o.hp[a].z;
              }
              const uint32_t w = a < 2 ? rec.cr.z : rec.cr.w;  // the corner's position
              if constexpr (PK::G4 > 0)
                lds_put(a % 2 ? lds_entry<GB, true>(w, c_at) : lds_entry<GB, false>(w, c_at),
                        Vx<R, 4>{vals[0], vals[1], vals[2], vals[3]});
              constexpr int c0 = 4 * PK::G4;
              if constexpr (PK::REM > 0) {
                const unsigned ra = a % 2 ? lds_entry<RB, true>(w, r_at) : lds_entry<RB, false>(w, r_at);
                if constexpr (PK::REM == 3)
                  lds_put(ra, Vx<R, 4>{vals[c0], vals[c0 + 1], vals[c0 + 2], R(0)});
                else if constexpr (PK::REM == 2)
                  lds_put(ra, Vx<R, 2>{vals[c0], vals[c0 + 1]});
                else
                  lds_put(ra, vals[c0]);
              }
            }
          }
        }
        if constexpr (EARLY_RED)
          if (c == nchunks - 1) wave_partials();
        if constexpr (SCATTER) __syncthreads();
        if constexpr (SCATTER) {
          // one position's channels: a 4-channel group per 16/32-byte load, then the remainder
          auto load_pos = [&](unsigned ga, unsigned ra, R (&t)[PK::NCHP]) {
            if constexpr (PK::G4 > 0) {
              const Vx<R, 4> w = lds_get<Vx<R, 4>>(ga);
#pragma unroll
              for (int i = 0; i < 4; ++i) t[i] = w[i];
            }
            constexpr int c0 = 4 * PK::G4;
            if constexpr (PK::REM == 3) {
              const V3<R> w = lds_get3<R>(ra);
              t[c0] = w.x;
              t[c0 + 1] = w.y;
              t[c0 + 2] = w.z;
            } else if constexpr (PK::REM == 2) {
              const Vx<R, 2> w = lds_get<Vx<R, 2>>(ra);
              t[c0] = w[0];
              t[c0 + 1] = w[1];
            } else if constexpr (PK::REM == 1) {
              t[c0] = lds_get<R>(ra);
            }
          };
#pragma unroll
          for (int k = 0; k < SPT; ++k) {
            const int item = tid + k * NTH;
            const bool mine = (item >> lg) < nloc;
            const int q = mine ? (int)(runs[k] & 0xffffu) + (item & (tps - 1)) : 0;
            const int q1 = mine ? (int)(runs[k] >> 16) : 0;
            // two positions per step, both loads first, each with its own address
            // (they advance by a uniform stride); the sums keep the sequential order
            int n = q1 - q;
            unsigned ga = c_at + (unsigned)GB * (unsigned)q, ra = r_at + (unsigned)RB * (unsigned)q;
            unsigned gb = ga + (unsigned)GB * tps, rb = ra + (unsigned)RB * tps;
            for (; n > tps; n -= 2 * tps) {
              R ta[PK::NCHP], tb[PK::NCHP];
              load_pos(ga, ra, ta);
              load_pos(gb, rb, tb);
              ga += 2 * GB * tps;
              gb += 2 * GB * tps;
              ra += 2 * RB * tps;
              rb += 2 * RB * tps;
#pragma unroll
              for (int ch = 0; ch < NCH; ++ch) acc[k][ch] = (acc[k][ch] + ta[ch]) + tb[ch];
            }
            if (n > 0) {
              R ta[PK::NCHP];
              load_pos(ga, ra, ta);
#pragma unroll
              for (int ch = 0; ch < NCH; ++ch) acc[k][ch] += ta[ch];
            }
          }
        }
        if constexpr (RED && SCATTER && !EARLY_RED)
          if (c == nchunks - 1) wave_partials();
        if constexpr (SCATTER) __syncthreads();
      }

      if constexpr (PREFETCH) {
        if (bn >= 0) {
          const int sb_n = constant_at(A.blk_loc_off, bn);
          const int nloc_n = constant_at(A.blk_loc_off, bn + 1) - sb_n;
          pf_b = bn;
          if (tid < nloc_n) {
            const unsigned g3 = 3u * (unsigned)at(A.loc_gid + sb_n, (unsigned)tid);
            pf_x[0] = at(A.x, g3);
            pf_x[1] = at(A.x, g3 + 1);
            pf_x[2] = at(A.x, g3 + 2);
            if constexpr (NEEDV) {
              pf_p[0] = at(A.p, g3);
              pf_p[1] = at(A.p, g3 + 1);
              pf_p[2] = at(A.p, g3 + 2);
            }
          }
        }
      }
      if constexpr (SCATTER) {
        // combine the lanes of a slot, then one partial per slot, at the
        // slot's place in the vertex-major order
        if (lg > 0) {
#pragma unroll
          for (int k = 0; k < SPT; ++k)
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) acc[k][ch] += dpp<R, DPP_QUAD_XOR1>(acc[k][ch]);
        }
        if (lg > 1) {
#pragma unroll
          for (int k = 0; k < SPT; ++k)
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) acc[k][ch] += dpp<R, DPP_QUAD_XOR2>(acc[k][ch]);
        }
#pragma unroll
        for (int k = 0; k < SPT; ++k) {
          const int item = tid + k * NTH;
          const int s = item >> lg;
          if (s < nloc && (item & (tps - 1)) == 0) {
            // (by element: a store of the whole record could be one to the block
            // tables for all the compiler knows, whose loads would no longer be scalar)
            auto& sums = run_at<NCH>(A.partial, (unsigned)dst_pre[k]);
#pragma unroll
            for (int ch = 0; ch < NCH; ++ch) sums.v[ch] = acc[k][ch];
          }
        }
      }
      if constexpr (RED && !SCATTER) {  // behind the prefetch, whose latency this hides
        wave_partials();
        __syncthreads();
      }
      if constexpr (RED) {
        if (tid == NTH - 64) {  // of the last wave, whose lanes have the fewest slots
#pragma unroll
          for (int col = 0; col < 2; ++col) {
            if (col == 0 && (WHAT & W_E) == 0) continue;
            if (col == 1 && !RED_Q) continue;
            double r = 0.0;
#pragma unroll
            for (int ww = 0; ww < NTH / 64; ++ww) r += red[2 * ww + col];
            if constexpr (DIR || CGD)
              S.hq[b] = r;
            else
              A.blk_red[(size_t)RED_STRIDE * b + col] = r;
          }
        }
      }
      // The next block's window may overwrite this one's: its readers are past
      // the barrier after the tets (the mixed passes have none).  The wave
      // partials and the contributions are written again only after the next
      // window's barrier.
      if constexpr (!SCATTER && !RED) __syncthreads();
      });
}

template <int MAT, unsigned WHAT, class R, class X, int SPT, bool LIST>
__global__ __launch_bounds__(NTH) void elem_kernel(ElemArgs<R, X> A) {
  elem_body<MAT, WHAT, R, X, SPT, LIST>(A, NoSolve{});
}

template <int MAT, unsigned WHAT, class R, class X, int SPT, bool LIST>
__global__ __launch_bounds__(NTH) void solve_elem_kernel(ElemArgs<R, X> A, SolveArgs<R> S) {
  elem_body<MAT, WHAT, R, X, SPT, LIST>(A, S);
}


// ------------------------------------------------------------------ launchers

template <class R, class X>
static ElemArgs<R, X> make_args(apl_mesh* m, const void* mu, const void* lam, const void* x, const void* p,
                                void* out_a, void* out_b, int accumulate, void* out_c, const Workspace* ws) {
  ElemArgs<R, X> A;
  A.dminv = (const R*)m->d.dminv;
  A.dV = (const R*)m->d.dV;
  A.corner = (const uint4*)m->d.corner;
  A.blk_tet_off = m->d.blk_tet_off;
  A.blk_loc_off = m->d.blk_loc_off;
  A.blk_inst = m->d.blk_inst;
  A.loc_gid = m->d.loc_gid;
  A.loc_dst = m->d.loc_dst;
  A.blk_co_off = m->d.blk_co_off;
  A.chunk_off = m->d.chunk_off;
  A.mu = (const R*)mu;
  A.lam = (const R*)lam;
  A.act = (const R*)m->activation;
  A.x = (const X*)x;
  A.p = (const R*)p;
  A.out_a = (R*)out_a;
  A.out_b = (R*)out_b;
  A.out_c = (R*)out_c;
  A.partial = (R*)(ws != nullptr ? ws->partial : m->d.partial);
  A.blk_red = ws != nullptr ? ws->blk_red : m->d.blk_red;
  A.T = (int)m->L.T;
  A.blk_list = nullptr;
  A.nblocks = (int)m->L.nblocks;
  A.nloc_max = m->L.nloc_max;
  A.accumulate = accumulate;
  return A;
}

// LDS of one element workgroup: wave partials, the vertex window (u in X,
// v in R when the pass needs it, 4 lanes per slot), the packed contribution
// buffer of the scatter passes and, in solves, the active-block list.
template <unsigned WHAT, class R, class X>
constexpr size_t smem_bytes_n(int nloc_max, bool filtered) {
  constexpr bool NEEDV = (WHAT & (W_HP | W_HQ | W_MIX | W_MIXA)) != 0;
  constexpr int NCH = ((WHAT & W_G) ? 3 : 0) + ((WHAT & W_H) ? 3 : 0) + ((WHAT & W_HP) ? 3 : 0);
  size_t n = 4 * (size_t)nloc_max * (sizeof(X) + (NEEDV ? sizeof(R) : 0));
  n += sizeof(R) * (size_t)(NCH > 0 ? Pack<NCH>::NCHP : 0) * 4 * NTH;
  if ((WHAT & W_FUSED) != 0) {
    if (n < SUMS_LDS) n = SUMS_LDS;  // the fused scalar step's sums share the window's space
    n += STATE_DOUBLES * sizeof(double);
  }
  n += 8 * sizeof(double);
  if (filtered) n += sizeof(int) * NTH;  // active-block list
  return n;
}

template <int MAT, unsigned WHAT, class R, class X>
static size_t smem_bytes(const apl_mesh* m, bool filtered) {
  return smem_bytes_n<WHAT, R, X>(m->L.nloc_max, filtered);
}

// blocks one launch of law MAT visits (model meshes: the law's own blocks)
inline int64_t launch_blocks(const apl_mesh* m, int mat) { return m->model ? m->law_nblk[mat] : m->L.nblocks; }

// Default element grid per pass, percent of occupancy x CUs: one resident
// round of persistent workgroups, except for the VALU-heavy ARAP gradient
// passes (4 waves per SIMD) and the Hessian-vector pass, which run faster
// with a second, non-resident round that the hardware dispatches as
// workgroups of the first finish (a dynamic balance of the last blocks).
// Whole FP32 evaluations, us at 100 / 200: 64^3 ARAP E, g, diag H 49.2 / 45.6,
// H v of SNH 28.0 / 27.7, muscle 33.0 / 30.1, ARAP 39.1 / 38.2; at 45^3 (1,780
// blocks) all equal but ARAP's H v, 19.2 / 20.9.  The passes left at 100 gain
// up to 5 % from 200 at 64^3 now that a block takes fewer latencies (SNH
// E, g, diag H 33.1 / 31.8, muscle 38.6 / 36.8, v.Hv of SNH 22.2 / 21.8, ARAP
// 31.1 / 30.0) and nothing to 32^3; the autotuner chooses per mesh.
constexpr int default_grid_pct(int mat, unsigned what) {
  return ((what & W_HP) != 0 || (mat == MAT_ARAP && (what & (W_G | W_H)) != 0)) ? 200 : 100;
}

// the kernel of one pass variant
template <int MAT, unsigned WHAT, class R, class X, int SPT, bool LIST>
constexpr auto pass_kernel() {
  if constexpr ((WHAT & W_SOLVER) != 0)
    return &solve_elem_kernel<MAT, WHAT, R, X, SPT, LIST>;
  else
    return &elem_kernel<MAT, WHAT, R, X, SPT, LIST>;
}

// row of a pass variant in the mesh's grid cache
constexpr int variant_index(unsigned what) {
  constexpr unsigned v[N_VARIANTS] = {W_E, W_E | W_G | W_H, W_G, W_H, W_HP, W_HQ, W_MIX, W_MIXA, W_MIX | W_MIXA,
                                      W_E | W_G | W_H | W_TRIAL, W_HQ | W_DIR, W_HP | W_VQ | W_CGD, W_HP | W_ACT,
                                      W_E | W_G | W_H | W_TRIAL | W_ONE, W_HQ | W_DIR | W_ONE,
                                      W_E | W_G | W_H | W_TRIAL | W_FUSED, W_HQ | W_DIR | W_FUSED,
                                      W_HP | W_VQ | W_CGD | W_FUSED};
  for (int i = 0; i < N_VARIANTS; ++i)
    if (v[i] == what) return i;
  return -1;
}

template <int MAT, unsigned WHAT, class R, class X, int SPT>
static int grid_for_spt(apl_mesh* m, bool filtered) {
  static_assert(variant_index(WHAT) >= 0, "pass variant without a grid cache entry");
  int& cached = m->grid_cache[MAT][2 * variant_index(WHAT) + (filtered ? 1 : 0)];
  if (cached > 0) return cached;
  const size_t smem = smem_bytes<MAT, WHAT, R, X>(m, filtered);
  int occ = 0;
  const hipError_t oe =
      m->model
          ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, pass_kernel<MAT, WHAT, R, X, SPT, true>(), NTH, smem)
          : hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, pass_kernel<MAT, WHAT, R, X, SPT, false>(), NTH, smem);
  if (oe != hipSuccess || occ < 1)
    occ = 1;
  const int pct = m->grid_pct > 0 ? m->grid_pct : default_grid_pct(MAT, WHAT);
  long long g = (long long)occ * m->n_cu * pct / 100;
  long long nb8 = ((launch_blocks(m, MAT) + 7) / 8) * 8;
  if (g > nb8) g = nb8;
  g = ((g + 7) / 8) * 8;
  if (g < 8) g = 8;
  cached = (int)g;
  return cached;
}

// slots per thread for this mesh's largest block window
inline int spt_for(const apl_mesh* m) { return m->L.nloc_max <= NTH ? 1 : (m->L.nloc_max <= 2 * NTH ? 2 : 4); }

// SPT of a pass variant on this mesh as a constant: go(integral_constant)
template <unsigned WHAT, class Go>
static int with_spt(const apl_mesh* m, Go go) {
  constexpr bool SCATTER = (WHAT & (W_G | W_H | W_HP)) != 0;
  if constexpr (SCATTER) {
    const int spt = spt_for(m);
    if (spt == 2) return go(std::integral_constant<int, 2>{});
    if (spt == 4) return go(std::integral_constant<int, 4>{});
  }
  return go(std::integral_constant<int, 1>{});
}

template <int MAT, unsigned WHAT, class R, class X>
static int grid_for(apl_mesh* m, bool filtered) {
  return with_spt<WHAT>(m, [&](auto spt) { return grid_for_spt<MAT, WHAT, R, X, decltype(spt)::value>(m, filtered); });
}

// One launch of a pass variant over law MAT's blocks.  `more`: the kernel's
// arguments after ElemArgs (SolveArgs of the solver's passes).
template <int MAT, unsigned WHAT, class R, class X, class... More>
static int launch_pass(apl_mesh* m, ElemArgs<R, X> A, bool filtered, int grid_override, hipStream_t s, More... more) {
  const size_t smem = smem_bytes<MAT, WHAT, R, X>(m, filtered);
  if (smem > ELEM_LDS_MAX) {
    set_error("element block needs more than 64 KiB of LDS (block window above the mesh's nloc cap)");
    return -1;
  }
  const int grid = grid_override > 0 ? ((grid_override + 7) / 8) * 8 : grid_for<MAT, WHAT, R, X>(m, filtered);
  if (m->model) {
    A.blk_list = m->d.law_blk[MAT];
    A.nblocks = (int)m->law_nblk[MAT];
  }
  with_spt<WHAT>(m, [&](auto spt) {
    constexpr int SPT = decltype(spt)::value;
    if (m->model)
      hipLaunchKernelGGL((pass_kernel<MAT, WHAT, R, X, SPT, true>()), dim3(grid), dim3(NTH), smem, s, A, more...);
    else
      hipLaunchKernelGGL((pass_kernel<MAT, WHAT, R, X, SPT, false>()), dim3(grid), dim3(NTH), smem, s, A, more...);
    return 0;
  });
  APL_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace apl
