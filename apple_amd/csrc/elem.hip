// Element passes of the C ABI: launches of the element kernel (elem_kernel.h)
// over the caller's displacements, the finish pass that sums the slot
// partials per vertex, and the allocation-free entry point.
#include "elem_kernel.h"
#include "flatsum.h"
#include "vsum.h"

#include <mutex>
#include <string>

namespace apl {

// Finish pass of an element pass, one launch: workgroups [0, ninst) sum one
// instance's block energies / quadratic forms in a fixed order (first, so
// their longer loops start early); workgroups [ninst, ninst + nvblk) form
// the vertex sums of the slot partials over an instance-aligned vertex
// block, one degree of freedom per thread and stride (ascending block order
// per vertex).
template <class R>
struct FinishArgs {
  const int32_t* vblk_off;
  const int32_t* vtx_slot_off;
  const R* partial;
  R* out_a;
  R* out_b;
  const double* blk_red;
  const int64_t* inst_blk_off;
  double* out_e;
  double* out_q;
  int ninst;  // instance workgroups (0: no energies / quadratic forms)
  int h_only;
  int accumulate;
  int n_verts;
};

// The vertex sums wait for one chain, offsets -> partials -> sums.  FP32
// passes of six channels on meshes of up to two vertex blocks per CU have all
// of a thread's loads of the partials in flight at once (WINDOW).  Whole SNH
// evaluations, us, with the loop of four / with the window: 141 vertex blocks
// 12.3 / 11.3, 381 19.2 / 18.3, 489 20.9 / 20.1, 519 21.3 / 20.8, 724 24.9 / 24.5,
// 887 28.5 / 28.5, 1,073 32.0-32.3 / 32.3; with three channels or in FP64 the
// loop is 0.2-0.4 us faster.  With one instance (SINGLE) the block's vertices
// follow from its number.
template <class R, int NCH, bool SINGLE, bool WINDOW>
__global__ __launch_bounds__(NTH) void finish_kernel(FinishArgs<R> A) {
  __shared__ double eq[2 * (NTH / 64 + 1)];
  if ((int)blockIdx.x < A.ninst) {
    const int i = (int)blockIdx.x;
    const long long b0 = A.inst_blk_off[i];
    flat_column_sums<2, NTH>(A.blk_red + RED_STRIDE * b0, RED_STRIDE * (A.inst_blk_off[i + 1] - b0), eq);
    if (threadIdx.x == 0) {
      if (A.out_e != nullptr) A.out_e[i] = A.accumulate ? A.out_e[i] + eq[0] : eq[0];
      if (A.out_q != nullptr) A.out_q[i] = A.accumulate ? A.out_q[i] + eq[1] : eq[1];
    }
    return;
  }
  if constexpr (NCH > 0) {
    const int vb = (int)blockIdx.x - A.ninst;
    __shared__ R win[VSUM_LDS_BYTES / sizeof(R)];
    const int v0 = SINGLE ? vb * NTH : A.vblk_off[vb];
    const int v1 = SINGLE ? min(v0 + NTH, A.n_verts) : A.vblk_off[vb + 1];
    const int i0 = 3 * v0, i1 = 3 * v1;
    VertexSums<R, NCH, NTH> vs{A.vtx_slot_off, A.partial, win};
    typename VertexSums<R, NCH, NTH>::template Window<16> w;
    if constexpr (WINDOW) vs.fetch(v0, v1, VSUM_LDS_BYTES / (int)sizeof(R), w);
    int k0[DOF_PER_THREAD], k1[DOF_PER_THREAD];
#pragma unroll
    for (int j = 0; j < DOF_PER_THREAD; ++j) {
      const int i = i0 + (int)threadIdx.x + j * NTH;
      k0[j] = k1[j] = 0;
      if (i < i1) {
        k0[j] = at(A.vtx_slot_off, (unsigned)(i / 3));
        k1[j] = at(A.vtx_slot_off, (unsigned)(i / 3) + 1);
      }
    }
    if constexpr (WINDOW)
      vs.store(w);
    else
      vs.stage(v0, v1, VSUM_LDS_BYTES / (int)sizeof(R));
#pragma unroll
    for (int j = 0; j < DOF_PER_THREAD; ++j) {
      const int i = i0 + (int)threadIdx.x + j * NTH;
      if (i >= i1) continue;
      R acc[NCH / 3];
      vs.sum_dof(k0[j], k1[j], i - 3 * (i / 3), acc);
#pragma unroll
      for (int grp = 0; grp < NCH / 3; ++grp) {
        R* out = A.h_only ? A.out_b : (grp == 0 ? A.out_a : A.out_b);
        if (A.accumulate)
          at(out, (unsigned)i) += acc[grp];
        else
          at(out, (unsigned)i) = acc[grp];
      }
    }
  }
}

// The pass variants the library instantiates.
#define APL_WHAT_LIST(X)         \
  X(W_E)                         \
  X(W_E | W_G | W_H)             \
  X(W_G)                         \
  X(W_H)                         \
  X(W_HP)                        \
  X(W_HQ)                        \
  X(W_MIX)

template <int MAT, unsigned WHAT, class R>
static int launch_one(apl_mesh* m, const void* mu, const void* lam, const void* x, const void* p, void* out_a,
                      void* out_b, int accumulate, hipStream_t s, void* out_c, const Workspace* ws) {
  if (launch_blocks(m, MAT) == 0) return 0;
  return launch_pass<MAT, WHAT, R, R>(m, make_args<R, R>(m, mu, lam, x, p, out_a, out_b, accumulate, out_c, ws), false,
                                      0, s);
}

template <int MAT, class R>
static int dispatch_what(apl_mesh* m, unsigned what, const void* mu, const void* lam, const void* x, const void* p,
                         void* out_a, void* out_b, int accumulate, hipStream_t s, void* out_c, const Workspace* ws) {
#define APL_CASE(W) \
  if (what == (W)) return launch_one<MAT, (W), R>(m, mu, lam, x, p, out_a, out_b, accumulate, s, out_c, ws);
  if constexpr (MAT == MAT_MUSCLE) {
    // activation derivatives, alone or with the mu / lambda ones
    APL_CASE(W_MIXA)
    APL_CASE(W_MIX | W_MIXA)
  }
  APL_WHAT_LIST(APL_CASE)
#undef APL_CASE
  set_error("unsupported combination of outputs for one element pass");
  return -1;
}

int launch_elem(apl_mesh* m, int material, unsigned what, const void* mu, const void* lam, const void* x,
                const void* p, void* out_a, void* out_b, int accumulate, hipStream_t s, void* out_c,
                const Workspace* ws) {
  auto go = [&](auto mat_c) -> int {
    constexpr int MAT = decltype(mat_c)::value;
    if (m->dtype == DT_F32)
      return dispatch_what<MAT, float>(m, what, mu, lam, x, p, out_a, out_b, accumulate, s, out_c, ws);
    return dispatch_what<MAT, double>(m, what, mu, lam, x, p, out_a, out_b, accumulate, s, out_c, ws);
  };
  if (material == MAT_MODEL) {
    // a model mesh: every law present, each over its own blocks (the muscle
    // law's activation derivatives only exist for that law)
    if (!m->model) {
      set_error("APL_MODEL needs a mesh created by apl_model_create");
      return -1;
    }
    for (int law = 0; law < N_MAT; ++law) {
      if (m->law_nblk[law] == 0) continue;
      unsigned w = what;
      if (law != MAT_MUSCLE) w &= ~W_MIXA;
      if (w == 0) continue;
      if (launch_elem(m, law, w, mu, lam, x, p, out_a, out_b, accumulate, s, out_c, ws)) return -1;
    }
    return 0;
  }
  if (material == MAT_SNH) return go(std::integral_constant<int, MAT_SNH>{});
  if (material == MAT_ARAP) return go(std::integral_constant<int, MAT_ARAP>{});
  if (material == MAT_MUSCLE) {
    if (m->activation == nullptr && launch_blocks(m, MAT_MUSCLE) > 0) {
      set_error("the muscle law needs the activation: call apl_mesh_set_activation first");
      return -1;
    }
    return go(std::integral_constant<int, MAT_MUSCLE>{});
  }
  set_error("unknown material");
  return -1;
}

template <int MAT>
static int grid_mat(apl_mesh* m, unsigned what) {
#define APL_CASE(W) \
  if (what == (W)) return m->dtype == DT_F32 ? grid_for<MAT, (W), float, float>(m, false) : grid_for<MAT, (W), double, double>(m, false);
  APL_WHAT_LIST(APL_CASE)
#undef APL_CASE
  return 0;
}

int elem_grid(apl_mesh* m, int material, unsigned what) {
  if (material == MAT_MODEL) {
    int g = 0;
    for (int law = 0; law < N_MAT; ++law)
      if (m->law_nblk[law] > 0) g = std::max(g, elem_grid(m, law, what));
    return g;
  }
  if (material == MAT_MUSCLE) return grid_mat<MAT_MUSCLE>(m, what);
  return material == MAT_SNH ? grid_mat<MAT_SNH>(m, what) : grid_mat<MAT_ARAP>(m, what);
}

// The largest block window (distinct vertices per block) every pass variant
// of a mesh of this dtype can stage within ELEM_LDS_MAX, filtered launches
// included: 1024 for FP32 meshes (also with the solver's FP64 displacements),
// 478 for FP64 meshes (pass A: 6 FP64 channels x 1024 positions + 32 B per slot).
template <class R, class X>
static bool fits(int n) {
  return smem_bytes_n<W_E | W_G | W_H, R, X>(n, true) <= ELEM_LDS_MAX &&
         smem_bytes_n<W_HP, R, R>(n, true) <= ELEM_LDS_MAX && smem_bytes_n<W_HQ, R, X>(n, true) <= ELEM_LDS_MAX &&
         smem_bytes_n<W_MIX | W_MIXA, R, R>(n, true) <= ELEM_LDS_MAX && smem_bytes_n<W_G, R, R>(n, true) <= ELEM_LDS_MAX &&
         smem_bytes_n<W_H, R, R>(n, true) <= ELEM_LDS_MAX;
}

int nloc_limit(int dtype) {
  int n = 1024;
  if (dtype == DT_F64) {
    while (n > 4 && !fits<double, double>(n)) --n;
  } else {
    while (n > 4 && !(fits<float, float>(n) && fits<float, double>(n))) --n;
  }
  return n;
}

int launch_finish(apl_mesh* m, unsigned what, void* out_a, void* out_b, double* out_e, double* out_q,
                  int accumulate, hipStream_t s, const Workspace* ws) {
  const bool g = what & W_G, h = what & W_H, hp = what & W_HP;
  const int nch = (g ? 3 : 0) + (h ? 3 : 0) + (hp ? 3 : 0);
  const bool inst = out_e != nullptr || out_q != nullptr;
  const int nvblk = nch > 0 ? (int)m->L.vblk_inst.size() : 0;
  const int ninst = inst ? (int)m->L.n_inst : 0;
  const int grid = nvblk + ninst;
  if (grid == 0) return 0;
  auto go = [&](auto* tag, auto nch_c) {
    using R = std::remove_pointer_t<decltype(tag)>;
    FinishArgs<R> A;
    A.vblk_off = m->d.vblk_off;
    A.vtx_slot_off = m->d.vtx_slot_off;
    A.partial = (const R*)(ws != nullptr ? ws->partial : m->d.partial);
    A.out_a = (R*)out_a;
    A.out_b = (R*)out_b;
    A.blk_red = ws != nullptr ? ws->blk_red : m->d.blk_red;
    A.inst_blk_off = m->d.inst_blk_off;
    A.out_e = out_e;
    A.out_q = out_q;
    A.ninst = ninst;
    A.h_only = (h && !g && !hp) ? 1 : 0;
    A.accumulate = accumulate;
    A.n_verts = (int)m->L.V;
    constexpr int NCH = decltype(nch_c)::value;
    constexpr bool CAN_WINDOW = NCH == 6 && sizeof(R) == 4;
    if (m->L.n_inst == 1 && CAN_WINDOW && nvblk <= 2 * m->n_cu)
      hipLaunchKernelGGL((finish_kernel<R, NCH, true, CAN_WINDOW>), dim3((unsigned)grid), dim3(NTH), 0, s, A);
    else if (m->L.n_inst == 1)
      hipLaunchKernelGGL((finish_kernel<R, NCH, true, false>), dim3((unsigned)grid), dim3(NTH), 0, s, A);
    else
      hipLaunchKernelGGL((finish_kernel<R, NCH, false, false>), dim3((unsigned)grid), dim3(NTH), 0, s, A);
  };
  using I0 = std::integral_constant<int, 0>;
  using I3 = std::integral_constant<int, 3>;
  using I6 = std::integral_constant<int, 6>;
  if (m->dtype == DT_F32) {
    float* t = nullptr;
    if (nch == 6) go(t, I6{}); else if (nch == 3) go(t, I3{}); else go(t, I0{});
  } else {
    double* t = nullptr;
    if (nch == 6) go(t, I6{}); else if (nch == 3) go(t, I3{}); else go(t, I0{});
  }
  APL_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace apl

// ------------------------------------------------------------ allocation-free entry point
//
// apl_elem_eval_static: apl_elem_eval with the element passes' scratch (slot
// partials and block sums) in a file-scope device array instead of the
// mesh's workspace.  Each GPU the library runs on holds its own copy of the
// array until the process ends; its device address is looked up once per
// device (hipGetSymbolAddress, with that device current) and only that
// address is handed to kernels.  Every call on one GPU shares the array, so
// calls that overlap on one GPU race.  Nothing in the array needs to start
// at zero: a pass writes every partial and block sum it later reads.

namespace apl {

constexpr size_t STATIC_SCRATCH_BYTES = size_t(32) << 20;  // 32 MiB per GPU
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[MAX_DEVICES] = {};

// device address of this GPU's scratch array (m->device is current)
static int static_scratch(int device, void** out) {
  if (device < 0 || device >= MAX_DEVICES) {
    set_error("device index out of range for the static scratch table");
    return -1;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error(std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
      (void)hipGetLastError();
      return -1;
    }
    g_scratch_ptr[device] = p;
  }
  *out = g_scratch_ptr[device];
  return 0;
}

}  // namespace apl

extern "C" size_t apl_static_scratch_bytes(void) { return apl::STATIC_SCRATCH_BYTES; }

extern "C" int apl_elem_eval_static(apl_mesh* m, int material, const void* mu, const void* lam, const void* u,
                                    const void* p, unsigned what, double* energy, void* grad, void* hess_diag,
                                    void* hess_prod, double* hess_quad, void* dmu, void* dlam, void* stream) {
  using namespace apl;
  if (m == nullptr) {
    set_error("mesh is NULL");
    return -1;
  }
  const size_t need = eval_scratch_bytes(m);
  if (need > STATIC_SCRATCH_BYTES) {
    set_error("mesh needs " + std::to_string(need) + " bytes of element-pass scratch; apl_elem_eval_static holds " +
              std::to_string(STATIC_SCRATCH_BYTES) + " (use apl_elem_eval)");
    return -1;
  }
  APL_CHECK_HIP(hipSetDevice(m->device));
  (void)hipGetLastError();  // drop errors left by unrelated earlier HIP calls
  void* base = nullptr;
  if (static_scratch(m->device, &base)) return -1;
  const size_t part = (size_t)MAX_CH * (size_t)std::max<int64_t>(m->L.n_slots, 1) * real_size(m);
  Workspace ws;
  ws.partial = base;
  ws.blk_red = reinterpret_cast<double*>(static_cast<unsigned char*>(base) + ((part + 255) / 256) * 256);
  return elem_eval_impl(m, material, mu, lam, u, p, what, energy, grad, hess_diag, hess_prod, hess_quad, dmu, dlam,
                        (hipStream_t)stream, &ws);
}
