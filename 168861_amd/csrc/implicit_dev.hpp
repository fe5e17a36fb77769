// Device state and per-row routines of the implicit step, shared by its kernels
// (implicit.hip: persistent grids and tree solves; krylov_block.hip: Krylov solves
// of small systems in one workgroup).
#pragma once
#include "nrt_internal.hpp"
#include "nrt_device.hpp"

namespace nrt {

enum : int32_t {
  RT_NORMAL = 1, RT_BRANCH = 2, RT_TERM = 4, RT_NEXT_TERM = 8, RT_FIRST_NORMAL = 16,
  RT_FIRST_BRANCH = 32, RT_OTHER = 64
};

struct ImpHH {
  double* m;
  double* h;
  double* n;
  const double* E_Na;
  const double* E_K;
  const double* E_L;
  const double* g_Na;
  const double* g_K;
  const double* G_L;
  const double* ls_Na;
  const double* ls_K;
  const double* rest;
  const int32_t* type;
  const int32_t* mat;
  const int32_t* dl;
  const int32_t* row;  // element (row) of each HH entry
};

struct ImpStats {
  unsigned long long iters_total;
  unsigned long long sweeps_total;  // refinement sweeps (FP32 forms)
  unsigned long long steps;
  int last_iters;
  int status;
  double last_rr;
  double last_bb;
  // first failure: step, iteration and the scalars of that iteration
  long long fail_step;
  int fail_iter;
  int restarts;
  double fail_rho, fail_apr, fail_w1, fail_w2, fail_rr;
  double fail_bb;    // |b|^2 of the failing step (refinement: |D^-1 b|^2)
  int fail_cycles;   // GMRES restart cycles / refinement sweeps of the failing step
};

struct ImpDev {
  int N;
  int H;
  int nblocks;  // workgroups working on this tree (its "virtual grid")
  int vb;       // this workgroup's index in that grid
  int rpb;  // rows per block
  double dT;
  double dt_ms;
  const int32_t* rowptr;
  const int32_t* col;
  double* val;
  const double* cmdx;
  const double* kdx;
  const double* input;
  const double* rdx;
  const double* dxv;
  const uint32_t* code;
  ImpHH hh;
  double* x;
  double* b;
  double* r0;
  double* r;
  double* p0;
  double* p1;
  double* v0;
  double* v1;
  double* s;
  double* t;
  double* part;
  unsigned* bar;
  unsigned* err;
  ImpStats* st;
  double tol;
  int tol_mode;
  int x0_mode;
  int check_every;
  int max_iter;
  unsigned long long spin_limit;
  long long first, num, a0, a1, interval;
  long long gl0;  // trace phase at step `first` (steps since the last sample)
  int trace_elem;  // element (BiCGSTAB) or its level-0 slot (tree solve)
  double* trace;
  // tree solve: the state in level-0 slot order (ns0 slots, padding included)
  int ns0;
  const double* scmdx;
  const double* skdx;
  const double* sinput;
  const uint32_t* scode;    // HH flag and index, or kCodeSkip for padding
  const int32_t* srowptr;   // the FP64 matrix with rows in slot order
  const int32_t* scol;      // column slots
  const uint8_t* srole;     // 0 diagonal, 1 coupling to the parent, 2 to a child
  const int32_t* hh_slot;   // slot of each HH entry's row
  // the tree solve's work arrays already hold this plan's matrix and factors (a
  // batch slot after its first launch): the launch skips the fill and the full
  // factorization (static chunks keep theirs between launches, dynamic ones are
  // eliminated again by every step)
  int keep_factors;
};

// breakdown restarts allowed per time step before the step reports NOT_CONVERGED
constexpr int kMaxRestarts = 64;

// HH gating (solverIm-gpu.cpp:61-98): the per-entry parameters, and one step of
// the gates at potential v (updates m, h, n; returns W and K).
struct HHGate {
  double rest, ls_Na, ls_K, g_Na, g_K, G_L, E_Na, E_K, E_L;
};
__device__ __forceinline__ HHGate hh_gate_load(const ImpHH& hd, int i) {
  return HHGate{hd.rest[i], hd.ls_Na[i], hd.ls_K[i], hd.g_Na[i], hd.g_K[i],
                hd.G_L[i],  hd.E_Na[i],  hd.E_K[i],  hd.E_L[i]};
}
// The rate functions (coupling.cpp:25-48) in precision R: FP64 for the FP64 forms;
// FP32 (expf, single-precision divisions) for the FP32 forms, whose gate state,
// conductances and currents stay FP64.
template <class R>
struct HHRates {
  double am, bm, ah, bh, an, bn;
};
template <class R>
__device__ __forceinline__ HHRates<R> hh_rates(const HHGate& q, double v) {
  double vna = v + q.ls_Na;
  double vk = v + q.ls_K;
  vna = (vna - q.rest) / 0.001;
  vk = (vk - q.rest) / 0.001;
  if constexpr (sizeof(R) == 4) {
    const float un = (float)vna, uk = (float)vk;
    return HHRates<R>{(2.5f - 0.1f * un) / (expf(2.5f - 0.1f * un) - 1.0f),
                      4.0f * expf(-un / 18.0f),
                      0.07f * expf(-un / 20.0f),
                      1.0f / (expf(3.0f - 0.1f * un) + 1.0f),
                      (0.1f - 0.01f * uk) / (expf(1.0f - 0.1f * uk) - 1.0f),
                      0.125f * expf(-uk / 80.0f)};
  } else {
    return HHRates<R>{(2.5 - 0.1 * vna) / (exp(2.5 - 0.1 * vna) - 1), 4 * exp(-vna / 18),
                      0.07 * exp(-vna / 20), 1 / (exp(3 - 0.1 * vna) + 1),
                      (0.1 - 0.01 * vk) / (exp(1 - 0.1 * vk) - 1), 0.125 * exp(-vk / 80)};
  }
}
template <class R = double>
__device__ __forceinline__ void hh_gate_step(const HHGate& q, double v, double dt_ms, double& m,
                                             double& h, double& n, double& W, double& K) {
  const HHRates<R> rt = hh_rates<R>(q, v);
  const double am = rt.am, bm = rt.bm, ah = rt.ah, bh = rt.bh, an = rt.an, bn = rt.bn;
  const double m0 = m, h0 = h, n0 = n;
  m = m0 + dt_ms * (am * (1 - m0) - bm * m0);
  h = h0 + dt_ms * (ah * (1 - h0) - bh * h0);
  n = n0 + dt_ms * (an * (1 - n0) - bn * n0);
  const double gna = q.g_Na * m * m * m * h;
  const double gk = q.g_K * n * n * n * n;
  const double gl = q.G_L;
  W = -(gna + gk + gl);
  K = gna * q.E_Na + gk * q.E_K + gl * q.E_L;
}
template <class R = double>
__device__ __forceinline__ void imp_gate(const ImpHH& hd, int i, double v, double dt_ms,
                                         double& W, double& K) {
  double m = hd.m[i], h = hd.h[i], n = hd.n[i];
  hh_gate_step<R>(hh_gate_load(hd, i), v, dt_ms, m, h, n, W, K);
  hd.m[i] = m;
  hd.h[i] = h;
  hd.n[i] = n;
}

// Update_Mat (solverIm-gpu.cpp:103-156) for the HH row of element iv: the row's
// fixed coefficients, and its refresh for a new W (returns false for identity
// rows, left as they are, else true with the new diagonal).
struct HHRow {
  int type, im;
  double alpha, inv_rdx, betaR, betaL, dxv, c_dt;
};
__device__ __forceinline__ HHRow hh_row_load(const ImpDev& d, int hh, int iv) {
  HHRow q{};
  q.type = d.hh.type[hh];
  // identity rows (ghosts, sealed ends) keep their 1 and read no neighbour
  if (q.type == RT_OTHER || q.type == RT_TERM) return q;
  q.im = d.hh.mat[hh];
  q.alpha = -1 / d.rdx[iv];
  q.inv_rdx = 1 / d.rdx[iv];
  q.betaR = 1 / d.rdx[iv + 1];
  q.dxv = d.dxv[iv];
  q.c_dt = d.cmdx[iv] / d.dT;
  if (q.type == RT_BRANCH || q.type == RT_FIRST_BRANCH) q.betaL = 1 / d.rdx[d.hh.dl[hh]];
  return q;
}
__device__ __forceinline__ bool hh_row_refresh(const HHRow& q, double W, double* v,
                                               double& diag) {
  if (q.type == RT_OTHER || q.type == RT_TERM) return false;
  const int im = q.im;
  const double alpha = q.alpha;
  const double betaR = q.betaR;
  const double betaMe = -(W * q.dxv) + q.inv_rdx;
  const double beta = q.c_dt + betaMe + betaR;
  const double delta = -betaR;
  const double betaL = q.betaL;
  switch (q.type) {
    case RT_NEXT_TERM:
      diag = beta + delta;
      v[im] = alpha;
      v[im + 1] = diag;
      return true;
    case RT_BRANCH:
      diag = beta + betaL;
      v[im] = alpha;
      v[im + 1] = diag;
      v[im + 2] = delta;
      v[im + 3] = -betaL;
      return true;
    case RT_NORMAL:
      diag = beta;
      v[im] = alpha;
      v[im + 1] = diag;
      v[im + 2] = delta;
      return true;
    case RT_FIRST_NORMAL:
      diag = alpha + beta;
      v[im] = diag;
      v[im + 1] = delta;
      return true;
    case RT_FIRST_BRANCH:
      diag = alpha + beta + betaL;
      v[im] = diag;
      v[im + 1] = delta;
      v[im + 2] = -betaL;
      return true;
    default:
      return false;
  }
}
__device__ __forceinline__ bool imp_update_row(const ImpDev& d, int hh, int iv, double W,
                                               double& diag) {
  return hh_row_refresh(hh_row_load(d, hh, iv), W, d.val, diag);
}

constexpr int kGmresMaxRestart = 512;
constexpr double kGmresInnerRel32 = 1e-6;

template <class T>
struct GmresDev {
  int m;           // restart length
  T* V;            // (m+1) x N basis (v_k at V + k N; only a block's own rows)
  T* w0;           // Arnoldi vectors, even and odd steps
  T* w1;
  double* R;       // per workgroup: packed R (m(m+1)/2), cs, sn (m), g (m+1), y (m)
  int64_t rstride;
  double* part;    // 2 sets x nblocks x (m+1) partial sums
  T* vals;         // matrix values of the Arnoldi SpMV (FP64: the matrix itself)
  double refine_tol;  // FP32: convergence of the FP64 residual, relative to |b|
};

}  // namespace nrt
