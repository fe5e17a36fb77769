// Krylov solves of small systems in one workgroup: the methods of
// implicit.hip's persistent grids (BiCGSTAB with the reference's recurrences,
// solverIm-gpu.cpp:725-843; GMRES(m) in FP64, solverIm-cpu.cpp:192-272) for matrices
// of which one CU holds every row.
//
// A thread owns the rows tid, tid + nt, ... (R of them): its matrix rows (at most 4
// entries, k_row_len), its entries of every Krylov vector and of x stay in registers
// for the whole launch, so an iteration touches no memory but LDS: the operand of a
// matrix product goes through LDS (one store, at most four loads a row) and a
// reduction is a DPP wave sum, one LDS slot a wave and one barrier. What bounds an
// iteration is the chain of its three reductions, two products and five divisions.
// Measured (333-row tree, 560 iterations a step): 12.0 us an iteration as a grid of
// one workgroup (its grid barriers' agent fences drop the caches, so each phase
// fetched the CSR rows and vectors again), 1.4 to 1.6 us here (1,000 rows: 16 -> 1.9;
// 2,000 rows: 22 -> 3.2). BiCGSTAB sums in the grid kernel's order (256 threads, rows tid,
// tid + 256, ...), so its iterates are that kernel's to the bit: where an iteration
// count depends on rounding, it stays what it was. GMRES(150), 1,002 rows, 50 to 62 Arnoldi
// steps a time step: 86 to 95 us an Arnoldi step -> 18 to 20. Its inner products sum in
// another order than the grid kernel's, so its iterates differ by rounding: over 24 axons
// of 200 to 2,200 rows the same Arnoldi steps, and the largest error against 64-bit
// elimination 0.87 times the grid kernel's in the mean (0.2 to 4.8), all below 5e-12 V.
#include <algorithm>
#include "implicit_dev.hpp"

namespace nrt {

constexpr int kKbMaxN = 2048;     // BiCGSTAB: 8 rows per thread of 256 (512 VGPRs a thread)
constexpr int kKbThreads = 256;   // BiCGSTAB: one wave a SIMD; the grid kernel's row order
constexpr int kKgMaxN = 4096;     // GMRES: 8 rows per thread of 512
constexpr int kKgThreads = 1024;  // GMRES: waves share out the basis vectors
constexpr int kRowMax = 4;       // entries of a matrix row (k_row_len)

// Sums of NV values over the workgroup, the same bits in every thread and uniform to
// the compiler. Each row of 16 lanes is summed by four DPP steps, one lane of it stores
// the row sum, and after the barrier every row of lanes combines the row sums: four to
// a wave, then the waves one after the other, which is block_sum's order. `lds` holds
// two sets of NV * 64 values used in turn (`par`), so one barrier is enough: a set is
// written again only after the other set's barrier. The slots of absent waves stay 0
// (kb_sum_clear).
template <int NV>
__device__ __forceinline__ void kb_rows16(double (&v)[NV]) {
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = v[k] + dpp_f64<0xB1>(v[k]);
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = v[k] + dpp_f64<0x4E>(v[k]);
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = v[k] + dpp_f64<0x141>(v[k]);
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = v[k] + dpp_f64<0x140>(v[k]);
}
constexpr int kKbSumLds = 2 * 3 * 64;
template <int NV, int NW>
__device__ __forceinline__ void kb_sum(double (&v)[NV], double* lds, int& par) {
  static_assert(NV <= 3, "kKbSumLds");
  const int lane = threadIdx.x & (kWave - 1);
  double* set = lds + par;
  par = kKbSumLds / 2 - par;
  kb_rows16(v);
  if ((lane & 15) == 0) {
#pragma unroll
    for (int k = 0; k < NV; k++) set[k * 64 + (threadIdx.x >> 4)] = v[k];
  }
  lds_sync();
  double t[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) t[k] = 0.0;
#pragma unroll
  for (int q = 0; q < NW; q += 4) {  // four waves at a time: lanes 4 w .. 4 w + 3 are wave w's
    double s[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) s[k] = set[k * 64 + q * 4 + (lane & 15)];
#pragma unroll
    for (int k = 0; k < NV; k++) s[k] = s[k] + dpp_f64<0xB1>(s[k]);
#pragma unroll
    for (int k = 0; k < NV; k++) s[k] = s[k] + dpp_f64<0x4E>(s[k]);
#pragma unroll
    for (int w = 0; w < 4; w++)
#pragma unroll
      for (int k = 0; k < NV; k++) t[k] = t[k] + readlane_f64(s[k], 4 * w);
  }
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = t[k];
}
__device__ __forceinline__ void kb_sum_clear(double* lds) {
  for (int i = threadIdx.x; i < kKbSumLds; i += blockDim.x) lds[i] = 0.0;
  __syncthreads();
}

// The rows of one thread. A row past the end has no entries and stands for slot N of
// the LDS vectors, so no lane branches: its vector entries stay 0.
template <int R>
struct KbRows {
  int i[R];
  bool live[R];
  double a[R][kRowMax];
  uint32_t c[R][kRowMax / 2];  // columns, two to a word (kKgMaxN < 65,536)
  bool hh[R];  // a Hodgkin-Huxley row: its values change every step

  __device__ __forceinline__ void values(const ImpDev& d, int k) {
    const int b = d.rowptr[i[k]], n = d.rowptr[i[k] + 1] - b;
#pragma unroll
    for (int q = 0; q < kRowMax; q++) a[k][q] = q < n ? d.val[b + q] : 0.0;
  }
  __device__ __forceinline__ void load(const ImpDev& d) {
#pragma unroll
    for (int k = 0; k < R; k++) {
      i[k] = (int)threadIdx.x + k * (int)blockDim.x;
      live[k] = i[k] < d.N;
      hh[k] = false;
      if (!live[k]) i[k] = d.N;
#pragma unroll
      for (int q = 0; q < kRowMax; q++) a[k][q] = 0.0;
#pragma unroll
      for (int q = 0; q < kRowMax / 2; q++) c[k][q] = (uint32_t)i[k] * 0x10001u;
      if (!live[k]) continue;
      const int b = d.rowptr[i[k]], n = d.rowptr[i[k] + 1] - b;
      values(d, k);
#pragma unroll
      for (int q = 0; q < kRowMax; q++)
        if (q < n)
          c[k][q / 2] = (c[k][q / 2] & (0xFFFFu << (16 - 16 * (q & 1)))) |
                        ((uint32_t)d.col[b + q] << (16 * (q & 1)));
      hh[k] = (d.code[i[k]] & kCodeHH) != 0;
    }
  }
  // y_i = sum over the row, in its column order (an absent entry adds 0 times the
  // row's own operand, which its diagonal multiplies too)
  __device__ __forceinline__ double mul(const double* sx, int k) const {
    double s = 0;
#pragma unroll
    for (int q = 0; q < kRowMax; q++) s = s + a[k][q] * sx[(c[k][q / 2] >> (16 * (q & 1))) & 0xFFFF];
    return s;
  }
  // Update phase of the own rows (gating, HH rows, right-hand side): v holds their
  // potentials and takes the right-hand sides (LDS, own entries only). A loop over
  // the rows and not unrolled: the gating's registers are needed once.
  __device__ __forceinline__ void rhs(const ImpDev& d, double* v, bool active) {
#pragma unroll 1
    for (int q = (int)threadIdx.x; q < d.N; q += (int)blockDim.x) {
      const double vq = v[q];
      const uint32_t code = d.code[q];
      double kd;
      if (code & kCodeHH) {
        const int h = (int)(code & kCodeIdx);
        double W, K, diag;
        imp_gate(d.hh, h, vq, d.dt_ms, W, K);
        (void)imp_update_row(d, h, q, W, diag);
        kd = K * d.dxv[q];
      } else {
        kd = d.kdx[q];
      }
      double b = d.cmdx[q] * vq / d.dT + kd;
      if (active) b = b + d.input[q];
      v[q] = b;
    }
#pragma unroll
    for (int k = 0; k < R; k++)
      if (live[k] && hh[k]) values(d, k);
  }
};

// What a launch adds to the handle's statistics (kept in registers until its end).
struct KbStats {
  unsigned long long iters = 0, cycles = 0, steps = 0;
  int last_iters = 0, restarts = 0;
  double rr = 0, bb = 0;
  __device__ __forceinline__ void store(ImpStats* st) const {
    st->iters_total += iters;
    st->sweeps_total += cycles;
    st->steps += steps;
    st->restarts += restarts;
    if (steps > 0) {
      st->last_iters = last_iters;
      st->last_rr = rr;
      st->last_bb = bb;
    }
  }
};

template <int R>
__global__ __launch_bounds__(kKbThreads) void k_bicgstab_block(ImpDev d) {
  __shared__ double lds[kKbSumLds];
  extern __shared__ double sdyn[];
  double* sp = sdyn;        // operand of A p (and of A x0)
  double* ss = sdyn + d.N + 1;  // operand of A s
  int par = 0;
  constexpr int NW = kKbThreads / kWave;
  kb_sum_clear(lds);
  KbRows<R> w;
  w.load(d);
  double x[R], r[R], r0[R], p[R], v[R], s[R], t[R], b[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    x[k] = w.live[k] ? d.x[w.i[k]] : 0.0;
    p[k] = v[k] = s[k] = t[k] = r[k] = r0[k] = b[k] = 0.0;
  }
  KbStats acc;
  long long gl = 0, ksamp = 0;
  for (long long step = d.first; step < d.first + d.num; step++) {
    const bool active = step >= d.a0 && step <= d.a1;
#pragma unroll
    for (int k = 0; k < R; k++)
      ss[w.i[k]] = x[k];
    w.rhs(d, ss, active);
#pragma unroll
    for (int k = 0; k < R; k++) {
      b[k] = ss[w.i[k]];
      if (d.x0_mode == NRT_X0_RHS) x[k] = b[k];
      sp[w.i[k]] = x[k];
    }
    __syncthreads();
    double red2[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < R; k++) {
      const double ri = b[k] + (-1.0) * w.mul(sp, k);
      r0[k] = r[k] = ri;
      red2[0] = red2[0] + ri * ri;
      red2[1] = red2[1] + b[k] * b[k];
    }
    kb_sum<3, NW>(red2, lds, par);
    double rho = red2[0], rr = red2[0];
    const double bb = red2[1];
    const double thr = d.tol_mode == NRT_TOL_RELATIVE ? d.tol * sqrt(bb) : d.tol;
    const double limit = thr * thr;
    int status = rr <= limit ? NRT_OK : NRT_ERR_NOT_CONVERGED;
    int it = 0, restarts = 0, since = 0;  // since: it modulo check_every
    double alpha = 0, omega = 0, beta = 0, f_apr = 0, f_w1 = 0, f_w2 = 0;
    bool first_it = true, restart = false;
    while (status == NRT_ERR_NOT_CONVERGED && it < d.max_iter) {
      // phase A: p = r + beta (p - omega v), v = A p, (v, r0); after a breakdown the
      // shadow residual restarts as r0 = r
      const double nomega = -omega;
#pragma unroll
      for (int k = 0; k < R; k++) {
          p[k] = first_it ? r[k] : r[k] + beta * (p[k] + nomega * v[k]);
        sp[w.i[k]] = p[k];
      }
      __syncthreads();
      double redA[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < R; k++) {
          v[k] = w.mul(sp, k);
        if (restart) r0[k] = r[k];
        redA[0] = redA[0] + v[k] * r0[k];
      }
      restart = false;
      {
        double one[1] = {redA[0]};
        kb_sum<1, NW>(one, lds, par);
        redA[0] = one[0];
      }
      f_apr = redA[0];
      if (!isfinite(redA[0])) {
        status = NRT_ERR_NUMERIC;
        break;
      }
      const double al = rho / redA[0];
      if (redA[0] == 0.0 || !isfinite(al)) {
        // Lanczos breakdown (v orthogonal to the shadow residual): restart
        it++;
        if (++since == d.check_every) since = 0;
        if (++restarts > kMaxRestarts) break;
        restart = true;
        first_it = true;
        rho = rr;
        continue;
      }
      alpha = al;
      const double nalpha = -al;
      // phase B: s = r - alpha v, t = A s, (t, s), (t, t), (s, s)
#pragma unroll
      for (int k = 0; k < R; k++) {
          s[k] = r[k] + nalpha * v[k];
        ss[w.i[k]] = s[k];
      }
      __syncthreads();
      double redB[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < R; k++) {
          t[k] = w.mul(ss, k);
        redB[0] = redB[0] + t[k] * s[k];
        redB[1] = redB[1] + t[k] * t[k];
        redB[2] = redB[2] + s[k] * s[k];
      }
      kb_sum<3, NW>(redB, lds, par);
      f_w1 = redB[0];
      f_w2 = redB[1];
      it++;
      if (++since == d.check_every) since = 0;
      if (!isfinite(redB[2]) || !isfinite(redB[1])) {
        status = NRT_ERR_NUMERIC;
        break;
      }
      if (redB[2] <= limit || redB[1] == 0.0) {
        // converged at the half step: x += alpha p, r = s
#pragma unroll
        for (int k = 0; k < R; k++) {
          x[k] = x[k] + alpha * p[k];
          r[k] = s[k];
        }
        rr = redB[2];
        status = NRT_OK;
        break;
      }
      omega = redB[0] / redB[1];
      const double nw = -omega;
      const double ao = alpha / omega;  // while the sums below are made
      // phase C: x += alpha p + omega s, r = s - omega t, (r, r0), (r, r)
      double redC[2] = {0.0, 0.0};
#pragma unroll
      for (int k = 0; k < R; k++) {
          x[k] = (x[k] + alpha * p[k]) + omega * s[k];
        r[k] = s[k] + nw * t[k];
        redC[0] = redC[0] + r[k] * r0[k];
        redC[1] = redC[1] + r[k] * r[k];
      }
      kb_sum<2, NW>(redC, lds, par);
      beta = ao * (redC[0] / rho);
      rho = redC[0];
      rr = redC[1];
      first_it = false;
      if (!isfinite(rr)) {
        status = NRT_ERR_NUMERIC;
        break;
      }
      if (since == 0 && rr <= limit) {
        status = NRT_OK;
        break;
      }
      if (!isfinite(beta) || rho == 0.0 || omega == 0.0) {
        // breakdown of the bi-orthogonality: restart with r0 = r, p = r
        if (++restarts > kMaxRestarts) break;
        restart = true;
        first_it = true;
        rho = rr;
      }
    }
    acc.iters += (unsigned long long)it;
    acc.steps++;
    acc.last_iters = it;
    acc.restarts += restarts;
    acc.rr = rr;
    acc.bb = bb;
    if (threadIdx.x == 0 && status != NRT_OK && d.st->status == NRT_OK) {
      d.st->status = status;
      d.st->fail_step = step;
      d.st->fail_iter = it;
      d.st->fail_rho = rho;
      d.st->fail_apr = f_apr;
      d.st->fail_w1 = f_w1;
      d.st->fail_w2 = f_w2;
      d.st->fail_rr = rr;
      d.st->fail_bb = bb;
      d.st->fail_cycles = restarts;
    }
    if (d.interval >= 0 && ++gl > d.interval) {
      gl = 0;
#pragma unroll
      for (int k = 0; k < R; k++)
        if (d.trace && w.live[k] && w.i[k] == d.trace_elem) d.trace[ksamp] = x[k];
      ksamp++;
    }
    __syncthreads();  // the next step's operand goes where this one's may still be read
  }
#pragma unroll
  for (int k = 0; k < R; k++)
    if (w.live[k]) d.x[w.i[k]] = x[k];
  if (threadIdx.x == 0) acc.store(d.st);
}

// h[0..cnt) = V_j . w: each wave takes every NW-th basis vector, two at a time, its
// lanes the rows (w from LDS), so 8 loads are in flight a lane (with 16, some of them
// repeated past the ends, an Arnoldi step on 1,002 rows took 26.2 us instead of 23.4:
// the CU's load rate counts, not the latency alone); no barrier inside.
template <int NW>
__device__ __forceinline__ void kg_dots(const double* __restrict__ V, int N, int cnt,
                                        const double* sw, double* h) {
  constexpr int J = 2, U = 4;
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  for (int j0 = wid; j0 < cnt; j0 += J * NW) {
    double s[J];
    const double* v[J];
#pragma unroll
    for (int q = 0; q < J; q++) {
      s[q] = 0;
      v[q] = V + (size_t)min(j0 + q * NW, cnt - 1) * N;
    }
    const bool both = j0 + NW < cnt;
    for (int i0 = lane; i0 < N; i0 += U * kWave) {
      double l[J][U];
#pragma unroll
      for (int q = 0; q < J; q++)
#pragma unroll
        for (int u = 0; u < U; u++)
          l[q][u] = i0 + u * kWave < N && (q == 0 || both) ? v[q][i0 + u * kWave] : 0.0;
#pragma unroll
      for (int u = 0; u < U; u++) {
        const double wi = i0 + u * kWave < N ? sw[i0 + u * kWave] : 0.0;
#pragma unroll
        for (int q = 0; q < J; q++) s[q] = s[q] + l[q][u] * wi;
      }
    }
    kb_rows16(s);
#pragma unroll
    for (int q = 0; q < J; q++) {
      s[q] = (readlane_f64(s[q], 0) + readlane_f64(s[q], 16)) +
             (readlane_f64(s[q], 32) + readlane_f64(s[q], 48));
      if (lane == 0 && j0 + q * NW < cnt) h[j0 + q * NW] = s[q];
    }
  }
}

// w_i -= sum_j h_j V_j[i] over the own rows (columns in increasing order).
template <int R>
__device__ __forceinline__ void kg_subtract(const KbRows<R>& w, const double* __restrict__ V,
                                            int N, int cnt, const double* h, double (&wv)[R]) {
  constexpr int U = R >= 4 ? 2 : 8;  // 8 loads in flight a lane (16 for R = 8)
  for (int j0 = 0; j0 < cnt; j0 += U) {
    double l[R][U];
#pragma unroll
    for (int u = 0; u < U; u++)
#pragma unroll
      for (int k = 0; k < R; k++)
        l[k][u] = j0 + u < cnt && w.live[k] ? V[(size_t)(j0 + u) * N + w.i[k]] : 0.0;
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (j0 + u >= cnt) break;
      const double hj = h[j0 + u];
#pragma unroll
      for (int k = 0; k < R; k++) wv[k] = wv[k] - hj * l[k][u];
    }
  }
}

// Restarted GMRES in FP64: k_implicit_gmres<double>'s iteration (CGS2, Givens
// rotations, x += V y) with one workgroup. The basis stays in memory (the CU's L2
// share; it is read four times an Arnoldi step: what bounds the step), the current
// vectors in registers and LDS, the rotations and the new column in LDS, the packed
// triangular factor in memory, written once a column.
template <int R, int BS>
__global__ __launch_bounds__(BS) void k_gmres_block(ImpDev d, GmresDev<double> g) {
  __shared__ double lds[kKbSumLds];
  __shared__ double fsh[2];
  extern __shared__ double sdyn[];
  const int N = d.N, m = g.m, tid = (int)threadIdx.x, nt = (int)blockDim.x;
  double* sx = sdyn;        // operand of the matrix product
  double* sw = sx + N + 1;  // Arnoldi vector
  double* h1 = sw + N + 1;  // projections and their corrections
  double* h2 = h1 + (m + 1);
  double* cs = h2 + (m + 1);
  double* sn = cs + m;
  double* gv = sn + m;
  double* yv = gv + (m + 1);
  double* col = yv + (m + 1);  // the new column of R
  double* Rp = g.R;  // packed R, column k at k (k + 1) / 2
  int par = 0;
  constexpr int NW = BS / kWave;
  kb_sum_clear(lds);
  KbRows<R> w;
  w.load(d);
  double x[R], b[R], r0[R], wv[R];
#pragma unroll
  for (int k = 0; k < R; k++) {
    x[k] = w.live[k] ? d.x[w.i[k]] : 0.0;
    b[k] = r0[k] = wv[k] = 0.0;
  }
  KbStats acc;
  long long gl = 0, ksamp = 0;
  for (long long step = d.first; step < d.first + d.num; step++) {
    const bool active = step >= d.a0 && step <= d.a1;
#pragma unroll
    for (int k = 0; k < R; k++)
      sw[w.i[k]] = x[k];
    w.rhs(d, sw, active);
#pragma unroll
    for (int k = 0; k < R; k++) {
      b[k] = sw[w.i[k]];
      if (d.x0_mode == NRT_X0_RHS) x[k] = b[k];
      else if (d.x0_mode == NRT_X0_ZERO) x[k] = 0.0;
    }
    int it = 0, status = NRT_ERR_NOT_CONVERGED, cycles = 0;
    double rr = 0, bb = 0, thr = 0;
    while (true) {
      // cycle start: r0 = b - A x, beta = |r0|
      __syncthreads();
#pragma unroll
      for (int k = 0; k < R; k++)
        sx[w.i[k]] = x[k];
      __syncthreads();
      double red[2] = {0.0, 0.0};
#pragma unroll
      for (int k = 0; k < R; k++) {
          r0[k] = b[k] - w.mul(sx, k);
        red[0] = red[0] + r0[k] * r0[k];
        red[1] = red[1] + b[k] * b[k];
      }
      kb_sum<2, NW>(red, lds, par);
      rr = red[0];
      if (cycles == 0) {
        bb = red[1];
        thr = d.tol_mode == NRT_TOL_RELATIVE ? d.tol * sqrt(bb) : d.tol;
      }
      if (!isfinite(rr)) {
        status = NRT_ERR_NUMERIC;
        break;
      }
      const double beta = sqrt(rr);
      if (beta <= thr) {
        status = NRT_OK;
        break;
      }
      if (it >= d.max_iter) break;
      cycles++;
      for (int j = tid; j <= m; j += nt) gv[j] = j == 0 ? beta : 0.0;
      double div = beta;
      int kk = 0;
      bool conv = false;
      for (int k = 0; k < m; k++) {
        it++;
        // v_k (stored) and w = A v_k
#pragma unroll
        for (int q = 0; q < R; q++) {
          const double vi = (k == 0 ? r0[q] : wv[q]) / div;
          sx[w.i[q]] = vi;
          if (w.live[q]) g.V[(size_t)k * N + w.i[q]] = vi;
        }
        lds_sync();
#pragma unroll
        for (int q = 0; q < R; q++) {
          wv[q] = w.mul(sx, q);
          sw[w.i[q]] = wv[q];
        }
        __syncthreads();
        // CGS2: h = V^T w; w -= V h; h2 = V^T w; w -= V h2
        kg_dots<NW>(g.V, N, k + 1, sw, h1);
        lds_sync();
        kg_subtract<R>(w, g.V, N, k + 1, h1, wv);
#pragma unroll
        for (int q = 0; q < R; q++)
          sw[w.i[q]] = wv[q];
        lds_sync();
        kg_dots<NW>(g.V, N, k + 1, sw, h2);
        lds_sync();
        kg_subtract<R>(w, g.V, N, k + 1, h2, wv);
        double nrm[1] = {0.0};
#pragma unroll
        for (int q = 0; q < R; q++) nrm[0] = nrm[0] + wv[q] * wv[q];
        kb_sum<1, NW>(nrm, lds, par);
        const double hn = sqrt(nrm[0]);
        // Givens rotations on the new column: a chain of k dependent rotations whose
        // running value stays in a register
        if (tid == 0) {
          constexpr int G = 4;  // rotations whose operands are read together
          double a = h1[0] + h2[0];
          for (int j0 = 0; j0 < k; j0 += G) {
            double hb[G], c[G], sg[G];
#pragma unroll
            for (int u = 0; u < G; u++) {
              const int j = min(j0 + u, k - 1);
              hb[u] = h1[j + 1] + h2[j + 1];
              c[u] = cs[j];
              sg[u] = sn[j];
            }
#pragma unroll
            for (int u = 0; u < G; u++) {
              if (j0 + u >= k) break;
              col[j0 + u] = c[u] * a + sg[u] * hb[u];
              a = -sg[u] * a + c[u] * hb[u];
            }
          }
          const double den = sqrt(a * a + hn * hn);
          const double ck = den == 0 ? 1.0 : a / den, sk = den == 0 ? 0.0 : hn / den;
          cs[k] = ck;
          sn[k] = sk;
          col[k] = den;
          const double g0 = gv[k], g1 = -sk * g0;
          gv[k + 1] = g1;
          gv[k] = ck * g0;
          fsh[0] = fabs(g1);
        }
        lds_sync();
        for (int j = tid; j <= k; j += nt) Rp[(size_t)k * (k + 1) / 2 + j] = col[j];
        const double res = fsh[0];
        kk = k + 1;
        if (!isfinite(res)) {
          status = NRT_ERR_NUMERIC;
          break;
        }
        if (res <= thr || hn == 0.0) {
          conv = true;
          rr = res * res;
          break;
        }
        if (it >= d.max_iter) break;
        div = hn;
      }
      if (status == NRT_ERR_NUMERIC) break;
      // R y = g by columns, wave 0: y_j, then its column's share of every row above
      __syncthreads();
      if (tid < kWave) {
        for (int j = kk - 1; j >= 0; j--) {
          const double* Rj = Rp + (size_t)j * (j + 1) / 2;
          const double y = gv[j] / Rj[j];
          for (int l = tid; l < j; l += kWave) gv[l] = gv[l] - Rj[l] * y;
          if (tid == 0) yv[j] = y;
          wave_lds_sync();
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < R; q++)
        if (w.live[q])
          for (int j = 0; j < kk; j++) x[q] = x[q] + yv[j] * g.V[(size_t)j * N + w.i[q]];
      if (conv) {
        status = NRT_OK;
        break;
      }
      if (it >= d.max_iter) break;
    }
    acc.iters += (unsigned long long)it;
    acc.cycles += (unsigned long long)cycles;
    acc.steps++;
    acc.last_iters = it;
    acc.restarts += cycles > 0 ? cycles - 1 : 0;
    acc.rr = rr;
    acc.bb = bb;
    if (tid == 0 && status != NRT_OK && d.st->status == NRT_OK) {
      d.st->status = status;
      d.st->fail_step = step;
      d.st->fail_iter = it;
      d.st->fail_rr = rr;
      d.st->fail_bb = bb;
      d.st->fail_cycles = cycles;
    }
    if (d.interval >= 0 && ++gl > d.interval) {
      gl = 0;
#pragma unroll
      for (int k = 0; k < R; k++)
        if (d.trace && w.live[k] && w.i[k] == d.trace_elem) d.trace[ksamp] = x[k];
      ksamp++;
    }
  }
#pragma unroll
  for (int k = 0; k < R; k++)
    if (w.live[k]) d.x[w.i[k]] = x[k];
  if (tid == 0) acc.store(d.st);
}

// ---------------------------------------------------------------- host side
static size_t kb_lds(int N) { return sizeof(double) * 2 * (size_t)(N + 1); }
static size_t kg_lds(int N, int m) {
  return sizeof(double) * (2 * (size_t)(N + 1) + 5 * (size_t)(m + 1) + 2 * (size_t)m);
}

// Whether a system runs here: every row in the threads' registers, the operands and
// (GMRES, FP64) the least-squares vectors in the LDS of one workgroup. GMRES:
// up to 4,096 rows (8 a thread, the first registers spilled; 4,000 rows: 67 us an
// Arnoldi step against 149 in a grid of two workgroups). BiCGSTAB: up to the 2,048 rows
// that the grid kernel gives to one workgroup; with 8 rows for each of 512 threads,
// 4,000 rows took 5.9 us an iteration against 33, but in another order of sums than the
// grid of two.
constexpr int kKbStaticLds = 4096;  // at most, beside the dynamic LDS
bool krylov_block_ok(int N, bool gmres, bool mixed, int restart, int max_lds) {
  if (N > (gmres ? kKgMaxN : kKbMaxN) || mixed) return false;
  return (gmres ? kg_lds(N, std::min(restart, N)) : kb_lds(N)) + kKbStaticLds <= (size_t)max_lds;
}

struct KbShape {
  const void* k;
  int threads;
  size_t lds;
};
static KbShape bicgstab_shape(int N) {
  // R > 1 takes all 256 threads: rows tid, tid + 256, ... as the grid kernel sums them
  const int R = N <= kKbThreads ? 1 : N <= 2 * kKbThreads ? 2 : N <= 4 * kKbThreads ? 4 : 8;
  const void* k = R == 1   ? (const void*)k_bicgstab_block<1>
                  : R == 2 ? (const void*)k_bicgstab_block<2>
                  : R == 4 ? (const void*)k_bicgstab_block<4>
                           : (const void*)k_bicgstab_block<8>;
  return KbShape{k, R == 1 ? grid_for(N, kWave) * kWave : kKbThreads, kb_lds(N)};
}
static KbShape gmres_shape(int N, int m) {
  // every wave also where the rows need fewer: they share out the basis vectors; above
  // 1,024 rows half of them, for the registers of 4 or 8 rows a thread
  if (N <= kKgThreads) return KbShape{(const void*)k_gmres_block<1, kKgThreads>, kKgThreads, kg_lds(N, m)};
  constexpr int half = kKgThreads / 2;
  const void* k = N <= 4 * half ? (const void*)k_gmres_block<4, half>
                                : (const void*)k_gmres_block<8, half>;
  return KbShape{k, half, kg_lds(N, m)};
}

// Once per handle: the kernel may use the LDS that its launches ask for (as much as any
// handle asks for: the limit is the kernel's, and handles of other sizes share it).
void krylov_block_prepare(int N, bool gmres, int m, int max_lds) {
  const KbShape q = gmres ? gmres_shape(N, m) : bicgstab_shape(N);
  if (q.lds > 48 * 1024)
    NRT_HIP(hipFuncSetAttribute(q.k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                max_lds - kKbStaticLds));
}

void bicgstab_block_launch(ImpDev d, hipStream_t s) {
  const KbShape q = bicgstab_shape(d.N);
  void* args[] = {&d};
  NRT_HIP(hipLaunchKernel(q.k, dim3(1), dim3(q.threads), args, q.lds, s));
}

void gmres_block_launch(ImpDev d, GmresDev<double> g, hipStream_t s) {
  const KbShape q = gmres_shape(d.N, g.m);
  void* args[] = {&d, &g};
  NRT_HIP(hipLaunchKernel(q.k, dim3(1), dim3(q.threads), args, q.lds, s));
}

}  // namespace nrt
