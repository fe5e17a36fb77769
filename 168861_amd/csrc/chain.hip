// Exact solve of an unbranched neurite (an axon with any number of Hodgkin-Huxley nodes
// up to one row in eight) with its rows resident in registers: a wave per 64 C rows.
//
// The matrix is tridiagonal. Levels, each the same elimination with one row kept:
//   lane  C rows: all but the last in terms of the last row of the lane before and its
//         own last row, x_i = y_i + p_i x_before + q_i x_last (Thomas, in registers)
//   wave  the lanes' last rows but lane 63's, by cyclic reduction over the lanes
//         (6 rounds of shuffles)
//   top   the waves' last rows (64 at most), by cyclic reduction; every wave does it
//         alone, from seven numbers that every wave sends to all
// so a step is one exchange and no barrier: the waves are workgroups of one, each on a
// CU of its own. The rows that gate are shared out over the lanes of their wave.
// What bounds a step is latency: the gating's exponentials, a chain of C reciprocals, two
// reductions of 6 rounds, the exchange. Measured, us a step: 1,012 rows (2 waves) 3.8,
// 20,202 rows (40 waves) 5.9, 60,602 rows (60 waves, 16 rows a lane) 6.8; by the general
// solve 43.7 (block form), 32.6 and 46.7 (local form).
// Its error against 64-bit elimination, 20 to 200 steps of axons of 1,012 to 60,602 rows:
// 8e-14 to 6.5e-11, that of the general solve 1.9e-12 to 1.6e-10.
#include <cstdlib>
#include "resident_dev.hpp"
#include "chain.hpp"

namespace nrt {

namespace {
struct Tri {  // x = d + a x_left + c x_right
  double a, c, d;
};
// One round at distance s among lanes 0 .. n-1: a neighbour s away is replaced by its own
// neighbours; a row whose neighbour on a side lies outside keeps its coefficient there.
__device__ __forceinline__ Tri chain_round(const Tri t, int lane, int s, int n) {
  const bool left = lane >= s && lane < n, right = lane + s < n;
  const int l = (lane - s) & 63, r = (lane + s) & 63;
  double aL = __shfl(t.a, l), cL = __shfl(t.c, l), dL = __shfl(t.d, l);
  double aR = __shfl(t.a, r), cR = __shfl(t.c, r), dR = __shfl(t.d, r);
  aL = left ? aL : 1.0;
  cL = left ? cL : 0.0;
  dL = left ? dL : 0.0;
  aR = right ? aR : 0.0;
  cR = right ? cR : 1.0;
  dR = right ? dR : 0.0;
  const double inv = rcp_newton(1.0 - fma(t.a, cL, t.c * aR));
  return {t.a * aL * inv, t.c * cR * inv, fma(t.a, dL, fma(t.c, dR, t.d)) * inv};
}
constexpr int kChRec = 7;  // a wave's numbers: A, B, D, S of its last row, y, p, q of its first
}  // namespace

template <int C>
__global__ __launch_bounds__(64) void k_chain(ImpDev d, ChainDev r, ResRun q) {
  __shared__ double s_v[C][64], s_dg[C][64], s_kd[C][64], s_cdt[C][64];
  const int lane = (int)threadIdx.x, w = (int)blockIdx.x, N = r.N, W = r.W;
  const int base = (w * 64 + lane) * C;
  double V[C], sub[C], sup[C];
  unsigned imask = 0;
  int tk = -1;
#pragma unroll
  for (int k = 0; k < C; k++) {
    const int j = base + k;
    const bool in = j < N;  // (rows past the end: 1 x = 0)
    const int at = in ? j : 0;
    const double v = r.x[at], a = r.sub[at], b = r.dg[at], c = r.sup[at], e = r.cdt[at],
                 f = r.kd[at];
    V[k] = in ? v : 0.0;
    sub[k] = in ? a : 0.0;
    sup[k] = in ? c : 0.0;
    s_dg[k][lane] = in ? b : 1.0;
    s_cdt[k][lane] = in ? e : 0.0;
    s_kd[k][lane] = in ? f : 0.0;
    if (r.inp && in && r.inp[j] != 0.0) imask |= 1u << k;
    if (q.trace && d.interval >= 0 && j == d.trace_elem) tk = k;
  }
  // the gating rows of this wave, one a lane
  const int e0 = r.woff[w], ne = r.woff[w + 1] - e0;
  const bool gates = lane < ne;
  HHGate gate{};
  HHRow hr{};
  double m = 0, h = 0, n = 0, hdx = 0;
  int hk = 0, ht = 0;
  if (gates) {
    const int row = r.hrow[e0 + lane], hh = r.hidx[e0 + lane];
    hk = row % C;
    ht = row / C - w * 64;
    gate = hh_gate_load(d.hh, hh);
    hr = hh_row_load(d, hh, row);
    hdx = d.dxv[row];
    const double* at = r.x + N + e0 + lane;
    m = at[0];
    h = at[r.H];
    n = at[2 * r.H];
  }
  long long gl = q.gl0, ks = 0;
  unsigned tag = q.tag0;
  unsigned long long most = q.first_limit;
  for (long long i = q.first; i < q.first + q.num; i++) {
    const bool active = i >= d.a0 && i <= d.a1;
    tag++;
    if (ne > 0) {
#pragma unroll
      for (int k = 0; k < C; k++) s_v[k][lane] = V[k];
      wave_lds_sync();
      if (gates) {
        double Wn, Kn;
        hh_gate_step(gate, s_v[hk][ht], d.dt_ms, m, h, n, Wn, Kn);
        s_dg[hk][ht] = hh_row_diag(hr, Wn);
        s_kd[hk][ht] = Kn * hdx;
      }
      wave_lds_sync();
    }
    // ---- the lane's rows
    double y[C - 1], p[C - 1], c[C - 1], bl;
    auto rhs = [&](int k) {
      double b = fma(s_cdt[k][lane], V[k], s_kd[k][lane]);
      if (active && (imask >> k & 1)) b = b + r.inp[base + k];
      return b;
    };
    {
      const double inv = rcp_newton(s_dg[0][lane]);
      y[0] = rhs(0) * inv;
      p[0] = -sub[0] * inv;
      c[0] = -sup[0] * inv;
    }
#pragma unroll
    for (int k = 1; k < C - 1; k++) {
      const double inv = rcp_newton(fma(sub[k], c[k - 1], s_dg[k][lane]));
      y[k] = fma(-sub[k], y[k - 1], rhs(k)) * inv;
      p[k] = -sub[k] * p[k - 1] * inv;
      c[k] = -sup[k] * inv;
    }
#pragma unroll
    for (int k = C - 3; k >= 0; k--) {  // c becomes q
      y[k] = fma(c[k], y[k + 1], y[k]);
      p[k] = fma(c[k], p[k + 1], p[k]);
      c[k] = c[k] * c[k + 1];
    }
    bl = rhs(C - 1);
    const double dl = s_dg[C - 1][lane], sl = sub[C - 1], sr = sup[C - 1];
    const double y6 = y[C - 2], p6 = p[C - 2], q6 = c[C - 2];
    // ---- the lanes' last rows
    Tri t;
    {
      const int nx = (lane + 1) & 63;
      const double yn = __shfl(y[0], nx), pn = __shfl(p[0], nx), qn = __shfl(c[0], nx);
      const double inv = rcp_newton(fma(sr, pn, fma(sl, q6, dl)));
      t = {-sl * p6 * inv, -sr * qn * inv, fma(-sr, yn, fma(-sl, y6, bl)) * inv};
    }
#pragma unroll
    for (int s = 1; s < 64; s *= 2) t = chain_round(t, lane, s, 63);
    // ---- the waves' last rows
    double rec[kChRec] = {};
    {
      const double a62 = __shfl(t.a, 62), c62 = __shfl(t.c, 62), d62 = __shfl(t.d, 62);
      // (lane 63: its row; lane 0: the wave's first row)
      const double A = sl * p6 * a62, B = fma(sl, fma(p6, c62, q6), dl);
      const double D = fma(-sl, fma(p6, d62, y6), bl);
      const double fy = fma(c[0], t.d, y[0]), fp = fma(c[0], t.a, p[0]), fq = c[0] * t.c;
      if (W == 1) {
        rec[0] = __shfl(A, 63);
        rec[1] = __shfl(B, 63);
        rec[2] = __shfl(D, 63);
      } else {
        unsigned long long* set = r.ll + (size_t)(tag & 1) * W * kChRec * 2;
        unsigned long long* o = set + (size_t)w * kChRec * 2;
        auto put = [&](int k, double v) {
          const unsigned long long tt = (unsigned long long)tag << 32;
          __hip_atomic_store(o + 2 * k, tt | (unsigned)__double2loint(v), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(o + 2 * k + 1, tt | (unsigned)__double2hiint(v), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        };
        if (lane == 63) {
          put(0, A);
          put(1, B);
          put(2, D);
          put(3, sr);
        }
        if (lane == 0) {
          put(4, fy);
          put(5, fp);
          put(6, fq);
        }
        __builtin_amdgcn_wave_barrier();  // both have put before any lane waits
        bool ok = true;
        if (lane < W) {
          const unsigned long long* at = set + (size_t)lane * kChRec * 2;
          unsigned long long x[2 * kChRec], spins = 0;
          while (true) {
            bool all = true;
#pragma unroll
            for (int k = 0; k < 2 * kChRec; k++) {
              x[k] = __hip_atomic_load(at + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              all = all && (unsigned)(x[k] >> 32) == tag;
            }
            if (all) break;
            // bounded; once another wave gave up, all do
            if (++spins > most ||
                ((spins & 255) == 0 &&
                 __hip_atomic_load(d.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
              __hip_atomic_store(d.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              ok = false;
              break;
            }
          }
#pragma unroll
          for (int k = 0; k < kChRec; k++)
            rec[k] = __hiloint2double((int)(unsigned)x[2 * k + 1], (int)(unsigned)x[2 * k]);
        }
        if (__any(!ok)) return;  // nothing was stored
        most = d.spin_limit;
      }
    }
    Tri u;
    {
      const int nx = (lane + 1) & 63;
      const bool last = lane >= W - 1;
      double fy = __shfl(rec[4], nx), fp = __shfl(rec[5], nx), fq = __shfl(rec[6], nx);
      const double S = last ? 0.0 : rec[3];
      fy = last ? 0.0 : fy;
      fp = last ? 0.0 : fp;
      fq = last ? 0.0 : fq;
      const double inv = rcp_newton(lane < W ? fma(S, fp, rec[1]) : 1.0);
      u = {-rec[0] * inv, -S * fq * inv, fma(-S, fy, rec[2]) * inv};
    }
    for (int s = 1; s < W; s *= 2) u = chain_round(u, lane, s, W);
    // ---- back
    const double xo = __shfl(u.d, w), xb = w > 0 ? __shfl(u.d, w - 1) : 0.0;
    const double xl = lane == 63 ? xo : fma(t.a, xb, fma(t.c, xo, t.d));
    double xp = __shfl(xl, (lane - 1) & 63);
    xp = lane == 0 ? xb : xp;
#pragma unroll
    for (int k = 0; k < C - 1; k++) V[k] = fma(p[k], xp, fma(c[k], xl, y[k]));
    V[C - 1] = xl;
    if (d.interval >= 0 && ++gl > d.interval) {
      gl = 0;
      if (tk >= 0) {
        double v = V[0];
#pragma unroll
        for (int k = 1; k < C; k++) v = tk == k ? V[k] : v;
        q.trace[ks] = v;
      }
      ks++;
    }
  }
#pragma unroll
  for (int k = 0; k < C; k++)
    if (base + k < N) r.xo[base + k] = V[k];
  if (gates) {
    double* at = r.xo + N + e0 + lane;
    at[0] = m;
    at[r.H] = h;
    at[2 * r.H] = n;
  }
}

void chain_launch(const ImpDev& d, const ChainDev& r, const ResRun& q, hipStream_t s) {
  if (r.C == 8) hipLaunchKernelGGL(k_chain<8>, dim3(r.W), dim3(64), 0, s, d, r, q);
  else hipLaunchKernelGGL(k_chain<16>, dim3(r.W), dim3(64), 0, s, d, r, q);
  NRT_HIP(hipGetLastError());
}

}  // namespace nrt
