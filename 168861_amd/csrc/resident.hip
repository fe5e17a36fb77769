// Tree solve with the rows resident in registers (resident.hpp): every row of a group's
// 512 units stays in its thread for the whole launch (V, c_m dx / dT, K dx and the two
// factors: 80 VGPRs for 8 rows), so a step touches memory only for the values that
// groups exchange.
#include <algorithm>
#include "resident_dev.hpp"

namespace nrt {

__device__ __forceinline__ double lane_get(double x, int byte_lane) {
  const int lo = __builtin_amdgcn_ds_bpermute(byte_lane, __double2loint(x));
  const int hi = __builtin_amdgcn_ds_bpermute(byte_lane, __double2hiint(x));
  return __hiloint2double(hi, lo);
}

// The dynamic rows' state in LDS (read by the service wave once a step: kept in its
// registers it would cost every wave of the workgroup the same registers).
struct DynRow {
  double v, m, h, n, cdt, kd, inp, diag0, s, u;  // s: static children's share of the pivot
  HHGate q;
  HHRow hr;
  int hh, row, parent;
  int src[2], node[2];  // children: published value (one group: piece) and top node
};
__device__ __forceinline__ void dyn_load(const ImpDev& d, const ResDev& r, int j, DynRow* out) {
  DynRow y{};
  y.row = r.drow[j];
  const double* at = r.x + (int64_t)r.G * kResC * r.T + j;
  y.v = at[0];
  y.cdt = d.cmdx[y.row] / d.dT;
  y.inp = d.input[y.row];
  y.diag0 = r.ddiag[j];
  y.s = r.ds[j];
  y.u = r.du[j];
  y.hh = r.dhh[j];
  if (y.hh >= 0) {
    y.m = at[r.nd];
    y.h = at[2 * r.nd];
    y.n = at[3 * r.nd];
    y.q = hh_gate_load(d.hh, y.hh);
    y.hr = hh_row_load(d, y.hh, y.row);
    y.kd = d.dxv[y.row];  // K comes with every step
  } else {
    y.kd = d.kdx[y.row];
  }
  const uint16_t* f = r.dinf + 6 * j;
  for (int k = 0; k < 2; k++) {
    y.src[k] = r.G > 1 ? f[2 * k] : f[2 * k] ? r.epiece[f[2 * k]] : r.T;
    y.node[k] = f[2 * k + 1];
  }
  y.parent = f[4] == 0xFFFF ? -1 : f[4];
  *out = y;
}
// The service wave, eight lanes a dynamic row: gating (hh_gate_step; lanes 0..5 of a row
// evaluate one rate function each, so it costs one exponential's latency instead of
// six), the diagonal and the right-hand side of the next step.
__device__ __forceinline__ void dyn_update(DynRow& y, const ImpDev& d, int lane, bool active,
                                           double& diag, double& b) {
  int k = lane & 7;
  asm volatile("" : "+v"(k));  // what depends on it is made again every step: kept, it would
                               // cost every wave of the workgroup its registers
  const double v = y.v;
  double kdx = y.kd;
  diag = y.diag0;
  if (y.hh >= 0) {
    const bool na = k < 4;  // m and h follow the sodium shift, n the potassium shift
    const double u = div_by((v + (na ? y.q.ls_Na : y.q.ls_K)) - y.q.rest, 0.001, 1000.0);
    // k: 0 am, 1 bm, 2 ah, 3 bh, 4 an, 5 bn; the operations of hh_rates: near 25 and 10 mV
    // am and an are quotients of two small numbers, whose errors cancel only where both
    // come from one rounded c0 - 0.1 u
    const bool quot = k == 0 || k == 3 || k == 4;
    const double c0 = k == 0 ? 2.5 : k == 3 ? 3.0 : 1.0;
    const double c1 = k == 1 ? 18.0 : k == 2 ? 20.0 : 80.0;
    const double y1 = k == 1 ? 1.0 / 18.0 : k == 2 ? 1.0 / 20.0 : 1.0 / 80.0;
    const double lin = c0 - 0.1 * u;
    const double e = exp(quot ? lin : div_by(-u, c1, y1));
    const double num = k == 0 ? lin : k == 4 ? 0.1 - 0.01 * u : 1.0;
    const double frac = num / (k == 3 ? e + 1 : e - 1);
    const double rate = k == 1 ? 4 * e : k == 2 ? 0.07 * e : k == 5 ? 0.125 * e : frac;
    const int base = (lane & ~7) * 4;
    const double am = lane_get(rate, base), bm = lane_get(rate, base + 4);
    const double ah = lane_get(rate, base + 8), bh = lane_get(rate, base + 12);
    const double an = lane_get(rate, base + 16), bn = lane_get(rate, base + 20);
    const double m0 = y.m, h0 = y.h, n0 = y.n, dt = d.dt_ms;
    const double m = m0 + dt * (am * (1 - m0) - bm * m0);
    const double h = h0 + dt * (ah * (1 - h0) - bh * h0);
    const double n = n0 + dt * (an * (1 - n0) - bn * n0);
    const double gna = y.q.g_Na * m * m * m * h;
    const double gk = y.q.g_K * n * n * n * n;
    const double gl = y.q.G_L;
    const double W = -(gna + gk + gl);
    const double K = gna * y.q.E_Na + gk * y.q.E_K + gl * y.q.E_L;
    diag = hh_row_diag(y.hr, W);
    kdx = K * y.kd;
    wave_lds_sync();
    y.m = m;  // the row's lanes store the same values
    y.h = h;
    y.n = n;
  }
  b = fma(y.cdt, v, kdx);
  if (active) b = b + y.inp;
}

// LDS of a workgroup. K dx of a thread's rows lies kResKd values apart (odd: no bank
// conflict, and one address register for all rows).
constexpr int kResKd = kResC + 1;
struct ResLds {
  double *kd, *O, *In, *X, *pub, *dO, *din, *dX, *tz, *te, *dd, *db, *dr;
  uint16_t* tinf;
  int32_t* thoff;
  int* fail;
  DynRow* dyn;
  __device__ static ResLds carve(unsigned char* p, const ResDev& r) {
    ResLds s;
    s.dyn = (DynRow*)p;
    double* q = (double*)(s.dyn + r.nd);
    auto take = [&](int n) {
      double* at = q;
      q += n;
      return at;
    };
    s.kd = take(kResKd * r.T);
    s.O = take(r.T + 1);
    s.In = take(r.T);
    s.X = take(r.T + 1);
    s.pub = take(r.npub);
    s.dO = take(r.nt + 1);
    s.din = take(r.nt + 1);
    s.dX = take(r.nt + 1 + r.nd);
    s.tz = take(r.nt);
    s.te = take(r.nt);
    s.dd = take(kResDyn);
    s.db = take(kResDyn);
    s.dr = take(kResDyn);
    s.tinf = (uint16_t*)q;
    s.thoff = (int32_t*)(s.tinf + 6 * r.nt);
    s.fail = (int*)(s.thoff + r.nth + 1);
    return s;
  }
};

__device__ __forceinline__ void ll_put(unsigned long long* ll, int e, unsigned tag, double v) {
  const unsigned long long t = (unsigned long long)tag << 32;
  __hip_atomic_store(ll + 2 * e, t | (unsigned)__double2loint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(ll + 2 * e + 1, t | (unsigned)__double2hiint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Top of the tree, its heights up: whole-workgroup heights with a barrier each, then
// the narrow ones by the first wave alone (LDS operations of a wave keep their order).
__device__ __forceinline__ void res_top_up(const ResLds& s, int j) {
  const uint16_t* f = s.tinf + 6 * j;
  const double in = (s.pub[f[0]] + s.dO[f[1]]) + (s.pub[f[2]] + s.dO[f[3]]);
  s.din[j] = in;
  s.dO[j] = s.tz[j] * in;
}
__device__ __forceinline__ void res_top_down(const ResLds& s, int j) {
  const uint16_t* f = s.tinf + 6 * j;
  s.dX[j] = s.te[j] * s.din[j] + s.tz[j] * (s.dX[f[4]] + s.pub[f[5]]);
}

// Dynamic rows: pivots and right-hand sides with the children's shares, elimination
// and back-substitution (lane 0 of the service wave; one row in most neurites). pub:
// where the children's values lie (one group: its pieces' own).
__device__ __forceinline__ void res_dyn_solve(const ResDev& r, const ResLds& s, const double* pub) {
  for (int j = 0; j < r.nd; j++) {
    const DynRow& y = s.dyn[j];
    s.dd[j] = s.dd[j] - y.s;
    s.dr[j] = s.db[j] + (pub[y.src[0]] + s.dO[y.node[0]]) + (pub[y.src[1]] + s.dO[y.node[1]]);
  }
  for (int j = 0; j < r.nd - 1; j++) {  // (the last row is the root or stands alone)
    const int p = s.dyn[j].parent;
    if (p < 0) continue;
    const double u = s.dyn[j].u, f = u / s.dd[j];
    s.dd[p] = s.dd[p] - f * u;
    s.dr[p] = s.dr[p] - f * s.dr[j];
  }
  for (int j = r.nd - 1; j >= 0; j--) {
    const int p = s.dyn[j].parent;
    const double up = p < 0 ? 0.0 : s.dyn[j].u * s.dX[r.nt + 1 + p];
    s.dX[r.nt + 1 + j] = (s.dr[j] - up) * rcp_newton(s.dd[j]);
  }
}

// Steps of one group. The block has T' >= T unit threads and one service wave; waves
// beyond the group's T units only take part in the barriers.
__device__ __forceinline__ void resident_steps(const ImpDev& d, const ResDev& r, const ResRun& q,
                                               int g, unsigned char* lds) {
  constexpr int C = kResC;
  const int T = r.T, tid = (int)threadIdx.x, lane = tid & (kWave - 1);
  const int nunit = (int)blockDim.x - kWave;
  const bool service = tid >= nunit;
  const bool on = tid < T && !service;
  const ResLds s = ResLds::carve(lds, r);
  const int np = r.ginfo[4 * g], nh = r.ginfo[4 * g + 1], hn = r.ginfo[4 * g + 2];
  const bool exch = r.ginfo[4 * g + 3] != 0 && r.G > 1;
  // ---- the group's rows and coefficients
  double V[C], cdt[C], F[C], I[C];  // K dx in LDS: 168 VGPRs are what nine waves get
  double uz = 0, ubel = 0, uabv = 0, ucum = 0, uein = 0, ubin = 0;
  uint32_t w0 = kResNone | (1u << 16), w1 = (uint32_t)r.nt,
           w2 = (uint32_t)r.nt | ((uint32_t)T << 16);
  const int64_t U = (int64_t)r.G * T, u0 = (int64_t)g * T + tid;
#pragma unroll
  for (int k = 0; k < C; k++) V[k] = cdt[k] = F[k] = I[k] = 0.0;
  unsigned inmask = 0;
  if (on) {
#pragma unroll
    for (int k = 0; k < C; k++) {
      const int64_t at = ((int64_t)g * C + k) * T + tid;
      V[k] = r.x[at];
      cdt[k] = r.cdt[at];
      s.kd[kResKd * tid + k] = r.kd[at];
      F[k] = r.F[at];
      I[k] = r.I[at];
      if (r.has_input && r.inp[at] != 0.0) inmask |= 1u << k;
    }
    uz = r.uco[kUZ * U + u0];
    ubel = r.uco[kUBelow * U + u0];
    uabv = r.uco[kUAbove * U + u0];
    ucum = r.uco[kUCum * U + u0];
    uein = r.uco[kUEin * U + u0];
    ubin = r.uco[kUBin * U + u0];
    w0 = r.uinf[3 * u0];
    w1 = r.uinf[3 * u0 + 1];
    w2 = r.uinf[3 * u0 + 2];
  }
  const int piece = (int)(w0 & 0x3FF), pos = (int)(w0 >> 10 & 63), len = (int)(w0 >> 16 & 127);
  const bool has = piece != kResNone, top = w0 >> 31 != 0;
  const bool first = has && pos == 0, last = has && pos + 1 == len;
  // coefficients of the lane scans: round i combines with the lane 2^i further
  double up[kResRounds], dn[kResRounds];
  up[0] = has && !last ? uz : 0.0;
  dn[0] = has && !first ? uz : 0.0;
#pragma unroll
  for (int i = 1; i < kResRounds; i++) {
    up[i] = up[i - 1] * lane_get(up[i - 1], ((lane + (1 << (i - 1))) & 63) * 4);
    dn[i] = dn[i - 1] * lane_get(dn[i - 1], ((lane - (1 << (i - 1))) & 63) * 4);
  }
  // pieces by height: thread p < np has piece p
  double pz = 0;
  int pc0 = T, pc1 = T, pp = T, ph = -1, pa = 0, px = 0;
  if (tid < np && !service) {
    const uint16_t* f = r.pinf + 8 * u0;
    pz = r.pz[u0];
    pc0 = f[0];
    pc1 = f[1];
    pp = f[2];
    ph = f[3];
    pa = f[4];
    px = f[5];
  }
  for (int i = tid; i < T; i += (int)blockDim.x) {
    s.O[i] = s.In[i] = s.X[i] = 0.0;
  }
  for (int i = tid; i < r.npub; i += (int)blockDim.x) s.pub[i] = 0.0;
  for (int i = tid; i < r.nt; i += (int)blockDim.x) {
    s.tz[i] = r.tz[i];
    s.te[i] = r.te[i];
  }
  for (int i = tid; i <= r.nt; i += (int)blockDim.x) s.dO[i] = s.din[i] = s.dX[i] = 0.0;
  for (int i = tid; i < 6 * r.nt; i += (int)blockDim.x) s.tinf[i] = r.tinf[i];
  for (int i = tid; i <= r.nth; i += (int)blockDim.x) s.thoff[i] = r.thoff[i];
  if (tid == 0) {
    s.O[T] = s.X[T] = 0.0;
    *s.fail = 0;
  }
  if (service && lane < r.nd) dyn_load(d, r, lane, s.dyn + lane);
  const bool dlane = service && (lane >> 3) < r.nd;
  // the probe's place
  int tk = -1;
  bool tdyn = false;
  if (d.interval >= 0 && q.trace) {
    const int64_t base = (int64_t)g * C * T, at = d.trace_elem;
    if (at >= base && at < base + (int64_t)C * T && on && (int)((at - base) % T) == tid)
      tk = (int)((at - base) / T);
    tdyn = service && lane == 0 && g == r.owner && at >= (int64_t)r.G * C * T;
  }
  long long gl = q.gl0, ksamp = 0;
  unsigned tag = q.tag0;
  bool stimulus = false;
  lds_sync();
  for (long long step = q.first; step < q.first + q.num; step++) {
    const bool active = step >= d.a0 && step <= d.a1;
    tag++;
    double rh[C], obel = 0;
    if (active != stimulus) {
      // the stimulus goes on or off: into K dx of the own rows that it enters
      stimulus = active;
      if (inmask != 0) {
#pragma unroll 1
        for (int k = 0; k < C; k++) {
          if (!(inmask >> k & 1)) continue;
          const int64_t at = ((int64_t)g * C + k) * T + tid;
          s.kd[kResKd * tid + k] = active ? r.kd[at] + r.inp[at] : r.kd[at];
        }
      }
    }
    if (!service) {
      // ---- right-hand sides, the units' values going up, scan over the piece
#pragma unroll
      for (int k = 0; k < C; k++) rh[k] = fma(cdt[k], V[k], on ? s.kd[kResKd * tid + k] : 0.0);
      double o = rh[C - 1];
#pragma unroll
      for (int k = C - 2; k >= 0; k--) o = fma(F[k + 1], o, rh[k]);
      o = F[0] * o;
#pragma unroll
      for (int i = 0; i < kResRounds; i++)
        if (i < r.rounds) o = fma(up[i], lane_get(o, ((lane + (1 << i)) & 63) * 4), o);
      if (first) s.O[piece] = o;
      obel = lane_get(o, ((lane + 1) & 63) * 4);
      if (!has || last) obel = 0.0;
    } else if (dlane) {
      double diag, b;
      dyn_update(s.dyn[lane >> 3], d, lane, active, diag, b);
      if ((lane & 7) == 0) {
        s.dd[lane >> 3] = diag;
        s.db[lane >> 3] = b;
      }
    }
    lds_sync();
    // ---- the group's pieces by heights, up
    for (int h = 1; h < hn; h++) {
      if (ph == h) {
        const double in = s.O[pc0] + s.O[pc1];
        s.In[tid] = in;
        s.O[tid] = fma(pz, in, s.O[tid]);
      }
      lds_sync();
    }
    if (tid < kWave) {
      for (int h = hn; h < nh; h++) {
        if (ph == h) {
          const double in = s.O[pc0] + s.O[pc1];
          s.In[tid] = in;
          s.O[tid] = fma(pz, in, s.O[tid]);
        }
        wave_lds_sync();
      }
    }
    lds_sync();
    unsigned long long* ll = r.ll + (size_t)(tag & 1) * 2 * r.npub;
    if (exch && pa) ll_put(ll, pa, tag, s.O[tid]);
    double scan = 0;
    if (!service) {
      // ---- units again with what enters below them, then down with nothing above
      double acc = has ? fma(ubel, s.In[piece], obel) : 0.0;
      acc = acc + rh[C - 1];
      rh[C - 1] = acc;
#pragma unroll
      for (int k = C - 2; k >= 0; k--) {
        acc = fma(F[k + 1], acc, rh[k]);
        rh[k] = acc;
      }
#pragma unroll
      for (int k = 0; k < C; k++) rh[k] = I[k] * rh[k];  // I r' from here on
      double x = rh[0];
#pragma unroll
      for (int k = 1; k < C; k++) x = fma(F[k], x, rh[k]);
#pragma unroll
      for (int i = 0; i < kResRounds; i++)
        if (i < r.rounds) x = fma(dn[i], lane_get(x, ((lane - (1 << i)) & 63) * 4), x);
      if (last) s.X[piece] = x;
      scan = lane_get(x, ((lane - 1) & 63) * 4);
      if (!has || first) scan = 0.0;
    } else if (!exch && lane == 0 && r.nd > 0) {
      res_dyn_solve(r, s, s.O);
    }
    lds_sync();
    // ---- pieces down (by descending height; leaves' values are used nowhere but in
    // what the group publishes)
    if (tid < kWave) {
      for (int h = nh - 1; h >= hn; h--) {
        if (ph == h) s.X[tid] = fma(pz, s.X[pp], s.X[tid]);
        wave_lds_sync();
      }
    }
    lds_sync();
    for (int h = hn - 1; h >= 1; h--) {
      if (ph == h) s.X[tid] = fma(pz, s.X[pp], s.X[tid]);
      lds_sync();
    }
    // ---- exchange and the top
    if (exch) {
      if (px) ll_put(ll, px, tag, ph == 0 ? fma(pz, s.X[pp], s.X[tid]) : s.X[tid]);
      const unsigned long long limit = step == q.first ? q.first_limit : d.spin_limit;
      for (int e = 1 + tid; e < r.npub; e += (int)blockDim.x) {
        unsigned long long a, b, spins = 0;
        while (true) {
          a = __hip_atomic_load(ll + 2 * e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          b = __hip_atomic_load(ll + 2 * e + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if ((unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag) break;
          // bounded: after `limit` polls, or once another workgroup gave up, drain
          if (++spins > limit ||
              ((spins & 255) == 0 &&
               __hip_atomic_load(d.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
            __hip_atomic_store(d.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *s.fail = 1;
            break;
          }
        }
        s.pub[e] = __hiloint2double((int)(unsigned)b, (int)(unsigned)a);
      }
      lds_sync();
      if (*s.fail) {  // uniform: read after the barrier
        // A launch from one buffer to the other has spoiled nothing: the host, which reads
        // *d.err, tries it again. In place, other groups may have taken the launch's last
        // step, so whichever gives up says that the neurite's state is lost.
        int ok = NRT_OK;
        if (tid == 0 && r.xo == r.x &&
            __hip_atomic_compare_exchange_strong(&d.st->status, &ok, (int)NRT_ERR_HIP,
                                                 __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
          d.st->fail_step = step;
        return;
      }
      for (int h = 0; h < r.top_narrow; h++) {
        for (int j = s.thoff[h] + tid; j < s.thoff[h + 1]; j += (int)blockDim.x) res_top_up(s, j);
        lds_sync();
      }
      if (tid < kWave) {
        for (int h = r.top_narrow; h < r.nth; h++) {
          const int j = s.thoff[h] + tid;
          if (j < s.thoff[h + 1]) res_top_up(s, j);
          wave_lds_sync();
        }
      }
      lds_sync();
      if (service && lane == 0 && r.nd > 0) res_dyn_solve(r, s, s.pub);
      lds_sync();
      if (tid < kWave) {
        for (int h = r.nth - 1; h >= r.top_narrow; h--) {
          const int j = s.thoff[h] + tid;
          if (j < s.thoff[h + 1]) res_top_down(s, j);
          wave_lds_sync();
        }
      }
      lds_sync();
      for (int h = r.top_narrow - 1; h >= 0; h--) {
        for (int j = s.thoff[h] + tid; j < s.thoff[h + 1]; j += (int)blockDim.x) res_top_down(s, j);
        lds_sync();
      }
    }
    // ---- the units' potentials
    if (!service) {
      double xin = has ? fma(uabv, s.X[w2 >> 16], scan) : 0.0;
      xin = fma(ucum, s.dX[w1 & 0xFFFF] + s.pub[w1 >> 16], xin);
      if (top) {
        const double di = s.din[w2 & 0xFFFF];
        xin = fma(uein, di, xin);
        double acc = ubin * di;
#pragma unroll
        for (int k = C - 1; k >= 0; k--) {
          rh[k] = fma(I[k], acc, rh[k]);
          acc = F[k] * acc;
        }
      }
      double x = xin;
#pragma unroll
      for (int k = 0; k < C; k++) {
        x = fma(F[k], x, rh[k]);
        V[k] = x;
      }
    } else if (lane < r.nd) {
      s.dyn[lane].v = s.dX[r.nt + 1 + lane];
    }
    if (d.interval >= 0 && ++gl > d.interval) {
      gl = 0;
      if (tk >= 0) {
        double v = V[0];
#pragma unroll
        for (int k = 1; k < C; k++) v = tk == k ? V[k] : v;
        q.trace[ksamp] = v;
      }
      if (tdyn) q.trace[ksamp] = s.dX[r.nt + 1 + (d.trace_elem - (int64_t)r.G * C * T)];
      ksamp++;
    }
    // (the next step's first writes to LDS, O and the dynamic rows' values, touch
    // nothing that is read since the last barrier)
  }
  if (on) {
#pragma unroll
    for (int k = 0; k < C; k++) r.xo[((int64_t)g * C + k) * T + tid] = V[k];
  }
  if (service && g == r.owner) {
    if (lane < r.nd) {
      const DynRow& y = s.dyn[lane];
      double* at = r.xo + (int64_t)r.G * C * T + lane;
      at[0] = y.v;
      at[r.nd] = y.m;
      at[2 * r.nd] = y.h;
      at[3 * r.nd] = y.n;
    }
    if (lane == 0 && q.num > 0) {
      d.st->iters_total += (unsigned long long)q.num;
      d.st->steps += (unsigned long long)q.num;
      d.st->last_iters = 1;
    }
  }
}

constexpr int kResBlock = kResT + kWave;

__global__ __launch_bounds__(kResBlock) void k_resident(ImpDev d, ResDev r, ResRun q) {
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  resident_steps(d, r, q, (int)blockIdx.x, dyn_lds);
}

// Slots of a batch: workgroup w of the launch order runs map[w] = (slot, group) for the
// slot's work[].steps steps. Workgroups take their place in that order when they start
// (a ticket), so of all neurites that exchange values at most one, the last begun, lacks
// workgroups that have not started: the others end and make room for them, however
// many neurites a launch holds.
__global__ __launch_bounds__(kResBlock) void k_resident_batch(const ResRec* __restrict__ recs,
                                                              const ResWork* __restrict__ work,
                                                              const int2* __restrict__ map,
                                                              unsigned* __restrict__ ticket) {
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  __shared__ unsigned mine;
  if (threadIdx.x == 0) mine = atomicAdd(ticket, 1u);
  __syncthreads();
  const int2 m = map[__builtin_amdgcn_readfirstlane(mine)];
  const ResRec& rec = recs[m.x];
  const ResWork wk = work[m.x];
  ResRun q{wk.done + 1, wk.steps, 0, (unsigned)wk.done, nullptr, rec.d.spin_limit};
  if (rec.d.interval >= 0) {
    q.gl0 = wk.done % (rec.d.interval + 1);
    if (rec.trace_base) q.trace = rec.trace_base + wk.done / (rec.d.interval + 1);
  }
  resident_steps(rec.d, rec.r, q, m.y, dyn_lds);
}

// ---------------------------------------------------------------- host side
size_t resident_lds(const ResDev& r) {
  return resident_lds_bytes(r.T, r.npub, r.nt, r.nth, r.nd) + sizeof(DynRow) * r.nd;
}

// Workgroups of T unit threads that can be resident at once on the device.
int resident_capacity(int device, int T, size_t lds) {
  int cus = 0, per = 0, max_lds = 0;
  NRT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  NRT_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
  if (lds > 48 * 1024)  // (near the device's limit: handles of other sizes keep theirs)
    for (const void* k : {(const void*)k_resident, (const void*)k_resident_batch})
      NRT_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, max_lds - 1024));
  NRT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_resident_batch,
                                                       T + kWave, lds));
  return cus * per;
}

void resident_launch(const ImpDev& d, const ResDev& r, const ResRun& q, hipStream_t s) {
  ImpDev dd = d;
  ResDev rr = r;
  ResRun qq = q;
  void* args[] = {&dd, &rr, &qq};
  NRT_HIP(hipLaunchKernel((const void*)k_resident, dim3(r.G), dim3(r.T + kWave), args,
                          resident_lds(r), s));
}

void resident_batch_launch(const void* recs, const void* work, const int2* map, unsigned* ticket,
                           int nwg, int T, size_t lds, hipStream_t s) {
  if (nwg <= 0) return;
  void* args[] = {(void*)&recs, (void*)&work, (void*)&map, (void*)&ticket};
  NRT_HIP(hipLaunchKernel((const void*)k_resident_batch, dim3(nwg), dim3(T + kWave), args, lds,
                          s));
}

}  // namespace nrt
