// Whole runs of an unbranched neurite (an axon, every element HH or not) by the explicit
// step, on several CUs.
//
// A thread owns one element: its coefficients, its gates and HH parameters stay in
// registers for the launch, and a step is one barrier (potentials double buffered in
// LDS). What bounds a step is an element's chain of six exponentials and ten divisions,
// so the elements are spread over many workgroups of 256 threads (one wave a SIMD), each
// with a halo of kCabHalo elements on either side that it computes as well: the halo's
// outermost element lacks a neighbour, so one element a step becomes wrong from the
// edges, and after kCabHalo steps the workgroups exchange the halos' values (V and the
// gates, as words tagged with the exchange's number, polled by the element's thread).
// One exchange costs about 2.5 us, a step about 0.8. Measured (1,002 HH elements, per
// step): 5.1 us in one workgroup of 1,024 threads that read the parameters from L2
// every step, 1.12 here; 20,000 elements 1.15 (a launch a step before).
//
// Every operation is explicit_element's, operand for operand; divisions by constants
// (0.001, 18, 20, 80, r_a dx) are made of the divisor's reciprocal and one correction
// (div_by), which rounds as the division does.
#include <chrono>
#include <memory>
#include <thread>
#include "explicit_dev.hpp"

namespace nrt {

std::shared_ptr<void> device_share(int device, int cus);  // implicit.hip

constexpr int kCabBlock = 256;
constexpr int kCabHalo = 8;
constexpr int kCabOwn = kCabBlock - 2 * kCabHalo;
constexpr int kCabState = 4;  // V, m, h, n

// x / c from y = 1 / c (rounded): the quotient's first estimate, its exact remainder,
// one correction.
__device__ __forceinline__ double div_by(double x, double c, double y) {
  const double q = x * y;
  return fma(fma(-c, q, x), y, q);
}

struct CabArgs {
  int N, G;
  const double* Vin;
  double* Vout;
  const double *coefA, *rdx, *wdx, *kdx;
  const uint32_t* code;
  const ExRec* recs;
  HHDev hd;                  // m, h, n of the step before
  double *mo, *ho, *no;      // after the run
  double dt_ms;
  long long first, num, a0, a1, interval;
  int trace_elem;
  double* trace;
  unsigned long long* ll;    // [2][G][2 sides][kCabHalo][kCabState] words of two
  unsigned* err;
  unsigned tag0;
  unsigned long long first_limit, limit;
};

// Both words of a value carry the exchange's tag (see resident.hip).
__device__ __forceinline__ void cab_put(unsigned long long* w, unsigned tag, double v) {
  const unsigned long long t = (unsigned long long)tag << 32;
  __hip_atomic_store(w, t | (unsigned)__double2loint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(w + 1, t | (unsigned)__double2hiint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(kCabBlock) void k_explicit_cable(CabArgs q) {
  __shared__ double sv[2][kCabBlock + 2];  // one more on either side: never valid
  __shared__ int fail;
  const int t = (int)threadIdx.x, g = (int)blockIdx.x;
  const int halo = q.G > 1 ? kCabHalo : 0;
  const int j = g * (kCabBlock - 2 * halo) - halo + t;  // the thread's element
  const bool in = j >= 0 && j < q.N;
  const int N = q.N;
  // (the last element takes the new potential of the one before it, so the two belong
  // to one workgroup)
  const int place = in && j == N - 1 && j > 0 ? t - 1 : t;
  const bool own = in && place >= halo && place < kCabBlock - halo;
  // ---- the element's constants
  double v = 0, a = 0, rj = 1, rp = 1, w = 0, k = 0, inp = 0;
  double m = 0, h = 0, n = 0;
  double rest = 0, lsn = 0, lsk = 0, gNa = 0, gK = 0, gL = 0, eNa = 0, eK = 0, eL = 0, dx = 0;
  int hh = -1;
  const bool computed = in && j >= 1 && j <= N - 2;
  if (in) {
    if (own) v = q.Vin[j];
    if (computed) {
      a = q.coefA[j];
      rj = q.rdx[j];
      rp = q.rdx[j + 1];
      w = q.wdx[j];
      k = q.kdx[j];
      const uint32_t c = q.code[j];
      if (c >> 29 == kExRecord) {  // an exception record: a stimulus, an HH source of a sealed end
        const ExRec& r = q.recs[c & kCodeIdx];
        hh = r.hh;
        if (r.flags & 2) inp = r.input;
      } else if (c >> 29 == kExHH) {
        hh = (int)(c & kCodeIdx);
      }
    }
  }
  if (hh >= 0) {
    rest = q.hd.rest[hh];
    lsn = q.hd.ls_Na[hh];
    lsk = q.hd.ls_K[hh];
    gNa = q.hd.g_Na[hh];
    gK = q.hd.g_K[hh];
    gL = q.hd.G_L[hh];
    eNa = q.hd.E_Na[hh];
    eK = q.hd.E_K[hh];
    eL = q.hd.E_L[hh];
    dx = q.hd.dx[hh];
    if (own) {
      m = q.hd.m[hh];
      h = q.hd.h[hh];
      n = q.hd.n[hh];
    }
  }
  const double yj = 1 / rj, yp = 1 / rp;
  if (t == 0) {
    sv[0][0] = sv[1][0] = 0.0;
    sv[0][kCabBlock + 1] = sv[1][kCabBlock + 1] = 0.0;
    fail = 0;
  }
  const bool put_l = halo && own && g > 0 && t < 2 * halo;                   // for g - 1
  const bool put_r = halo && own && g + 1 < q.G && t >= kCabBlock - 2 * halo;  // for g + 1
  const bool get = in && !own;
  // a halo element's values: side 1 of the left neighbour, side 0 of the right one
  const int src_g = t < halo ? g - 1 : g + 1, src_side = t < halo ? 1 : 0;
  const int src_k = t < halo ? t : t - (kCabBlock - halo);
  long long gl = 0, ks = 0;
  unsigned tag = q.tag0;
  int p = 0;
  int left = 0;  // steps until the next exchange
  bool first_ex = true;
  for (long long i = q.first; i < q.first + q.num; i++) {
    if (halo && left == 0) {
      left = halo;
      tag++;
      unsigned long long* ll =
          q.ll + (size_t)(tag & 1) * q.G * 2 * kCabHalo * kCabState * 2;
      auto at = [&](int gg, int side, int kk) {
        return ll + ((((size_t)gg * 2 + side) * kCabHalo + kk) * kCabState) * 2;
      };
      if (put_l) {
        unsigned long long* o = at(g, 0, t - halo);
        cab_put(o, tag, v);
        if (hh >= 0) {
          cab_put(o + 2, tag, m);
          cab_put(o + 4, tag, h);
          cab_put(o + 6, tag, n);
        }
      }
      if (put_r) {
        unsigned long long* o = at(g, 1, t - (kCabBlock - 2 * halo));
        cab_put(o, tag, v);
        if (hh >= 0) {
          cab_put(o + 2, tag, m);
          cab_put(o + 4, tag, h);
          cab_put(o + 6, tag, n);
        }
      }
      if (get) {
        const unsigned long long* o = at(src_g, src_side, src_k);
        const int nw = hh >= 0 ? 2 * kCabState : 2;
        const unsigned long long most = first_ex ? q.first_limit : q.limit;
        unsigned long long x[2 * kCabState], spins = 0;
        while (true) {
          bool all = true;
#pragma unroll
          for (int e = 0; e < 2 * kCabState; e++)
            if (e < nw) {
              x[e] = __hip_atomic_load(o + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              all = all && (unsigned)(x[e] >> 32) == tag;
            }
          if (all) break;
          // bounded; once another workgroup gave up, all do
          if (++spins > most ||
              ((spins & 255) == 0 &&
               __hip_atomic_load(q.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u)) {
            __hip_atomic_store(q.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            fail = 1;
            break;
          }
        }
        v = __hiloint2double((int)(unsigned)x[1], (int)(unsigned)x[0]);
        if (hh >= 0) {
          m = __hiloint2double((int)(unsigned)x[3], (int)(unsigned)x[2]);
          h = __hiloint2double((int)(unsigned)x[5], (int)(unsigned)x[4]);
          n = __hiloint2double((int)(unsigned)x[7], (int)(unsigned)x[6]);
        }
      }
      first_ex = false;
      sv[p][t + 1] = v;
      lds_sync();
      if (fail) return;  // uniform: read after the barrier; nothing was stored
    } else if (i == q.first) {
      sv[p][t + 1] = v;
      lds_sync();
    }
    left--;
    const bool active = i >= q.a0 && i <= q.a1;
    const double vm = sv[p][t], vp = sv[p][t + 2];
    double wd = w, kd = k;
    if (hh >= 0) {
      const double un = div_by((v + lsn) - rest, 0.001, 1000.0);
      const double uk = div_by((v + lsk) - rest, 0.001, 1000.0);
      const double am = (2.5 - 0.1 * un) / (exp(2.5 - 0.1 * un) - 1);
      const double bm = 4 * exp(div_by(-un, 18.0, 1.0 / 18.0));
      const double ah = 0.07 * exp(div_by(-un, 20.0, 1.0 / 20.0));
      const double bh = 1 / (exp(3 - 0.1 * un) + 1);
      const double an = (0.1 - 0.01 * uk) / (exp(1 - 0.1 * uk) - 1);
      const double bn = 0.125 * exp(div_by(-uk, 80.0, 1.0 / 80.0));
      const double m0 = m, h0 = h, n0 = n;
      m = m0 + q.dt_ms * (am * (1 - m0) - bm * m0);
      h = h0 + q.dt_ms * (ah * (1 - h0) - bh * h0);
      n = n0 + q.dt_ms * (an * (1 - n0) - bn * n0);
      const double gna = gNa * m * m * m * h;
      const double gk = gK * n * n * n * n;
      const double W = -(gna + gk + gL);
      const double K = gna * eNa + gk * eK + gL * eL;
      wd = W * dx;
      kd = K * dx;
    }
    double s = div_by(vp - v, rp, yp);
    s = s + div_by(vm - v, rj, yj);
    s = s + wd * v;
    s = s + kd;
    if (active && inp != 0.0) s = s + inp;
    double vn = v + a * s;
    p ^= 1;
    // sealed ends: element 0 takes element 1's potential, element N - 1 that before it
    if (computed) {
      sv[p][t + 1] = vn;
      if (j == 1) sv[p][t] = vn;
      if (j == N - 2) sv[p][t + 2] = vn;
    } else if (!in) {
      sv[p][t + 1] = 0.0;
    }
    lds_sync();
    v = computed ? vn : sv[p][t + 1];
    if (q.interval >= 0 && ++gl > q.interval) {
      gl = 0;
      if (q.trace && own && j == q.trace_elem) q.trace[ks] = v;
      ks++;
    }
  }
  if (own) {
    q.Vout[j] = v;
    if (hh >= 0) {
      q.mo[hh] = m;
      q.ho[hh] = h;
      q.no[hh] = n;
    }
  }
}

// ---------------------------------------------------------------- host side
// Unbranched neurites whose sealed ends are the first and the last element, with no HH
// element among those two: any mix of HH and passive elements, stimuli anywhere; up to
// kResMaxN elements, above which a run is specified as a launch a step.
void cable_prepare(nrt_handle* hnd, Explicit* e, const HostProblem& p, bool in_batch) {
  const int N = p.N;
  if (in_batch || N < 4 || N > kResMaxN) return;
  for (int j = 1; j < N - 1; j++)
    if (p.mother[j] != j - 1 || p.dr[j] != j + 1 || p.branching[j]) return;
  bool last = false;
  for (int k = 0; k < p.T; k++) {
    if (p.terminals[k] != 0 && p.terminals[k] != N - 1) return;
    if (k > 0 && p.terminals[k] == 0) return;
    last = last || p.terminals[k] == N - 1;
  }
  if (p.T < 1 || p.terminals[0] != 0 || !last || p.mother[N - 1] != N - 2) return;
  for (int i = 0; i < p.H; i++)
    if (p.hh_elem[i] == 0 || p.hh_elem[i] == N - 1) return;
  const int G = N <= kCabBlock ? 1 : grid_for(N - 1, kCabOwn);
  int cus = 0, per = 0;
  NRT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, hnd->device));
  NRT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_explicit_cable, kCabBlock, 0));
  if (G > cus * per) return;
  e->cable_groups = G;
  e->m2.alloc(p.H);
  e->h2.alloc(p.H);
  e->n2.alloc(p.H);
  e->err.alloc(1);
  NRT_HIP(hipMemsetAsync(e->err.p, 0, sizeof(unsigned), hnd->stream));
  if (G > 1) {
    e->ll.alloc((size_t)2 * G * 2 * kCabHalo * kCabState * 2);
    NRT_HIP(hipMemsetAsync(e->ll.p, 0, sizeof(unsigned long long) * e->ll.n, hnd->stream));
  }
}

bool cable_run(nrt_handle* hnd, Explicit* e, int64_t first, int64_t num, int64_t a0, int64_t a1,
               int32_t trace_elem, int64_t interval, double* trace, hipEvent_t t0,
               hipEvent_t t1) {
  if (e->cable_groups == 0) return false;
  const int G = e->cable_groups;
  unsigned long long limit = 1ull << 28;
  const char* sl = getenv("NRT_SPIN_LIMIT");
  if (sl) limit = strtoull(sl, nullptr, 10);
  const auto share = device_share(hnd->device, G > 1 ? G : 0);
  const auto until = std::chrono::steady_clock::now() + std::chrono::seconds(sl ? 1 : 180);
  for (int attempt = 0;; attempt++) {
    CabArgs q{e->N, G, e->V[e->cur].p, e->V[1 - e->cur].p, e->coefA.p, e->rdx.p, e->wdx.p,
              e->kdx.p, e->code.p, e->recs.p, e->hd(), e->m2.p, e->h2.p, e->n2.p, e->dt_ms,
              (long long)first, (long long)num, (long long)a0, (long long)a1,
              (long long)interval, trace_elem, trace, e->ll.p, e->err.p, e->tag,
              std::min(limit, 20000ull), limit};
    e->tag += (unsigned)(num / kCabHalo + 2);
    NRT_HIP(hipEventRecord(t0, hnd->stream));
    hipLaunchKernelGGL(k_explicit_cable, dim3(G), dim3(kCabBlock), 0, hnd->stream, q);
    NRT_HIP(hipGetLastError());
    NRT_HIP(hipEventRecord(t1, hnd->stream));
    unsigned err = 0;
    if (G > 1) {
      NRT_HIP(hipMemcpyAsync(&err, e->err.p, sizeof(unsigned), hipMemcpyDeviceToHost, hnd->stream));
      NRT_HIP(hipStreamSynchronize(hnd->stream));
    }
    if (!err) break;
    // workgroups that did not all start in time (another process holds part of the
    // device): nothing was stored, the run is tried again
    NRT_HIP(hipMemsetAsync(e->err.p, 0, sizeof(unsigned), hnd->stream));
    NRT_REQUIRE(std::chrono::steady_clock::now() < until, NRT_ERR_HIP,
                "exchange timed out inside the cable kernel (its workgroups were not all "
                "resident at once: another launch held part of the device)");
    std::this_thread::sleep_for(std::chrono::microseconds(
        100 * std::min(attempt + 1, 50) + (int)((uint32_t)((uintptr_t)e >> 6) * 2654435761u >> 22)));
  }
  e->cur = 1 - e->cur;
  std::swap(e->m.p, e->m2.p);
  std::swap(e->h.p, e->h2.p);
  std::swap(e->n.p, e->n2.p);
  return true;
}

}  // namespace nrt
