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
      ExWord* ll =
          (ExWord*)q.ll + (size_t)(tag & 1) * q.G * 2 * kCabHalo * kCabState * 2;
      auto at = [&](int gg, int side, int kk) {
        return ll + ((((size_t)gg * 2 + side) * kCabHalo + kk) * kCabState) * 2;
      };
      if (put_l) {
        ExWord* o = at(g, 0, t - halo);
        ex_put(o, tag, v);
        if (hh >= 0) {
          ex_put(o + 2, tag, m);
          ex_put(o + 4, tag, h);
          ex_put(o + 6, tag, n);
        }
      }
      if (put_r) {
        ExWord* o = at(g, 1, t - (kCabBlock - 2 * halo));
        ex_put(o, tag, v);
        if (hh >= 0) {
          ex_put(o + 2, tag, m);
          ex_put(o + 4, tag, h);
          ex_put(o + 6, tag, n);
        }
      }
      __builtin_amdgcn_wave_barrier();  // a wave's lanes all put before any waits
      if (get) {
        const ExWord* o = at(src_g, src_side, src_k);
        double x[kCabState] = {};
        if (!ex_get(o, tag, hh >= 0 ? kCabState : 1, first_ex ? q.first_limit : q.limit, q.err, x))
          fail = 1;
        v = x[0];
        if (hh >= 0) {
          m = x[1];
          h = x[2];
          n = x[3];
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
  e->err.take();
  if (G > 1) {
    e->ll.alloc((size_t)2 * G * 2 * kCabHalo * kCabState * 2);
    NRT_HIP(hipMemsetAsync(e->ll.p, 0, sizeof(unsigned long long) * e->ll.n, hnd->stream));
  }
}

void run_exchanging(nrt_handle* hnd, Explicit* e, int G,
                    const std::function<void(unsigned long long, unsigned long long)>& launch,
                    hipEvent_t t0, hipEvent_t t1) {
  unsigned long long limit = 1ull << 28;
  const char* sl = getenv("NRT_SPIN_LIMIT");
  if (sl) limit = strtoull(sl, nullptr, 10);
  const auto share = device_share(hnd->device, G > 1 ? G : 0);
  const auto until = std::chrono::steady_clock::now() + std::chrono::seconds(sl ? 1 : 180);
  for (int attempt = 0;; attempt++) {
    if (t0) NRT_HIP(hipEventRecord(t0, hnd->stream));
    launch(std::min(limit, 20000ull), limit);
    NRT_HIP(hipGetLastError());
    NRT_HIP(hipEventRecord(t1, hnd->stream));
    if (G == 1) break;
    NRT_HIP(hipStreamSynchronize(hnd->stream));
    if (!e->err.get()) break;
    // workgroups that did not all start in time (another process holds part of the
    // device): nothing that counts was stored, the run is tried again
    e->err.clear();
    NRT_REQUIRE(std::chrono::steady_clock::now() < until, NRT_ERR_HIP,
                "exchange timed out inside an explicit kernel (its workgroups were not all "
                "resident at once: another launch held part of the device)");
    std::this_thread::sleep_for(std::chrono::microseconds(
        100 * std::min(attempt + 1, 50) + (int)((uint32_t)((uintptr_t)e >> 6) * 2654435761u >> 22)));
  }
  // the run's results become the current ones
  e->cur = 1 - e->cur;
  std::swap(e->m.p, e->m2.p);
  std::swap(e->h.p, e->h2.p);
  std::swap(e->n.p, e->n2.p);
}

int64_t cable_run(nrt_handle* hnd, Explicit* e, int64_t first, int64_t num, int64_t a0, int64_t a1,
                  int32_t trace_elem, int64_t interval, double* trace, hipEvent_t t0,
                  hipEvent_t t1) {
  // One step of a short neurite, or two of a very short one, are done by one workgroup
  // before this launch has set up its registers (runs of 1 / 2 / 4 steps there and here, us,
  // with the launch and the wait: 402 elements 19 / 22 / 30 and 24 / 24 / 26, 1,002
  // 21 / 26 / 36 and 24 / 25 / 27, 5,000 35 / 53 / 89 and 25 / 25 / 27).
  if (e->cable_groups == 0 || (num <= 2 && num * e->N <= 2048)) return 0;
  const int G = e->cable_groups;
  run_exchanging(
      hnd, e, G,
      [&](unsigned long long first_limit, unsigned long long limit) {
        CabArgs q{e->N, G, e->V[e->cur].p, e->V[1 - e->cur].p, e->coefA.p, e->rdx.p, e->wdx.p,
                  e->kdx.p, e->code.p, e->recs.p, e->hd(), e->m2.p, e->h2.p, e->n2.p, e->dt_ms,
                  (long long)first, (long long)num, (long long)a0, (long long)a1,
                  (long long)interval, trace_elem, trace, e->ll.p, e->err.p, e->tag,
                  first_limit, limit};
        e->tag += (unsigned)(num / kCabHalo + 2);
        hipLaunchKernelGGL(k_explicit_cable, dim3(G), dim3(kCabBlock), 0, hnd->stream, q);
      },
      t0, t1);
  return 1;
}

}  // namespace nrt
