// Explicit steps of branching neurites with few HH elements: every element resident in
// registers for the whole run (records and division of the work: explicit_tree.hpp).
//
// A step of the kernels that go over memory reads 48 B an element and stores 8, and what
// it computes depends on the neighbours of one step only; here an element's potential
// and its five constants stay in its thread's registers, a thread reads three
// neighbours' potentials from LDS (double buffered) and stores its two ends, and a step
// is one barrier. What bounds it: the FP64 operations, about 13 an element and step
// (8 elements a thread; 2 waves a SIMD at kExT units), the barrier, and the exchange
// between groups, a round trip through memory, once in 16 steps. Measured, us a step
// before (small neurites from LDS and L2 in one workgroup, others a launch a step) and
// here: 700 elements 2.3 and 0.6, 3,001 3.8 and 0.65, 30,000 4.2 and 0.7, 300,000 5.7 and
// 0.8, 902,037 10.7 and 1.5; a batch of 512 trees (5.5 M elements) 55 and 8.
//
// Every operation is explicit_element's, operand for operand (an axial term of an element
// and its mother is computed once: it enters the two with opposite signs, which loses
// nothing), so the results are those of the other kernels bit for bit.
#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdlib>
#include <cstring>
#include <system_error>
#include "explicit_dev.hpp"

namespace nrt {

struct ExTreeDev {
  int N, G, T, slots, every;
  const ExUnit* unit;
  const ExDynUnit* dyn;
  double* V[2];
  const double *coefA, *rdx, *wdx, *kdx;
  HHDev hd;
  double *m2, *h2, *n2;  // second set of gates; a run goes from the set of `cur` to the other
  double dt_ms;
  unsigned long long* ll;  // [2][slots][kExSlotVals] words of two
  unsigned* err;
  long long a0, a1, interval;
  int trace_elem;
};

struct ExTreeRun {
  int cur;               // V and gates of the step before `first`
  long long first, num;  // steps first .. first + num - 1
  long long gl0;         // steps since the last sample
  double* trace;         // the next sample
  unsigned tag0;         // exchanges so far
  unsigned long long first_limit, limit;
};

// Most units per group, as long as the groups are at most the CUs: with the HH elements' wave
// four waves, one a SIMD (0.68 us a step for 30,000 elements; with 256 units, two waves on
// one SIMD, 0.97) and three workgroups a CU in a batch (five-wave ones only one: 100 steps
// of 512 trees 1.5 ms, with 192 units 1.05).
constexpr int kExTBatch = 192;
constexpr int kExTBlock = kExT + kWave;

// What the loop over the steps needs of the records stays in scalar registers: a batch's
// records lie in memory, and the compiler would read them again every step.
template <class X>
__device__ __forceinline__ X pinned_s(X x) {
  asm volatile("" : "+s"(x));
  return x;
}
template <class P>
__device__ __forceinline__ __attribute__((address_space(1))) P* as_global(P* p) {
  return (__attribute__((address_space(1))) P*)p;
}

// Eight doubles from an address that is a multiple of 8, two a load.
__device__ __forceinline__ void ex_load8(const __attribute__((address_space(1))) double* p,
                                         double (&x)[kExC]) {
  typedef double D2 __attribute__((ext_vector_type(2), aligned(8)));
  const auto* q = (const __attribute__((address_space(1))) D2*)p;
#pragma unroll
  for (int k = 0; k < kExC / 2; k++) {
    const D2 d = q[k];
    x[2 * k] = d.x;
    x[2 * k + 1] = d.y;
  }
}

__device__ __forceinline__ void ex_tree_steps(const ExTreeDev& d, const ExTreeRun& q, int g) {
  constexpr int C = kExC;
  __shared__ double val[2][kExVals];
  __shared__ int fail;
  const int tid = (int)threadIdx.x, lane = tid & (kWave - 1);
  const int T = pinned_s(d.T), probe_elem = d.trace_elem;
  const auto* Vin = as_global((const double*)d.V[q.cur]);
  auto* Vout = as_global(d.V[1 - q.cur]);
  const auto *coefA = as_global(d.coefA), *rdx = as_global(d.rdx), *wdx = as_global(d.wdx),
             *kdx = as_global(d.kdx);
  auto* trace = as_global(pinned_s(q.trace));
  const long long a0 = pinned_s(d.a0), a1 = pinned_s(d.a1), interval = pinned_s(d.interval);
  const double dt_ms = pinned_s(d.dt_ms);
  if (tid == 0) {
    fail = 0;
    val[0][kExMissing] = val[1][kExMissing] = 0.0;
  }
  const bool service = tid >= T && tid < T + kWave;
  // what an exchange needs, and when
  const int every = pinned_s(d.slots > 0 ? d.every : INT_MAX);
  auto words = [&](unsigned tag, int slot) {
    return as_global(d.ll) + ((size_t)(tag & 1) * d.slots + slot) * kExSlotVals * 2;
  };
  long long gl = q.gl0, ks = 0;
  unsigned tag = q.tag0;
  int p = 0, left = every;
  unsigned long long most = q.first_limit;
  const long long first = pinned_s(q.first), end = pinned_s(first + q.num);
  // a step's sample is due: advances the count
  auto sample = [&]() {
    if (interval < 0 || ++gl <= interval) return false;
    gl = 0;
    return true;
  };
  if (tid < T) {
    // ------------------------------------------------------------ a unit's thread
    const ExUnit u = ((const ExUnit*)d.unit)[(size_t)g * T + tid];
    const bool on = u.flags & kExUOn, halo = u.flags & kExUHalo, ghost = u.flags & kExUGhost;
    const bool branch = u.flags & kExUBranch, term = u.flags & kExUTerm;
    const int f = on ? (int)(u.flags & 7) : C;  // unused places
    const int ik = u.flags & kExUInput ? (int)(u.flags >> 8 & 7) : -1;
    double V[C], a[C], r[C], y[C], w[C], kd[C];
    // (an unused place reads what lies before the unit, or, at the arrays' beginning, the
    // unit's first element: no load waits for another)
    const int at = u.first - f;
    if (on && at >= 0) {
      ex_load8(Vin + at, V);
      ex_load8(coefA + at, a);
      ex_load8(rdx + at, r);
      ex_load8(wdx + at, w);
      ex_load8(kdx + at, kd);
    } else {
#pragma unroll
      for (int k = 0; k < C; k++) {
        const int j = k >= f ? at + k : u.first;
        V[k] = Vin[j];
        a[k] = coefA[j];
        r[k] = rdx[j];
        w[k] = wdx[j];
        kd[k] = kdx[j];
      }
    }
#pragma unroll
    for (int k = 0; k < C; k++) {
      const bool used = k >= f;
      V[k] = used ? V[k] : 0.0;
      a[k] = used ? a[k] : 0.0;
      r[k] = used ? r[k] : 1.0;
      w[k] = used ? w[k] : 0.0;
      kd[k] = used ? kd[k] : 0.0;
      y[k] = 1 / r[k];
    }
    const double rR = on ? rdx[u.el_right] : 1.0, rL = on ? rdx[u.el_left] : 1.0;
    const double yR = 1 / rR, yL = 1 / rL;
    double v0 = ghost ? Vin[0] : 0.0;
    const int up = on ? u.up : kExMissing, right = on && !term ? u.right : kExMissing;
    const int lft = on && branch ? u.left : kExMissing;
    const bool some_pads = __any(f > 0), some_ghost = __any(ghost), some_branch = __any(branch);
    const bool some_term = __any(term), some_input = __any(ik >= 0);
    // place of the probed element (C: the copied first element)
    int tk = -1;
    if (on && !halo && trace) {
      const int k = probe_elem - u.first + f;
      if (probe_elem > 0 && k >= f && k < C) tk = k;
      if (probe_elem == 0 && ghost) tk = C;
    }
    auto head = [&]() {
      double x = V[0];
      if (some_pads) {
#pragma unroll
        for (int k = 1; k < C; k++) x = f == k ? V[k] : x;
      }
      return x;
    };
    auto publish = [&]() {
      val[p][tid] = head();
      val[p][kExT + tid] = V[C - 1];
    };
    publish();
    lds_sync();
    for (long long i = first; i < end; i++) {
      if (left == 0) {
        left = every;
        tag++;
        const bool has = on && u.slot >= 0;
        auto* o = words(tag, has ? u.slot : 0);
        if (has && !halo) {
#pragma unroll
          for (int k = 0; k < C; k++) ex_put(o + 2 * k, tag, V[k]);
        }
        __builtin_amdgcn_wave_barrier();  // a wave's lanes all put before any waits
        if (has && halo) {
          if (!ex_get<C>(o, tag, C, most, d.err, V)) fail = 1;
          publish();
          if (ghost) v0 = head();  // (its copy, since a step has been taken)
        }
        most = q.limit;
        lds_sync();
        if (fail) return;  // uniform: read after the barrier
      }
      left--;
      const double vu = some_ghost && ghost ? v0 : val[p][up];
      const double vr = val[p][right];
      double vl = 0;
      if (some_branch) vl = val[p][lft];
      if (some_pads) {
#pragma unroll
        for (int k = 0; k < C - 1; k++) V[k] = k < f ? vu : V[k];
      }
      const bool stim = some_input && i >= a0 && i <= a1;
      double t = div_by(V[0] - vu, r[0], y[0]);
#pragma unroll
      for (int k = 0; k < C; k++) {
        double tn, s;
        if (k < C - 1) {
          tn = div_by(V[k + 1] - V[k], r[k + 1], y[k + 1]);
          s = tn;
        } else {
          tn = div_by(vr - V[k], rR, yR);
          s = tn;
          if (some_branch) {
            const double tl = div_by(vl - V[k], rL, yL);
            s = branch ? tl + tn : tn;
          }
        }
        s = s - t;
        s = s + w[k] * V[k];
        s = s + kd[k];
        if (stim) s = ik == k ? s + u.input : s;
        V[k] = V[k] + a[k] * s;
        t = tn;
      }
      if (some_term) V[C - 1] = term ? V[C - 2] : V[C - 1];
      p ^= 1;
      const double hd = head();
      if (some_ghost) v0 = hd;
      val[p][tid] = hd;
      val[p][kExT + tid] = V[C - 1];
      if (sample()) {
        if (tk >= 0) {
          double x = tk == C ? v0 : V[0];
#pragma unroll
          for (int k = 1; k < C; k++) x = tk == k ? V[k] : x;
          trace[ks] = x;
        }
        ks++;
      }
      lds_sync();
    }
    if (on && !halo) {
      if (f == 0) {
        typedef double D2 __attribute__((ext_vector_type(2), aligned(8)));
        auto* o = (__attribute__((address_space(1))) D2*)(Vout + u.first);
#pragma unroll
        for (int k = 0; k < C / 2; k++) o[k] = (D2){V[2 * k], V[2 * k + 1]};
      } else {
#pragma unroll
        for (int k = 1; k < C; k++)
          if (k >= f) Vout[u.first + k - f] = V[k];
      }
      if (ghost) Vout[0] = v0;
    }
  } else if (service) {
    // ------------------------------------------------------------ HH elements
    // Eight lanes each: lanes 0..5 a rate (am, bm, ah, bh, an, bn), lanes 0, 2, 4 a gate.
    const ExDynUnit u = d.dyn[(size_t)g * kExDyn + (lane >> 3)];
    const int e = lane & 7, at = 2 * kExT + (lane >> 3), base = lane & ~7;
    const bool on = u.elem >= 0, halo = u.flags & kExUHalo, ghost = u.flags & kExUGhost;
    const bool branch = u.flags & kExUBranch, input = u.flags & kExUInput;
    const int j = on ? u.elem : 0, hh = on ? u.hh : 0;
    double v = 0, v0 = 0, m = 0, h = 0, n = 0, rest = 0, ls = 0, gNa = 0, gK = 0, gL = 0, eNa = 0,
           eK = 0, eL = 0, dx = 0, a = 0, rj = 1, rR = 1, rL = 1;
    if (on) {
      v = Vin[j];
      if (ghost) v0 = Vin[0];
      m = (q.cur ? d.m2 : d.hd.m)[hh];
      h = (q.cur ? d.h2 : d.hd.h)[hh];
      n = (q.cur ? d.n2 : d.hd.n)[hh];
      rest = d.hd.rest[hh];
      ls = (e < 4 ? d.hd.ls_Na : d.hd.ls_K)[hh];
      gNa = d.hd.g_Na[hh];
      gK = d.hd.g_K[hh];
      gL = d.hd.G_L[hh];
      eNa = d.hd.E_Na[hh];
      eK = d.hd.E_K[hh];
      eL = d.hd.E_L[hh];
      dx = d.hd.dx[hh];
      a = coefA[j];
      rj = rdx[j];
      rR = rdx[u.el_right];
      rL = rdx[u.el_left];
    }
    const double yj = 1 / rj, yR = 1 / rR, yL = 1 / rL;
    // exp(c0 - 0.1 u) or exp(-u / c1); a rate is num / (exp +- 1) or c2 exp
    const bool quot = e == 0 || e == 3 || e == 4;
    const double c0 = e == 0 ? 2.5 : (e == 3 ? 3.0 : 1.0);
    const double c1 = e == 1 ? 18.0 : (e == 2 ? 20.0 : 80.0);
    const double y1 = e == 1 ? 1.0 / 18.0 : (e == 2 ? 1.0 / 20.0 : 1.0 / 80.0);
    const double c2 = e == 1 ? 4.0 : (e == 2 ? 0.07 : 0.125);
    const double one = e == 3 ? 1.0 : -1.0;
    double gate = e < 2 ? m : (e < 4 ? h : n);
    const bool probe = on && !halo && e == 0 && trace &&
                       (probe_elem == j || (probe_elem == 0 && ghost));
    if (e == 0) val[p][at] = v;
    lds_sync();
    for (long long i = first; i < end; i++) {
      if (left == 0) {
        left = every;
        tag++;
        const bool has = on && u.slot >= 0;
        auto* o = words(tag, has ? u.slot : 0);
        if (has && !halo && e == 0) {
          ex_put(o, tag, v);
          ex_put(o + 2, tag, m);
          ex_put(o + 4, tag, h);
          ex_put(o + 6, tag, n);
        }
        __builtin_amdgcn_wave_barrier();
        if (has && halo) {
          double x[4] = {};
          if (!ex_get<4>(o, tag, 4, most, d.err, x)) fail = 1;
          v = x[0];
          if (ghost) v0 = v;
          gate = e < 2 ? x[1] : (e < 4 ? x[2] : x[3]);
          if (e == 0) val[p][at] = v;
        }
        most = q.limit;
        lds_sync();
        if (fail) return;
      }
      left--;
      if (on) {
        const double un = div_by((v + ls) - rest, 0.001, 1000.0);
        const double lin = c0 - 0.1 * un;
        const double x = exp(quot ? lin : div_by(-un, c1, y1));
        const double num = e == 0 ? lin : (e == 3 ? 1.0 : 0.1 - 0.01 * un);
        const double quo = num / (x + one);
        const double rate = quot ? quo : c2 * x;
        const double other = __shfl(rate, lane ^ 1);
        gate = gate + dt_ms * (rate * (1 - gate) - other * gate);
        m = __shfl(gate, base);
        h = __shfl(gate, base + 2);
        n = __shfl(gate, base + 4);
        const double gna = gNa * m * m * m * h;
        const double gk = gK * n * n * n * n;
        const double W = -(gna + gk + gL);
        const double K = gna * eNa + gk * eK + gL * eL;
        const double wd = W * dx, kd = K * dx;
        const double vm = ghost ? v0 : val[p][u.up];
        double s = div_by(val[p][u.right] - v, rR, yR);
        if (branch) s = div_by(val[p][u.left] - v, rL, yL) + s;
        s = s + div_by(vm - v, rj, yj);
        s = s + wd * v;
        s = s + kd;
        if (input && i >= a0 && i <= a1) s = s + u.input;
        v = v + a * s;
        if (ghost) v0 = v;
        if (e == 0) val[p ^ 1][at] = v;
      }
      p ^= 1;
      if (sample()) {
        if (probe) trace[ks] = v;
        ks++;
      }
      lds_sync();
    }
    if (on && !halo && e == 0) {
      Vout[j] = v;
      if (ghost) Vout[0] = v0;
      (q.cur ? d.hd.m : d.m2)[hh] = m;
      (q.cur ? d.hd.h : d.h2)[hh] = h;
      (q.cur ? d.hd.n : d.n2)[hh] = n;
    }
  }
}

__global__ __launch_bounds__(kExTBlock) void k_explicit_tree(ExTreeDev d, ExTreeRun q) {
  ex_tree_steps(d, q, (int)blockIdx.x);
}

// Slots of a batch: workgroup w of the launch order runs map[w] = (slot, group) for the
// slot's work[].steps steps; a workgroup takes its place in that order when it starts
// (see k_resident_batch).
struct ExTreeRec {
  ExTreeDev d;
  double* trace_base;
};
__global__ __launch_bounds__(kExTBatch + kWave) void k_explicit_tree_batch(
    const ExTreeRec* __restrict__ recs, const ExTreeWork* __restrict__ work,
    const int2* __restrict__ map, unsigned* __restrict__ ticket, unsigned long long limit) {
  __shared__ unsigned mine;
  if (threadIdx.x == 0) mine = atomicAdd(ticket, 1u);
  __syncthreads();
  const int2 m = map[__builtin_amdgcn_readfirstlane(mine)];
  const ExTreeRec& rec = recs[m.x];
  const ExTreeWork wk = work[m.x];
  ExTreeRun q{wk.cur, wk.done + 1, wk.steps, 0, nullptr, wk.tag, limit, limit};
  if (rec.d.interval >= 0) {
    q.gl0 = wk.done % (rec.d.interval + 1);
    if (rec.trace_base) q.trace = rec.trace_base + wk.done / (rec.d.interval + 1);
  }
  ex_tree_steps(rec.d, q, m.y);
}

// ---------------------------------------------------------------- host side
namespace {
constexpr int kExTLarge = 448;

// Groups that are sure to be resident at once: one a CU. (Where the registers allow two
// of 256 unit threads, 477 of 512 did not all start.)
int tree_capacity(int device, int T) {
  static std::atomic<int> known{0};  // (device + 1) << 16 | CUs: asked for every slot of a batch
  const int k = known.load(std::memory_order_relaxed);
  if (k >> 16 == device + 1) return k & 0xFFFF;
  int cus = 0, per = 0;
  NRT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  NRT_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_explicit_tree,
                                                       T + kWave, 0));
  if (per == 0) cus = 0;
  known.store((device + 1) << 16 | cus, std::memory_order_relaxed);
  return cus;
}
}  // namespace

// Device memory of the plan beyond what a batch's admission reckons with per element is
// only taken while this much stays free for other slots.
constexpr int64_t kExPlanBytesPerElem = 12;
constexpr int64_t kExPlanReserve = 512ll << 20;
constexpr int kExPlanAlone = 16384;  // elements

static bool tree_room(int device, const ExPlanHost& P) {
  const int64_t bytes = (int64_t)(P.unit.size() * sizeof(ExUnit) + P.dyn.size() * sizeof(ExDynUnit)) +
                        (int64_t)P.slots * 2 * kExSlotVals * 2 * 8;
  if (bytes <= kExPlanBytesPerElem * P.N) return true;
  size_t free_b = 0, total_b = 0;
  NRT_HIP(hipMemGetInfo(&free_b, &total_b));
  return (int64_t)free_b + pool_cached_bytes(device) >= bytes + kExPlanReserve;
}

// The plan, of a large neurite on a thread of its own beside the rest of the creation: a
// handle that is only stepped has no use for it. Creation in ms without a plan, with it made
// in line, and so: 902,037 elements 19.1, 26.9, 20.0; 200,000 2.0, 3.4, 2.2; 30,000 0.39,
// 0.54, 0.46; 17,000 0.29, 0.37, 0.34 (below kExPlanAlone in line: the thread costs as much).
ExPlan tree_plan(nrt_handle* hnd, const HostProblem& p, bool in_batch) {
  // (a run of an unbranched neurite is the cable kernel's or specified as a launch a step;
  // one or two steps are no run of this form)
  const int cap = tree_capacity(hnd->device, kExT);
  const auto make = [&p, in_batch, cap] {
    ExPlanHost P;
    bool branching = in_batch, fits = false;
    for (int j = 1; j < p.N - 1 && !branching; j++) branching = p.branching[j] != 0;
    std::string why;
    const auto plan = [&](int T, int most) {
      // (strands of some 50 elements and halos: 4 to 6% more units than N / kExC)
      if (!branching || p.N / kExC * 1.03 > (double)most * T) return;
      for (int every : {kExEvery, kExEveryDense})
        if (!fits && build_explicit_plan(p, T, every, P, why)) fits = P.G <= most;
    };
    // (larger groups where there are not CUs enough: seven or eight waves of units)
    plan(kExTBatch, cap);
    if (!in_batch && !fits) plan(kExTLarge, cap);
    if (!in_batch && !fits) plan(kExT, cap);
    if (!fits) P = ExPlanHost();
    return P;
  };
  if (p.N >= kExPlanAlone) {
    try {
      return std::async(std::launch::async, make);
    } catch (const std::system_error&) {  // (no thread to be had)
    }
  }
  return std::async(std::launch::deferred, make);
}

// The plan's device state; leaves the solver without the form where the plan refuses or the
// memory is not there. (P: uploaded from until the stream is waited for)
void tree_prepare(nrt_handle* hnd, Explicit* e, const HostProblem& p, const ExPlanHost& P) {
  if (P.G == 0 || !tree_room(hnd->device, P)) return;
  try {
    e->tunit.upload(P.unit, hnd->stream);
    e->tdyn.upload(P.dyn, hnd->stream);
    e->m2.alloc(p.H);
    e->h2.alloc(p.H);
    e->n2.alloc(p.H);
    if (P.slots > 0) e->ll.alloc((size_t)2 * P.slots * kExSlotVals * 2);
  } catch (const Error& err) {
    if (err.status != NRT_ERR_NOMEM) throw;
    NRT_HIP(hipStreamSynchronize(hnd->stream));
    e->tunit.release();
    e->tdyn.release();
    for (DBuf<double>* b : {&e->m2, &e->h2, &e->n2}) b->release();
    return;
  }
  e->err.take();
  if (P.slots > 0)
    NRT_HIP(hipMemsetAsync(e->ll.p, 0, sizeof(unsigned long long) * e->ll.n, hnd->stream));
  e->tree_groups = P.G;
  e->tree_T = P.T;
  e->tree_slots = P.slots;
  e->tree_every = P.every;
}

static ExTreeDev tree_dev(Explicit* e, int from, unsigned* err, long long a0, long long a1,
                          long long interval, int trace_elem) {
  return {e->N, e->tree_groups, e->tree_T, e->tree_slots, e->tree_every, e->tunit.p, e->tdyn.p,
          {e->V[from].p, e->V[1 - from].p}, e->coefA.p, e->rdx.p, e->wdx.p, e->kdx.p, e->hd(),
          e->m2.p, e->h2.p, e->n2.p, e->dt_ms, e->ll.p, err, a0, a1, interval, trace_elem};
}

int64_t tree_run(nrt_handle* hnd, Explicit* e, int64_t first, int64_t num, int64_t a0, int64_t a1,
                 int32_t trace_elem, int64_t interval, double* trace, hipEvent_t t0,
                 hipEvent_t t1) {
  // One or two steps, and three of a short neurite, are done without the registers, as fast as
  // these are filled and emptied (run of 1 / 2 / 3 / 4 steps there and here, us, with the
  // launch and the wait: 300 elements 18 / 21 / 23 / 25 and 23 / 24 / 24 / 25; 2,000
  // 20 / 23 / 26 / 29 and 24 / 25 / 26 / 26; 30,000 18 / 22 / 27 / 30 and 24 / 24 / 25 / 25;
  // 902,037 23 / 33 / 43 / 53 and 30 / 32 / 33 / 33).
  if (e->tree_groups == 0 || num <= (e->N <= 1500 ? 3 : 2)) return 0;
  // (pieces: see run_persistent in implicit.hip; 8,192 steps of 902,037 elements 12 ms)
  constexpr int64_t kShareSteps = 8192;
  constexpr int kShareCus = 64;
  const int64_t most = e->tree_groups > kShareCus ? kShareSteps : num;
  const int64_t per = interval >= 0 ? interval + 1 : 1;
  int64_t done = 0, launches = 0;
  for (; done < num; launches++) {
    const int64_t n = std::min(most, num - done);
    try {
      run_exchanging(
          hnd, e, e->tree_groups,
          [&](unsigned long long first_limit, unsigned long long limit) {
            const ExTreeDev d = tree_dev(e, e->cur, e->err.p, a0, a1, interval, trace_elem);
            ExTreeRun q{0, (long long)(first + done), (long long)n, done % per,
                        trace ? trace + done / per : nullptr, e->tag, first_limit, limit};
            e->tag += (unsigned)(n / e->tree_every + 2);
            hipLaunchKernelGGL(k_explicit_tree, dim3(e->tree_groups), dim3(e->tree_T + kWave), 0,
                               hnd->stream, d, q);
          },
          done == 0 ? t0 : nullptr, t1);
    } catch (...) {
      hnd->stats.steps += done;  // (as the statistics of the implicit forms count them)
      throw;
    }
    done += n;
  }
  return launches;
}

// ---- slots of a batch (batch.cpp): their gates stay where they are and the work names
// the current set, as it names the current potentials
bool explicit_tree_slot(const nrt_handle* h) { return h->ex && h->ex->tree_groups > 0; }
size_t explicit_tree_rec_bytes() { return sizeof(ExTreeRec); }
size_t explicit_tree_work_bytes() { return sizeof(ExTreeWork); }
void explicit_tree_shape(nrt_handle* h, int* groups, int* T) {
  *groups = h->ex->tree_groups;
  *T = h->ex->tree_T;
}
void explicit_tree_fill(nrt_handle* h, unsigned* err, long long a0, long long a1, int trace_elem,
                        long long interval, double* trace, void* out) {
  const ExTreeRec r{tree_dev(h->ex, 0, err, a0, a1, interval, trace_elem), trace};
  memcpy(out, &r, sizeof(r));
}
// The work of a launch; the slot's current potentials are what it will have made.
void explicit_tree_work(nrt_handle* h, long long done, long long steps, void* out) {
  Explicit* e = h->ex;
  const ExTreeWork w{done, steps, e->cur, e->tag};
  memcpy(out, &w, sizeof(w));
  if (steps <= 0) return;
  e->tag += (unsigned)(steps / e->tree_every + 2);
  e->cur = 1 - e->cur;
}
// A launch that timed out: the potentials before it are the current ones again.
void explicit_tree_undo(nrt_handle* h, const void* work, long long* done, long long* steps) {
  ExTreeWork w;
  memcpy(&w, work, sizeof(w));
  h->ex->cur = w.cur;
  *done = w.done;
  *steps = w.steps;
}
void explicit_tree_batch_launch(const void* recs, const void* work, const int2* map,
                                unsigned* ticket, int nwg, int T, hipStream_t s) {
  const char* sl = getenv("NRT_SPIN_LIMIT");
  hipLaunchKernelGGL(k_explicit_tree_batch, dim3(nwg), dim3(T + kWave), 0, s,
                     (const ExTreeRec*)recs, (const ExTreeWork*)work, map, ticket,
                     sl ? strtoull(sl, nullptr, 10) : 1ull << 28);
  NRT_HIP(hipGetLastError());
}

}  // namespace nrt
