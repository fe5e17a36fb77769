// State of an explicit solver, shared by its kernels (explicit.hip: a step per launch,
// small neurites in one workgroup, batches; explicit_cable.hip: unbranched neurites).
#pragma once
#include <functional>
#include <future>
#include "explicit_tree.hpp"
#include "nrt_device.hpp"
#include "nrt_internal.hpp"

namespace nrt {

// Element kinds of the explicit step (code >> 29; the low 29 bits are an index):
// the flag bits kCodeHH, kCodeRec, kCodeSkip alone or HH with Skip keep their
// meaning (chain element, HH chain element with its HH index, exception record,
// terminal/ghost); the three unused combinations carry an element with one
// exception and no record: a daughter (index = its mother), a branch point (index =
// its left daughter), a source of the sealed end right after it (no index).
constexpr uint32_t kExPlain = 0, kExSkip = 1, kExRecord = 2, kExBranch = 3, kExHH = 4,
                   kExSkipHH = 5, kExDaughter = 6, kExCopyNext = 7;

struct HHDev {
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
  const double* dx;
};

struct Explicit {
  int N = 0, H = 0, R = 0;
  double dT = 0, dt_ms = 0;
  DBuf<double> V[2];
  DBuf<double> coefA, rdx, wdx, kdx;
  DBuf<uint32_t> code;
  DBuf<ExRec> recs;
  DBuf<double> m, h, n, E_Na, E_K, E_L, g_Na, g_K, G_L, ls_Na, ls_K, rest, hdx;
  DBuf<double> trace;
  int cur = 0;  // buffer holding the latest potential (the reference's prevT)
  int64_t trace_cap = 0;
  bool res_attr = false;  // the resident kernel's LDS limit is raised
  // unbranched neurites (explicit_cable.hip): workgroups of a run, the second set of
  // gates (m, h, n; a run goes from one set to the other, as V does), what workgroups
  // exchange, and the count of exchanges so far
  int cable_groups = 0;
  DBuf<double> m2, h2, n2;
  DBuf<unsigned long long> ll;
  HostWord err;  // an exchange timed out
  unsigned tag = 0;
  // branching neurites with their elements in registers (explicit_tree.hip); they use
  // the second gates and the exchange of the fields above
  int tree_groups = 0, tree_T = 0, tree_slots = 0, tree_every = 0;
  DBuf<ExUnit> tunit;
  DBuf<ExDynUnit> tdyn;
  HHDev hd() {
    return HHDev{m.p, h.p, n.p, E_Na.p, E_K.p, E_L.p, g_Na.p, g_K.p, G_L.p, ls_Na.p, ls_K.p,
                 rest.p, hdx.p};
  }
};

// Largest neurite whose whole run is one launch (k_explicit_resident: two potentials of
// 8 B, 128 KiB of LDS).
constexpr int kResMaxN = 8192;

// A value that workgroups exchange: two words of 32 data bits, each with the exchange's
// number, so that whoever polls them needs no other flag.
typedef __attribute__((address_space(1))) unsigned long long ExWord;
__device__ __forceinline__ void ex_put(ExWord* w, unsigned tag, double v) {
  const unsigned long long t = (unsigned long long)tag << 32;
  __hip_atomic_store(w, t | (unsigned)__double2loint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(w + 1, t | (unsigned)__double2hiint(v), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// Waits for the NV values of exchange `tag` at w (the first nv of them). Bounded: after
// `most` polls, or once another workgroup gave up, sets *err (a word of host memory) and
// returns false.
template <int NV>
__device__ __forceinline__ bool ex_get(const ExWord* w, unsigned tag, int nv,
                                       unsigned long long most, unsigned* err, double (&v)[NV]) {
  // The last word alone is polled until it is there, then all are read, until all are:
  // polls of every word by hundreds of workgroups fill the fabric between the XCDs.
  unsigned long long x[2 * NV], spins = 0;
  const ExWord* last = w + 2 * nv - 1;
  bool ok = true;
  const auto give_up = [&] {
    if (++spins > most ||
        ((spins & 255) == 0 &&
         __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0u)) {
      __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      ok = false;
    }
    return !ok;
  };
  while ((unsigned)(__hip_atomic_load(last, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 32) !=
         tag)
    if (give_up()) break;
  while (ok) {
    bool all = true;
#pragma unroll
    for (int e = 0; e < 2 * NV; e++)
      if (e < 2 * nv) {
        x[e] = __hip_atomic_load(w + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        all = all && (unsigned)(x[e] >> 32) == tag;
      }
    if (all || give_up()) break;
  }
  if (!ok) return false;
#pragma unroll
  for (int e = 0; e < NV; e++)
    if (e < nv) v[e] = __hiloint2double((int)(unsigned)x[2 * e + 1], (int)(unsigned)x[2 * e]);
  return true;
}

// A batch slot's work in a launch (explicit_tree.hip): steps done before it and taken by it,
// the set that holds potentials and gates before it, exchanges so far.
struct ExTreeWork {
  long long done, steps;
  int cur;
  unsigned tag;
};

// explicit_cable.hip
// A launch whose G workgroups exchange values, until it ends without a time-out:
// launch(polls of the first exchange, of the others).
void run_exchanging(nrt_handle* hnd, Explicit* e, int G,
                    const std::function<void(unsigned long long, unsigned long long)>& launch,
                    hipEvent_t t0, hipEvent_t t1);
void cable_prepare(nrt_handle* hnd, Explicit* e, const HostProblem& p, bool in_batch);
// A run by the cable kernel, waited for; its launches (0: the kernel does not apply).
int64_t cable_run(nrt_handle* hnd, Explicit* e, int64_t first, int64_t num, int64_t a0, int64_t a1,
                  int32_t trace_elem, int64_t interval, double* trace, hipEvent_t t0,
                  hipEvent_t t1);

// explicit_tree.hip
// The plan (G = 0: none), begun; it reads p until it has been got.
using ExPlan = std::future<ExPlanHost>;
ExPlan tree_plan(nrt_handle* hnd, const HostProblem& p, bool in_batch);
void tree_prepare(nrt_handle* hnd, Explicit* e, const HostProblem& p, const ExPlanHost& P);
int64_t tree_run(nrt_handle* hnd, Explicit* e, int64_t first, int64_t num, int64_t a0, int64_t a1,
                 int32_t trace_elem, int64_t interval, double* trace, hipEvent_t t0,
                 hipEvent_t t1);

}  // namespace nrt
