// State of an explicit solver, shared by its kernels (explicit.hip: a step per launch,
// small neurites in one workgroup, batches; explicit_cable.hip: unbranched neurites).
#pragma once
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
  DBuf<unsigned> err;
  unsigned tag = 0;
  HHDev hd() {
    return HHDev{m.p, h.p, n.p, E_Na.p, E_K.p, E_L.p, g_Na.p, g_K.p, G_L.p, ls_Na.p, ls_K.p,
                 rest.p, hdx.p};
  }
};

// Largest neurite whose whole run is one launch (k_explicit_resident: two potentials of
// 8 B, 128 KiB of LDS).
constexpr int kResMaxN = 8192;

// explicit_cable.hip
void cable_prepare(nrt_handle* hnd, Explicit* e, const HostProblem& p, bool in_batch);
// A run by the cable kernel, waited for; false where it does not apply.
bool cable_run(nrt_handle* hnd, Explicit* e, int64_t first, int64_t num, int64_t a0, int64_t a1,
               int32_t trace_elem, int64_t interval, double* trace, hipEvent_t t0, hipEvent_t t1);

}  // namespace nrt
