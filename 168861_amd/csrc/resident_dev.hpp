// Device view of a resident tree solve (resident.hpp), one per neurite.
#pragma once
#include "implicit_dev.hpp"
#include "resident.hpp"

namespace nrt {

// Diagonal of the HH row q for the membrane term W (hh_row_refresh without the row's
// values in memory).
__device__ __forceinline__ double hh_row_diag(const HHRow& q, double W) {
  const double betaMe = -(W * q.dxv) + q.inv_rdx;
  const double beta = q.c_dt + betaMe + q.betaR;
  switch (q.type) {
    case RT_NEXT_TERM: return beta + -q.betaR;
    case RT_BRANCH: return beta + q.betaL;
    case RT_FIRST_NORMAL: return q.alpha + beta;
    case RT_FIRST_BRANCH: return q.alpha + beta + q.betaL;
    default: return beta;
  }
}

struct ResDev {
  int G, T, nd, nt, npub, nth, top_narrow, rounds, owner, has_input;
  // rows, slot order
  const double* cdt;   // c_m dx / dT
  const double* kd;    // K dx
  const double* inp;   // stimulus (has_input)
  const double* F;
  const double* I;
  const double* x;     // state of the step before a launch: rows, then the dynamic rows'
  double* xo;          // V, m, h, n; and after it (a handle's launches go from one buffer
                       // to the other, so one that gave up leaves the state as it was)
  // units, pieces, groups
  const double* uco;
  const uint32_t* uinf;
  const double* pz;
  const uint16_t* pinf;
  const int32_t* ginfo;
  // top
  const double* tz;
  const double* te;
  const uint16_t* tinf;
  const int32_t* thoff;
  // dynamic rows: element, static diagonal (not HH), static children's share, coupling
  // to the parent, refs; HH entry (-1: none)
  const int32_t* drow;
  const int32_t* dhh;
  const double* ddiag;
  const double* ds;
  const double* du;
  const uint16_t* dinf;
  const uint16_t* epiece;
  // published values: two sets used in turn, two 64-bit words each (half a double and
  // the step's tag)
  unsigned long long* ll;
};

// One launch of a neurite: its steps, and the tag of the step before them.
struct ResRun {
  long long first, num, gl0;
  unsigned tag0;
  double* trace;
  unsigned long long first_limit;  // polls of the first exchange (all workgroups are
                                   // resident once it is over)
};

// A slot of a batch: its device view, and per launch the steps it has done and takes.
struct ResWork {
  long long done, steps;
};
struct ResRec {
  ImpDev d;
  ResDev r;
  double* trace_base;
};

}  // namespace nrt
