// Device view of an unbranched neurite whose rows stay in registers (chain.hip).
#pragma once
#include "resident_dev.hpp"

namespace nrt {

constexpr int kChWaves = 64;   // most waves (a lane of the top each)
constexpr int kChGates = 64;   // most gating rows per wave

struct ChainDev {
  int N, W, C, H;  // rows, waves, rows per lane, gating rows
  const double *sub, *dg, *sup;  // the matrix (dg of gating rows changes)
  const double *cdt, *kd;        // c_m dx / dT, K dx
  const double* inp;             // stimulus (null: none)
  const int32_t *woff, *hrow, *hidx;  // a wave's gating rows: range, rows, HH entries
  const double* x;               // V, then m, h, n of the gating rows in their order; a
  double* xo;                    // launch goes from x to xo
  unsigned long long* ll;        // [2][W][7] words of two
};

void chain_launch(const ImpDev& d, const ChainDev& r, const ResRun& q, hipStream_t s);

}  // namespace nrt
