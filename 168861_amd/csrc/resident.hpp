// Tree solve with the rows resident in registers ("resident form"), for trees whose
// matrix changes in a few rows only (a Hodgkin-Huxley soma on passive dendrites).
//
// Gaussian elimination from the leaves to the root (Hines) of the static rows always
// gives the same pivots, so they are computed once, on the host, and a step is two
// linear recurrences over the tree with constant coefficients:
//   up:    r'_p = r_p + sum_c F_c r'_c        F_c = -A[p][c] / d'_c
//   down:  x_i  = I_i r'_i + F_i x_parent     I_i = 1 / d'_i   (A[p][c] = A[c][p])
// Rows whose pivot changes (an HH row and the rows above it, "dynamic" rows) form the
// root part; they are eliminated every step.
//
// Decomposition (static rows):
//   unit    kResC consecutive rows of a chain (a run of rows each of which is the only
//           child of the row before it), held by one thread; short units are padded
//           with rows that pass values through (r = 0, I = 0, F = 1)
//   piece   consecutive units of a chain in the lanes of one wave; a scan over lanes
//           with constant coefficients combines them
//   group   the units of one workgroup (T of them); its pieces form a forest that is
//           swept by heights, at each piece the affine map
//             o = a + Z in,  x_bottom = q + Z x_above
//           (in: the sum of its children's o, entering at its bottom row)
//   strand  a chain's part in one group. A strand with a descendant in another group
//           is a node of the "top": what a group computes alone is provisional and is
//           corrected by the two numbers that its strand lacked, the input d_in from
//           other groups at its bottom and the value d_x above its head:
//             d_o = Z d_in,   d_x(bottom) = E d_in + Z d_x(above)
//           Every workgroup solves the whole top alone, from the values that the
//           groups publish (o of a strand whose parent is elsewhere, the provisional x
//           at a bottom whose child is elsewhere): one exchange a step.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

namespace nrt {

constexpr int kResC = 8;         // rows per unit
constexpr int kResT = 512;       // most units per group
constexpr int kResDyn = 8;       // most dynamic rows (eight lanes of one wave gate each)
constexpr int kResTopMax = 1900; // most top nodes (their LDS: 68 B each and the published values)
constexpr int kResRounds = 6;    // lane-scan rounds of a piece of 64 units

// Per-unit coefficients (arrays of G * T doubles).
enum { kUZ = 0,     // product of F over the unit's rows
       kUBelow,     // product of Z over the units below it in its piece
       kUAbove,     // product of Z over the units above it in its piece
       kUCum,       // response of the value above it to the value above its strand's
                    // outermost non-top ancestor (or of its own strand, when top)
       kUEin,       // top strands: response of the value above it to d_in
       kUBin,       // top strands: d_in as it reaches the unit's bottom row
       kUnitArrays };

struct ResPlanHost {
  int N = 0, G = 0, T = 0, nd = 0, nt = 0, npub = 1, nth = 0, top_narrow = 0, rounds = 0;
  int owner = 0;                   // group that stores the dynamic rows' state
  std::vector<int32_t> slot;       // [N] slot of each row: (g * C + k) * T + t; dynamic
                                   // row j at G * C * T + j (its gates follow)
  std::vector<double> F, I;        // [G * C * T]
  std::vector<double> uco;         // kUnitArrays x [G * T]
  std::vector<uint32_t> uinf;      // 3 words per unit: piece | pos << 10 | len << 16 |
                                   // top << 31; na | pa << 16; the strand's own top node
                                   // (nt: none) | parent piece << 16
  std::vector<double> pz;          // [G * T] Z of each piece
  std::vector<uint16_t> pinf;      // 8 per piece: child pieces, parent piece, height,
                                   // published o, published x, 0, 0
  std::vector<int32_t> ginfo;      // 4 per group: pieces, heights, first narrow height,
                                   // flags (1: takes part in the exchange)
  std::vector<double> tz, te;      // top nodes, by height
  std::vector<uint16_t> tinf;      // 6 per node: (published, node) of up to two
                                   // children, (node, published) of the value above
  std::vector<int32_t> thoff;      // [nth + 1]
  std::vector<int32_t> dyn_row;    // children before parents
  std::vector<double> dyn_s, dyn_u;  // static children's share of the pivot; coupling to
                                     // the parent (both directions)
  std::vector<uint16_t> dinf;      // 6 per dynamic row: (published, node) x 2, parent
                                   // (0xFFFF none), 0
  std::vector<uint16_t> epiece;    // G = 1: piece of each published o
  int64_t ns0() const { return (int64_t)G * kResC * T + 4 * nd; }  // (V, m, h, n each)
};

constexpr int kResNone = 0x3FF;    // uinf: no piece (an idle lane)

// Builds the plan. diag/up/dn: A[i][i], A[i][par], A[par][i]. hh_row: rows whose
// diagonal changes every step. Returns false (and says why) where the form does not
// apply: too many dynamic rows, an asymmetric coupling, more than two children, a top
// that does not fit.
bool build_resident_plan(int N, const std::vector<int32_t>& par, const std::vector<double>& diag,
                         const std::vector<double>& up, const std::vector<double>& dn,
                         const std::vector<int32_t>& hh_row, int T, ResPlanHost& P,
                         std::string& why);

// The step's solve as the kernel does it, phase by phase, on the host (tests).
void resident_solve_host(const ResPlanHost& P, const double* b, const double* dyn_diag, double* x);

// Bytes of dynamic LDS of one workgroup.
inline size_t resident_lds_bytes(int T, int npub, int nt, int nth, int nd) {
  return 8 * ((size_t)((3 + kResC + 1) * T + 2) + npub + 5 * (size_t)nt + 3 + nd + 3 * kResDyn) +
         12 * (size_t)nt + 4 * (size_t)(nth + 2) + 16;
}

}  // namespace nrt
