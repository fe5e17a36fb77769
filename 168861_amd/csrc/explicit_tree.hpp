// Explicit steps of a branching neurite with its elements resident in registers: the
// plan (made on the host) and the kernel's records.
//
// A unit is kExC consecutive elements of a chain (each the mother of the next), one
// thread's; a chain is cut from its end, so its first unit may begin with unused
// places. At most kExDyn HH elements stand outside the units, each with lanes of its own.
// A group (workgroup) owns consecutive units and computes, besides, every unit with an
// element at most `every` elements away from one that it owns (its halo): without the
// neighbours that are missing there, the halo's values become wrong from its outside, one
// element a step, and reach no owned element within `every` steps, after which the
// halo's values are fetched from their owners. `every` is kExEvery, or kExEveryDense where
// a halo of that width would not fit (branches a few elements apart: the halo doubles at
// each).
#pragma once
#include <cstdint>
#include <string>
#include <vector>
#include "nrt_internal.hpp"

namespace nrt {

constexpr int kExC = 8;      // elements per unit
constexpr int kExT = 512;    // most units (owned and halo) per group
constexpr int kExDyn = 8;    // most HH elements
constexpr int kExEvery = 16, kExEveryDense = 4;  // steps between exchanges

// Unit flags; the number of unused places is in bits 0..2, the place of the element with
// a stimulus (one at most) in bits 8..10.
constexpr uint32_t kExUOn = 8, kExUBranch = 16, kExUTerm = 32, kExUGhost = 64, kExUHalo = 128,
                   kExUInput = 2048;

// A neighbour's potential in a group's LDS values: first elements of units at 0, last
// ones at kExT, HH elements at 2 kExT, then one place for a neighbour that is missing.
constexpr int kExVals = 2 * kExT + kExDyn + 1;
constexpr int kExMissing = kExVals - 1;

struct ExUnit {
  int32_t first;              // element in the first used place
  uint32_t flags;
  uint16_t up, right, left, pad;  // LDS places: mother, right and left daughter
  int32_t el_right, el_left;  // daughters' elements (their r_a dx)
  int32_t slot;               // exchanged values (-1: not exchanged)
  double input;
};
struct ExDynUnit {
  int32_t elem, hh;           // elem -1: unused
  uint32_t flags;             // kExUBranch, kExUGhost, kExUHalo
  uint16_t up, right, left, pad;
  int32_t el_right, el_left;
  int32_t slot;
  double input;
};
static_assert(sizeof(ExUnit) == 40 && sizeof(ExDynUnit) == 40, "plan records");
constexpr int kExSlotVals = kExC;  // doubles of an exchange slot (V; of an HH element V, m, h, n)

struct ExPlanHost {
  int N = 0, G = 0, T = 0, slots = 0, units = 0, every = 0;
  std::vector<ExUnit> unit;    // [G * T]
  std::vector<ExDynUnit> dyn;  // [G * kExDyn]
};

// Groups of at most T <= kExT units (one of as many as needed, where that is enough).
bool build_explicit_plan(const HostProblem& p, int T, int every, ExPlanHost& P, std::string& why);

}  // namespace nrt
