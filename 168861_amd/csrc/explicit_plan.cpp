// Host plan of the resident explicit step (explicit_tree.hpp), and the step as the
// kernel does it, on the host (tests).
#include <algorithm>
#include <cmath>
#include <cstring>
#include "explicit_tree.hpp"

namespace nrt {

bool build_explicit_plan(const HostProblem& p, int T, int every, ExPlanHost& P, std::string& why) {
  constexpr int C = kExC;
  P = ExPlanHost();
  const int N = p.N;
  P.N = N;
  P.T = T;
  P.every = every;
  auto no = [&](const char* w) {
    why = w;
    return false;
  };
  if (N < 4 || p.T < 1 || p.terminals[0] != 0) return no("first terminal");
  std::vector<uint8_t> mark(N + 8, 0);  // 1: sealed end, 2: HH element, 4: stimulus
  struct Bit {
    const uint8_t* m;
    uint8_t b;
    bool operator[](int j) const { return m[j] & b; }
  };
  const Bit term{mark.data(), 1}, hh{mark.data(), 2};
  for (int k = 0; k < p.T; k++) {
    if (k > 0 && p.terminals[k] == 0) return no("first terminal twice");
    mark[p.terminals[k]] = 1;
  }
  if (!term[N - 1]) return no("last element is no sealed end");
  if (p.H > kExDyn) return no("too many HH elements");
  for (int i = 0; i < p.H; i++) {
    const int e = p.hh_elem[i];
    if (mark[e]) return no("HH element");
    mark[e] = 2;
  }
  auto hh_index = [&](int e) {
    return (int)(std::find(p.hh_elem.begin(), p.hh_elem.end(), e) - p.hh_elem.begin());
  };
  if (p.mother[1] != 0) return no("element 1");
  // amid[j]: a passive, unbranched element after its mother and before its only daughter, by
  // its own entries (eight at a time below: most elements are amid a strand)
  std::vector<uint8_t> amid(N + 8, 0);
  {
    const int32_t *mo = p.mother.data(), *dr = p.dr.data();
    const uint8_t *br = p.branching.data(), *mk = mark.data();
    uint8_t* __restrict__ to = amid.data();
    for (int j = 1; j < N; j++) {
      const unsigned off = ((unsigned)mo[j] ^ (unsigned)(j - 1)) |
                           ((unsigned)dr[j] ^ (unsigned)(j + 1)) | br[j] | mk[j];
      to[j] = off == 0 ? 1 : 0;
    }
  }
  const auto all_amid = [&](int j) {  // of j .. j + 7
    uint64_t w;
    std::memcpy(&w, amid.data() + j, 8);
    return w == 0x0101010101010101ull;
  };
  // every computed element: its daughters name it as their mother, and the other way
  auto daughter = [&](int j, int d) { return d >= 1 && d < N && p.mother[d] == j; };
  for (int j = 1; j < N; j++) {
    while (all_amid(j - 1)) j += 6;
    if (amid[j - 1] & amid[j] & amid[j + 1]) continue;  // (all of the below)
    const int m = p.mother[j];
    if (term[j]) {
      // a sealed end: the next element after a passive, unbranched source
      if (m != j - 1 || m < 1 || term[m] || hh[m] || p.branching[m] || p.dr[m] != j)
        return no("sealed end");
      continue;
    }
    if (j >= 2) {
      if (m < 1 || m >= j || term[m]) return no("mother");
      if (p.dr[m] != j && !(p.branching[m] && p.dl[m] == j)) return no("mother's daughters");
    }
    if (!daughter(j, p.dr[j])) return no("right daughter");
    if (p.branching[j]) {
      if (!daughter(j, p.dl[j]) || p.dl[j] == p.dr[j] || term[p.dl[j]] || term[p.dr[j]])
        return no("left daughter");
    } else if (hh[j] && term[p.dr[j]]) {
      return no("sealed end of an HH element");
    }
  }
  {
    const double* in = p.input.data();
    uint8_t* __restrict__ to = mark.data();
    for (int j = 1; j < N; j++) to[j] |= in[j] != 0.0 ? 4 : 0;
  }
  // ---- nodes in element order: units (chains cut from their ends) and HH elements
  struct Node {
    int32_t first, n, last, dyn;  // dyn -1: a unit
    int32_t up, right, left;      // nodes (-1: none)
  };
  std::vector<Node> node;
  node.reserve(N / C + N / 16 + 16);
  std::vector<int32_t> node_of(N, -1);  // of first and last elements
  for (int j = 1; j < N;) {
    if (hh[j]) {
      node_of[j] = (int)node.size();
      node.push_back({j, 1, j, hh_index(j), -1, -1, -1});
      j++;
      continue;
    }
    int e = j;  // last element of the chain that starts at j
    while (all_amid(e)) e += 7;
    while (e + 1 < N && !term[e] && !hh[e + 1] && p.mother[e + 1] == e && p.dr[e] == e + 1 &&
           !p.branching[e])
      e++;
    int n = (e - j) % C + 1;
    for (int at = j; at <= e; at += n, n = C) {
      node_of[at] = node_of[at + n - 1] = (int)node.size();
      node.push_back({at, n, at + n - 1, -1, -1, -1, -1});
    }
    j = e + 1;
  }
  const int nn = (int)node.size();
  for (Node& q : node) {
    if (q.first > 1) q.up = node_of[p.mother[q.first]];
    if (term[q.last]) continue;
    q.right = node_of[p.dr[q.last]];
    if (p.branching[q.last]) q.left = node_of[p.dl[q.last]];
  }
  P.units = nn - p.H;
  // ---- groups
  if (P.units <= T) T = std::max(64, (P.units + 63) / 64 * 64);
  P.T = T;
  struct Visit {
    int32_t node, dist, from;
    bool from_up;  // entered at its first element
  };
  std::vector<Visit> todo;
  std::vector<int32_t> in(nn, -1), at(nn, 0), slot(nn, -1), own, halo, fresh;
  std::vector<int32_t> owner(nn, -1);
  std::vector<std::vector<int32_t>> members;  // own nodes, then the halo's
  std::vector<int32_t> nown;
  for (int s = 0; s < nn;) {
    const int g = P.G++;
    own.clear();
    halo.clear();
    int units = 0;
    while (s < nn) {
      // node s and what its owner needs besides
      fresh.clear();
      todo.clear();
      auto see = [&](int w, int dist, int from, bool from_up) {
        // (what lies beyond an owned node is nearer to that one, and there already)
        if (w >= 0 && dist <= every && owner[w] != g) todo.push_back({w, dist, from, from_up});
      };
      see(node[s].up, 1, s, false);
      see(node[s].right, 1, s, true);
      see(node[s].left, 1, s, true);
      for (size_t k = 0; k < todo.size(); k++) {
        const Visit v = todo[k];
        const Node& q = node[v.node];
        if (in[v.node] != g) fresh.push_back(v.node);
        if (v.from_up) {
          see(q.right, v.dist + q.n, v.node, true);
          see(q.left, v.dist + q.n, v.node, true);
        } else {
          see(q.up, v.dist + q.n, v.node, false);
          if (q.right != v.from) see(q.right, v.dist + 1, v.node, true);
          if (q.left != v.from) see(q.left, v.dist + 1, v.node, true);
        }
      }
      int more = in[s] != g && node[s].dyn < 0 ? 1 : 0;
      for (int w : fresh) more += node[w].dyn < 0 ? 1 : 0;
      if (units + more > T) break;
      units += more;
      in[s] = g;
      owner[s] = g;
      own.push_back(s);
      for (int w : fresh) {
        in[w] = g;
        halo.push_back(w);
      }
      s++;
    }
    if (own.empty()) return no("a group's halo");
    nown.push_back((int)own.size());
    for (int w : halo)
      if (owner[w] != g) own.push_back(w);
    members.push_back(own);
  }
  // ---- records
  const int G = P.G;
  P.unit.assign((size_t)G * T, ExUnit{});
  P.dyn.assign((size_t)G * kExDyn, ExDynUnit{});
  for (ExDynUnit& d : P.dyn) d.elem = -1;
  for (int g = 0; g < G; g++)
    for (size_t k = nown[g]; k < members[g].size(); k++) {
      int32_t& sl = slot[members[g][k]];
      if (sl < 0) sl = P.slots++;
    }
  for (int g = 0; g < G; g++) {
    const auto& mem = members[g];
    // units with unused places side by side, then other ends of chains: fewer waves do
    // what only these need
    int next[4] = {0, 0, 0, 0};  // of the kinds: 0 HH elements, 1 .. 3 units
    const auto kind = [&](const Node& q) {
      return q.dyn >= 0 ? 0 : q.n < C ? 1 : term[q.last] || q.left >= 0 ? 2 : 3;
    };
    for (int w : mem) next[kind(node[w])]++;
    next[3] = next[1] + next[2];
    next[2] = next[1];
    next[0] = next[1] = 0;
    for (int w : mem) {
      in[w] = g;
      at[w] = next[kind(node[w])]++;
    }
    auto head = [&](int w) {
      if (w < 0 || in[w] != g) return (uint16_t)kExMissing;
      return (uint16_t)(node[w].dyn < 0 ? at[w] : 2 * kExT + at[w]);
    };
    auto bottom = [&](int w) {
      if (w < 0 || in[w] != g) return (uint16_t)kExMissing;
      return (uint16_t)(node[w].dyn < 0 ? kExT + at[w] : 2 * kExT + at[w]);
    };
    for (size_t k = 0; k < mem.size(); k++) {
      const int w = mem[k];
      const Node& q = node[w];
      uint32_t fl = kExUOn | (q.up < 0 ? kExUGhost : 0) | (q.left >= 0 ? kExUBranch : 0) |
                    (term[q.last] ? kExUTerm : 0) | (owner[w] != g ? kExUHalo : 0);
      const int er = q.right >= 0 ? p.dr[q.last] : q.last, el = q.left >= 0 ? p.dl[q.last] : q.last;
      double input = 0;
      uint64_t marks;  // (of the unit's elements, and perhaps some after them)
      std::memcpy(&marks, mark.data() + q.first, 8);
      for (int k = 0; k < q.n && (marks & 0x0404040404040404ull); k++) {
        const int j = q.first + k;
        if (term[j] || p.input[j] == 0.0) continue;
        if (fl & kExUInput) return no("two stimuli in a unit");
        input = p.input[j];
        fl |= kExUInput | (uint32_t)(C - q.n + k) << 8;
      }
      if (q.dyn < 0) {
        P.unit[(size_t)g * T + at[w]] = {q.first, fl | (uint32_t)(C - q.n), bottom(q.up),
                                         head(q.right), head(q.left), 0, er, el, slot[w], input};
      } else {
        P.dyn[(size_t)g * kExDyn + at[w]] = {q.first, q.dyn, fl, bottom(q.up), head(q.right),
                                             head(q.left), 0, er, el, slot[w], input};
      }
    }
  }
  return true;
}

}  // namespace nrt

// Steps of a problem by the plan, every group by itself with exchanges between, with host
// arrays for the kernel's registers and LDS (a missing neighbour is NaN) and IEEE
// divisions, in the kernel's order of operations.
extern "C" int nrt_test_explicit_tree_host(const nrt_problem* np, int T, int steps, int a0, int a1,
                                           double* V, int32_t* info, char* why, int why_len) {
  using namespace nrt;
  constexpr int C = kExC;
  HostProblem p;
  try {
    p = load_problem(np);
  } catch (const std::exception&) {
    return 1;
  }
  ExPlanHost P;
  std::string w;
  const bool ok = build_explicit_plan(p, T, kExEvery, P, w) ||
                  build_explicit_plan(p, T, kExEveryDense, P, w);
  if (why && why_len > 0) {
    std::strncpy(why, w.c_str(), (size_t)why_len - 1);
    why[why_len - 1] = 0;
  }
  if (!ok) return 7;
  T = P.T;
  const int G = P.G;
  struct Dyn {
    double v, m, h, n;
  };
  std::vector<double> R((size_t)G * T * C), v0(G, p.V0[0]), slots((size_t)P.slots * kExSlotVals, NAN);
  std::vector<Dyn> D((size_t)G * kExDyn);
  auto count = [&](const ExUnit& u) { return C - (int)(u.flags & 7); };
  for (int i = 0; i < G * T; i++)
    for (int k = 0; k < count(P.unit[i]) && (P.unit[i].flags & kExUOn); k++)
      R[(size_t)i * C + k] = p.V0[P.unit[i].first + k];
  for (size_t i = 0; i < D.size(); i++)
    if (P.dyn[i].elem >= 0)
      D[i] = {p.V0[P.dyn[i].elem], p.m[P.dyn[i].hh], p.h[P.dyn[i].hh], p.n[P.dyn[i].hh]};
  auto rdx = [&](int j) { return p.r_a[j] * p.dx[j]; };
  for (int st = 1; st <= steps; st++) {
    const bool active = st >= a0 && st <= a1;
    if (st > 1 && (st - 1) % P.every == 0)
      for (int put = 1; put >= 0; put--) {
        for (int i = 0; i < G * T; i++) {
          const ExUnit& u = P.unit[i];
          if (!(u.flags & kExUOn) || u.slot < 0 || (put == 1) == ((u.flags & kExUHalo) != 0)) continue;
          for (int k = 0; k < C; k++) {
            double &a = slots[(size_t)u.slot * kExSlotVals + k], &b = R[(size_t)i * C + k];
            put ? a = b : b = a;
          }
          if (!put && (u.flags & kExUGhost)) v0[i / T] = R[(size_t)i * C];
        }
        for (size_t i = 0; i < D.size(); i++) {
          const ExDynUnit& u = P.dyn[i];
          if (u.elem < 0 || u.slot < 0 || (put == 1) == ((u.flags & kExUHalo) != 0)) continue;
          Dyn& a = *(Dyn*)&slots[(size_t)u.slot * kExSlotVals];
          put ? a = D[i] : D[i] = a;
          if (!put && (u.flags & kExUGhost)) v0[i / kExDyn] = a.v;
        }
      }
    for (int g = 0; g < G; g++) {
      std::vector<double> lds(kExVals, NAN);
      for (int t = 0; t < T; t++) {
        const ExUnit& u = P.unit[(size_t)g * T + t];
        if (!(u.flags & kExUOn)) continue;
        lds[t] = R[((size_t)g * T + t) * C];
        lds[kExT + t] = R[((size_t)g * T + t) * C + count(u) - 1];
      }
      for (int i = 0; i < kExDyn; i++) lds[2 * kExT + i] = D[g * kExDyn + i].v;
      double ghost = v0[g];
      auto finish = [&](int j, double v, double tdr, bool br, double tdl, double tmo, double wd,
                        double kd, bool stim, double input) {
        double s = br ? tdl + tdr : tdr;
        s = s + tmo;
        s = s + wd * v;
        s = s + kd;
        if (active && stim) s = s + input;
        return v + p.dT / (p.c_m[j] * p.dx[j]) * s;
      };
      for (int t = 0; t < T; t++) {
        const ExUnit& u = P.unit[(size_t)g * T + t];
        if (!(u.flags & kExUOn)) continue;
        double* v = &R[((size_t)g * T + t) * C];
        double above = u.flags & kExUGhost ? v0[g] : lds[u.up];
        for (int k = 0; k < count(u); k++) {
          const int j = u.first + k;
          const bool end = k == count(u) - 1;
          if (end && (u.flags & kExUTerm)) {
            v[k] = v[k - 1];
            continue;
          }
          const double below = end ? lds[u.right] : v[k + 1], was = v[k];
          const double tdr = (below - was) / rdx(end ? u.el_right : j + 1);
          const bool br = end && (u.flags & kExUBranch);
          const double tdl = br ? (lds[u.left] - was) / rdx(u.el_left) : 0.0;
          v[k] = finish(j, was, tdr, br, tdl, -((was - above) / rdx(j)), p.W[j] * p.dx[j],
                        p.K[j] * p.dx[j],
                        (u.flags & kExUInput) && (int)(u.flags >> 8 & 7) == k + (int)(u.flags & 7),
                        u.input);
          above = was;
        }
        if (u.flags & kExUGhost) ghost = v[0];
      }
      for (int i = 0; i < kExDyn; i++) {
        const ExDynUnit& d = P.dyn[(size_t)g * kExDyn + i];
        if (d.elem < 0) continue;
        Dyn& y = D[(size_t)g * kExDyn + i];
        const int j = d.elem, k = d.hh;
        const double dt = p.dT * 1000, v = y.v, un = ((v + p.ls_Na[k]) - p.rest[k]) / 0.001,
                     uk = ((v + p.ls_K[k]) - p.rest[k]) / 0.001;
        const double am = (2.5 - 0.1 * un) / (exp(2.5 - 0.1 * un) - 1), bm = 4 * exp(-un / 18),
                     ah = 0.07 * exp(-un / 20), bh = 1 / (exp(3 - 0.1 * un) + 1),
                     an = (0.1 - 0.01 * uk) / (exp(1 - 0.1 * uk) - 1), bn = 0.125 * exp(-uk / 80);
        y.m = y.m + dt * (am * (1 - y.m) - bm * y.m);
        y.h = y.h + dt * (ah * (1 - y.h) - bh * y.h);
        y.n = y.n + dt * (an * (1 - y.n) - bn * y.n);
        const double gna = p.g_Na[k] * y.m * y.m * y.m * y.h,
                     gk = p.g_K[k] * y.n * y.n * y.n * y.n, gl = p.G_L[k];
        const double Wd = -(gna + gk + gl) * p.dx[j],
                     Kd = (gna * p.E_Na[k] + gk * p.E_K[k] + gl * p.E_L[k]) * p.dx[j];
        const bool br = d.flags & kExUBranch;
        const double vm = d.flags & kExUGhost ? v0[g] : lds[d.up];
        y.v = finish(j, v, (lds[d.right] - v) / rdx(d.el_right), br,
                     br ? (lds[d.left] - v) / rdx(d.el_left) : 0.0, (vm - v) / rdx(j), Wd, Kd,
                     d.flags & kExUInput, d.input);
        if (d.flags & kExUGhost) ghost = y.v;
      }
      v0[g] = ghost;
    }
  }
  std::fill(V, V + p.N, NAN);
  for (int i = 0; i < G * T; i++) {
    const ExUnit& u = P.unit[i];
    if (!(u.flags & kExUOn) || (u.flags & kExUHalo)) continue;
    for (int k = 0; k < count(u); k++) V[u.first + k] = R[(size_t)i * C + k];
    if (u.flags & kExUGhost) V[0] = v0[i / T];
  }
  for (size_t i = 0; i < D.size(); i++) {
    const ExDynUnit& u = P.dyn[i];
    if (u.elem < 0 || (u.flags & kExUHalo)) continue;
    V[u.elem] = D[i].v;
    if (u.flags & kExUGhost) V[0] = v0[i / kExDyn];
  }
  const int32_t out[5] = {G, P.T, P.slots, P.units, P.every};
  if (info) std::memcpy(info, out, sizeof(out));
  return 0;
}
