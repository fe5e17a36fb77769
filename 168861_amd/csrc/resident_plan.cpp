// Host plan of the resident tree solve (resident.hpp).
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include "resident.hpp"

namespace nrt {

namespace {
struct Strand {
  int first, last;     // rows
  int chain;
  int group;
  int parent;          // strand, -1: none, -2 - j: dynamic row j
  int piece0, npiece;  // pieces in the group, from the head
  bool top = false;
  int node = -1, height = 0, edge = 0, xpub = 0;
  int child[2] = {-1, -1};
  // attachment of the strand's value above its head
  int na = 0, pa = 0;
  double cum = 0, z = 1, e = 0;
};
struct Piece {
  int strand, lane0, units, first;  // first row
  int parent = -1, child[2] = {-1, -1}, height = 0, order = 0;
};
}  // namespace

bool build_resident_plan(int N, const std::vector<int32_t>& par, const std::vector<double>& diag,
                         const std::vector<double>& up, const std::vector<double>& dn,
                         const std::vector<int32_t>& hh_row, int T, ResPlanHost& P,
                         std::string& why) {
  constexpr int C = kResC;
  P = ResPlanHost();
  P.N = N;
  P.T = T;
  // ---- dynamic rows: HH rows and every row above one
  std::vector<int32_t> dynj(N, -1);
  std::vector<int32_t> dyn;
  for (int r : hh_row)
    for (int i = r; i >= 0 && dynj[i] < 0; i = par[i]) {
      dynj[i] = 0;
      dyn.push_back(i);
      if ((int)dyn.size() > kResDyn) {
        why = "too many rows change";
        return false;
      }
    }
  std::sort(dyn.begin(), dyn.end(), std::greater<int>());  // children before parents
  P.nd = (int)dyn.size();
  for (int j = 0; j < P.nd; j++) dynj[dyn[j]] = j;
  P.dyn_row.assign(dyn.begin(), dyn.end());
  // ---- children, factors of the static rows
  std::vector<int32_t> kid(2 * (size_t)N, -1);
  for (int i = 0; i < N; i++) {
    const int p = par[i];
    if (p < 0) continue;
    if (p >= i) {
      why = "a parent after its child";
      return false;
    }
    int32_t* k = &kid[2 * (size_t)p];
    if (k[0] < 0) k[0] = i;
    else if (k[1] < 0) k[1] = i;
    else {
      why = "more than two children";
      return false;
    }
    if (up[i] != dn[i]) {
      why = "asymmetric coupling";
      return false;
    }
  }
  // (in extended precision: what is rounded once here acts in every step)
  std::vector<long double> d(diag.begin(), diag.end());
  std::vector<double> F(N, 0.0), I(N, 0.0);
  std::vector<long double> dyn_s(P.nd, 0.0L);
  P.dyn_s.assign(P.nd, 0.0);
  P.dyn_u.assign(P.nd, 0.0);
  for (int i = N - 1; i >= 0; i--) {
    const int p = par[i];
    if (dynj[i] >= 0) {
      P.dyn_u[dynj[i]] = p >= 0 ? up[i] : 0.0;
      continue;
    }
    const long double inv = 1.0L / d[i], u = up[i];
    I[i] = (double)inv;
    if (p < 0) continue;
    F[i] = (double)(-u * inv);
    if (dynj[p] >= 0) dyn_s[dynj[p]] += u * u * inv;
    else d[p] -= u * u * inv;
  }
  for (int j = 0; j < P.nd; j++) P.dyn_s[j] = (double)dyn_s[j];
  // ---- chains of static rows (single rows without parent and child apart)
  struct Chain {
    int first, last, depth;
  };
  std::vector<Chain> chains;
  std::vector<int32_t> chain_of(N, -1), singles;
  for (int i = 0; i < N; i++) {
    if (dynj[i] >= 0) continue;
    const int p = par[i];
    if (p < 0 && kid[2 * (size_t)i] < 0) {
      singles.push_back(i);
      continue;
    }
    const bool goes_on = p == i - 1 && p >= 0 && dynj[p] < 0 && kid[2 * (size_t)p + 1] < 0;
    if (goes_on) {
      chain_of[i] = chain_of[p];
      chains[chain_of[p]].last = i;
    } else {
      chain_of[i] = (int)chains.size();
      chains.push_back({i, i, p < 0 || dynj[p] >= 0 ? 0 : chains[chain_of[p]].depth + 1});
    }
  }
  // (a child that is not the next row hangs at its parent's chain end: a row with a
  // child elsewhere and one at the next row has two children, so its chain ends there;
  // a row whose only child is elsewhere is followed by a row that starts a chain)
  // ---- groups: chains in row order, at most T lanes each; a piece stays in its wave.
  // A full group is cut, within its last eighth, where the fewest strands lead up to
  // the cut (they become top nodes), a chain's inside counting one more than its head.
  std::vector<Strand> strands;
  std::vector<std::vector<Piece>> pieces;  // per group
  std::vector<int32_t> last_strand((size_t)chains.size(), -1);
  auto place_group = [&](size_t& ci, int& row) {
    struct Put {
      size_t chain;
      int first, rows, lane;
    };
    std::vector<Put> puts;
    struct Cut {
      size_t puts, chain;
      int row, cost;
    };
    Cut best{0, 0, 0, -1};
    int lane = 0;
    size_t c = ci;
    int r = row;
    bool full = false;
    while (c < chains.size() && !full) {
      if (lane >= T - T / 8 && r == chains[c].first && lane < T) {
        const Cut k{puts.size(), c, r, chains[c].depth};
        if (best.cost < 0 || k.cost <= best.cost) best = k;
      }
      int left = chains[c].last - r + 1;
      const int units = (left + C - 1) / C;
      const int room = 64 - lane % 64;
      if (units <= 8 && units > room) lane += room;
      while (left > 0) {
        if (lane >= T) {
          full = true;
          break;
        }
        const int n = std::min((left + C - 1) / C, 64 - lane % 64);
        const int rows = std::min(left, n * C);
        puts.push_back({c, r, rows, lane});
        lane += n;
        r += rows;
        left -= rows;
      }
      if (!full) {
        c++;
        if (c < chains.size()) r = chains[c].first;
      }
    }
    if (full) {
      const bool inside = r != chains[c].first;
      const int cost = chains[c].depth + (inside ? 1 : 0);
      if (best.cost < 0 || cost <= best.cost) best = {puts.size(), c, r, cost};
      puts.resize(best.puts);
      c = best.chain;
      r = best.row;
    }
    const int g = (int)pieces.size();
    pieces.emplace_back();
    for (const Put& q : puts) {
      Strand* s = strands.empty() ? nullptr : &strands.back();
      if (!s || s->group != g || s->chain != (int)q.chain) {
        Strand n{};
        n.first = q.first;
        n.last = q.first - 1;
        n.chain = (int)q.chain;
        n.group = g;
        n.piece0 = (int)pieces[g].size();
        n.npiece = 0;
        n.z = 1;
        const int hp = par[q.first];
        if (q.first != chains[q.chain].first) n.parent = last_strand[q.chain];
        else if (hp < 0) n.parent = -1;
        else if (dynj[hp] >= 0) n.parent = -2 - dynj[hp];
        else n.parent = last_strand[chain_of[hp]];
        strands.push_back(n);
        s = &strands.back();
        last_strand[q.chain] = (int)strands.size() - 1;
      }
      Piece p;
      p.strand = (int)strands.size() - 1;
      p.lane0 = q.lane;
      p.units = (q.rows + C - 1) / C;
      p.first = q.first;
      pieces[g].push_back(p);
      s->npiece++;
      s->last = q.first + q.rows - 1;
    }
    ci = c;
    row = r;
  };
  size_t ci = 0;
  int row = chains.empty() ? 0 : chains[0].first;
  while (ci < chains.size()) place_group(ci, row);
  // single rows: C to a unit, in the lanes that the pieces leave free, then in further
  // groups
  std::vector<std::pair<int, int>> single_at;  // (group, lane) per unit of singles
  const size_t nsu = (singles.size() + C - 1) / C;
  for (int g = 0; single_at.size() < nsu; g++) {
    if (g == (int)pieces.size()) pieces.emplace_back();
    std::vector<uint8_t> used(T, 0);
    for (const Piece& p : pieces[g])
      for (int u = 0; u < p.units; u++) used[p.lane0 + u] = 1;
    for (int t = 0; t < T && single_at.size() < nsu; t++)
      if (!used[t]) single_at.push_back({g, t});
  }
  if (pieces.empty()) pieces.emplace_back();
  const int G = P.G = (int)pieces.size();
  const int nst = (int)strands.size();
  // ---- strands: children, top set, cut edges
  for (int s = 0; s < nst; s++) {
    const int p = strands[s].parent;
    if (p < 0) continue;
    Strand& q = strands[p];
    q.child[q.child[0] < 0 ? 0 : 1] = s;
    if (q.group != strands[s].group)
      for (int a = p; a >= 0 && !strands[a].top; a = strands[a].parent) strands[a].top = true;
  }
  int edges = 0;
  std::vector<uint8_t> exch(G, 0);
  std::vector<std::pair<int, int>> edge_at;  // (group, strand)
  for (int s = 0; s < nst; s++) {
    Strand& q = strands[s];
    const bool cut = q.parent <= -2 || (q.parent >= 0 && strands[q.parent].group != q.group);
    if (!cut) continue;
    q.edge = ++edges;
    edge_at.push_back({q.group, s});
    exch[q.group] = 1;
  }
  int xs = 0;
  for (int s = 0; s < nst; s++) {
    Strand& q = strands[s];
    for (int k = 0; k < 2; k++)
      if (q.child[k] >= 0 && strands[q.child[k]].group != q.group && q.xpub == 0) {
        q.xpub = 1 + edges + xs++;
        exch[q.group] = 1;
      }
  }
  P.npub = 1 + edges + xs;
  for (int g = G - 1; g >= 0; g--)
    if (exch[g]) P.owner = g;
  // ---- top nodes by height (children have larger strand numbers than their parents)
  std::vector<int> tops;
  for (int s = nst - 1; s >= 0; s--) {
    Strand& q = strands[s];
    if (!q.top) continue;
    tops.push_back(s);
    q.height = 0;
    for (int k = 0; k < 2; k++)
      if (q.child[k] >= 0 && strands[q.child[k]].top)
        q.height = std::max(q.height, strands[q.child[k]].height + 1);
  }
  std::stable_sort(tops.begin(), tops.end(),
                   [&](int a, int b) { return strands[a].height < strands[b].height; });
  const int nt = P.nt = (int)tops.size();
  if (nt > kResTopMax) {
    why = "the top does not fit";
    return false;
  }
  for (int j = 0; j < nt; j++) strands[tops[j]].node = j;
  P.nth = nt ? strands[tops.back()].height + 1 : 0;
  P.thoff.assign(P.nth + 1, 0);
  for (int s : tops) P.thoff[strands[s].height + 1]++;
  for (int h = 0; h < P.nth; h++) P.thoff[h + 1] += P.thoff[h];
  P.top_narrow = P.nth;
  while (P.top_narrow > 0 && P.thoff[P.top_narrow] - P.thoff[P.top_narrow - 1] <= 64) P.top_narrow--;
  // ---- strand coefficients and attachments (parents first)
  P.F.assign((size_t)G * C * T, 0.0);
  P.I.assign((size_t)G * C * T, 0.0);
  P.slot.assign(N, -1);
  P.uco.assign((size_t)kUnitArrays * G * T, 0.0);
  P.uinf.assign(3 * (size_t)G * T, 0);
  P.pz.assign((size_t)G * T, 0.0);
  P.pinf.assign(8 * (size_t)G * T, 0);
  P.ginfo.assign(4 * (size_t)G, 0);
  for (size_t u = 0; u < (size_t)G * T; u++) {
    P.uinf[3 * u] = kResNone | (1u << 16);
    P.uinf[3 * u + 1] = (uint32_t)nt;             // zero entries
    P.uinf[3 * u + 2] = (uint32_t)nt | ((uint32_t)T << 16);
  }
  auto uco = [&](int a, int g, int t) -> double& { return P.uco[((size_t)a * G + g) * T + t]; };
  std::vector<double> pr, xr;  // per row of a strand: product of F below it, response to d_in
  for (int s = 0; s < nst; s++) {
    Strand& q = strands[s];
    if (q.parent <= -2) {
      q.na = nt + 1 + (-2 - q.parent);
      q.cum = 1;
    } else if (q.parent == -1) {
      q.na = nt;
      q.cum = 0;
    } else {
      const Strand& a = strands[q.parent];
      if (a.group != q.group) {
        q.na = a.node;
        q.pa = a.xpub;
        q.cum = 1;
      } else if (a.top) {
        q.na = a.node;
        q.cum = 1;
      } else {
        q.na = a.na;
        q.pa = a.pa;
        q.cum = a.cum * a.z;
      }
    }
    const int n = q.last - q.first + 1;
    pr.assign(n, 1.0);
    xr.assign(n, 0.0);
    for (int k = n - 2; k >= 0; k--) pr[k] = pr[k + 1] * F[q.first + k + 1];
    for (int k = 0; k < n; k++) {
      const int i = q.first + k;
      xr[k] = I[i] * pr[k] + (k > 0 ? F[i] * xr[k - 1] : 0.0);
    }
    q.e = xr[n - 1];
    q.z = 1;
    double above = 1;  // product of Z over the strand's units above
    for (int pi = q.piece0; pi < q.piece0 + q.npiece; pi++) {
      Piece& p = pieces[q.group][pi];
      const int prow1 = pi + 1 < q.piece0 + q.npiece ? pieces[q.group][pi + 1].first : q.last + 1;
      double pabove = 1;
      for (int u = 0; u < p.units; u++) {
        const int t = p.lane0 + u, g = q.group;
        const int r0 = p.first + u * C, r1 = std::min(prow1, r0 + C);
        double z = 1;
        for (int k = 0; k < C; k++) {
          const size_t at = ((size_t)g * C + k) * T + t;
          const int i = r0 + k;
          if (i < r1) {
            // (the root row's own F is 0: nothing above it)
            P.F[at] = F[i];
            P.I[at] = I[i];
            P.slot[i] = (int32_t)at;
          } else {
            P.F[at] = 1.0;
          }
          z *= P.F[at];
        }
        uco(kUZ, g, t) = z;
        uco(kUAbove, g, t) = pabove;
        uco(kUCum, g, t) = q.cum * above;
        if (q.top) {
          uco(kUEin, g, t) = r0 > q.first ? xr[r0 - q.first - 1] : 0.0;
          uco(kUBin, g, t) = pr[r1 - 1 - q.first];
        }
        pabove *= z;
        above *= z;
      }
      double below = 1;
      for (int u = p.units - 1; u >= 0; u--) {
        const int t = p.lane0 + u;
        uco(kUBelow, q.group, t) = below;
        below *= uco(kUZ, q.group, t);
      }
      P.pz[(size_t)q.group * T + p.lane0] = pabove;  // by lane for now, by order below
    }
    q.z = above;
  }
  // ---- pieces: forest of each group by heights
  int longest = 1;
  P.epiece.assign(P.npub, 0);
  for (int g = 0; g < G; g++) {
    std::vector<Piece>& ps = pieces[g];
    const int np = (int)ps.size();
    std::vector<double> z(np);
    for (int k = 0; k < np; k++) {
      const Strand& q = strands[ps[k].strand];
      z[k] = P.pz[(size_t)g * T + ps[k].lane0];
      longest = std::max(longest, ps[k].units);
      if (k > q.piece0) ps[k].parent = k - 1;
      else if (q.parent >= 0 && strands[q.parent].group == g)
        ps[k].parent = strands[q.parent].piece0 + strands[q.parent].npiece - 1;
      if (ps[k].parent >= 0) {
        Piece& a = ps[ps[k].parent];
        a.child[a.child[0] < 0 ? 0 : 1] = k;
      }
    }
    for (int k = 0; k < np; k++) P.pz[(size_t)g * T + ps[k].lane0] = 0;
    int nh = 0;
    for (int k = np - 1; k >= 0; k--) {
      nh = std::max(nh, ps[k].height + 1);
      if (ps[k].parent >= 0)
        ps[ps[k].parent].height = std::max(ps[ps[k].parent].height, ps[k].height + 1);
    }
    std::vector<int> ord(np);
    for (int k = 0; k < np; k++) ord[k] = k;
    std::stable_sort(ord.begin(), ord.end(),
                     [&](int a, int b) { return ps[a].height > ps[b].height; });
    for (int k = 0; k < np; k++) ps[ord[k]].order = k;
    int narrow = nh;  // heights from here sit in the first wave
    std::vector<int> from(nh + 1, 0);  // pieces of at least this height
    for (const Piece& p : ps) from[p.height]++;
    for (int h = nh - 1; h >= 0; h--) from[h] += h + 1 < nh ? from[h + 1] : 0;
    while (narrow > 1 && from[narrow - 1] <= 64) narrow--;
    P.ginfo[4 * g] = np;
    P.ginfo[4 * g + 1] = nh;
    P.ginfo[4 * g + 2] = narrow;
    P.ginfo[4 * g + 3] = exch[g];
    for (int k = 0; k < np; k++) {
      const Piece& p = ps[k];
      const Strand& q = strands[p.strand];
      uint16_t* f = &P.pinf[8 * ((size_t)g * T + p.order)];
      auto ord_of = [&](int c) { return (uint16_t)(c < 0 ? T : ps[c].order); };
      f[0] = ord_of(p.child[0]);
      f[1] = ord_of(p.child[1]);
      f[2] = ord_of(p.parent);
      f[3] = (uint16_t)p.height;
      f[4] = (uint16_t)(k == q.piece0 ? q.edge : 0);
      f[5] = (uint16_t)(k == q.piece0 + q.npiece - 1 ? q.xpub : 0);
      if (f[4]) P.epiece[f[4]] = (uint16_t)p.order;
      P.pz[(size_t)g * T + p.order] = z[k];
      for (int u = 0; u < p.units; u++) {
        uint32_t* w = &P.uinf[3 * ((size_t)g * T + p.lane0 + u)];
        w[0] = (uint32_t)p.order | (uint32_t)u << 10 | (uint32_t)p.units << 16 |
               (q.top ? 1u << 31 : 0u);
        w[1] = (uint32_t)q.na | (uint32_t)q.pa << 16;
        w[2] = (uint32_t)(q.top ? q.node : nt) | (uint32_t)f[2] << 16;
      }
    }
  }
  while ((1 << P.rounds) < longest) P.rounds++;
  // single rows: independent rows of a unit (F = 0)
  for (size_t k = 0; k < singles.size(); k++) {
    const auto [g, t] = single_at[k / C];
    const size_t at = ((size_t)g * C + k % C) * T + t;
    P.I[at] = I[singles[k]];
    P.slot[singles[k]] = (int32_t)at;
  }
  for (int j = 0; j < P.nd; j++) P.slot[dyn[j]] = (int32_t)((size_t)G * C * T + j);
  // ---- top nodes and dynamic rows
  P.tz.resize(nt);
  P.te.resize(nt);
  P.tinf.assign(6 * (size_t)nt, 0);
  auto child_ref = [&](int c, int group, uint16_t* f) {  // (published, node) of child strand c
    f[0] = 0;
    f[1] = (uint16_t)nt;
    if (c < 0) return;
    const Strand& q = strands[c];
    if (q.group != group) f[0] = (uint16_t)q.edge;
    if (q.top) f[1] = (uint16_t)q.node;
  };
  for (int j = 0; j < nt; j++) {
    const Strand& q = strands[tops[j]];
    P.tz[j] = q.z;
    P.te[j] = q.e;
    uint16_t* f = &P.tinf[6 * (size_t)j];
    child_ref(q.child[0], q.group, f);
    child_ref(q.child[1], q.group, f + 2);
    f[4] = (uint16_t)q.na;
    f[5] = (uint16_t)q.pa;
  }
  P.dinf.assign(6 * (size_t)P.nd, 0);
  for (int j = 0; j < P.nd; j++) {
    uint16_t* f = &P.dinf[6 * (size_t)j];
    int n = 0;
    f[1] = f[3] = (uint16_t)nt;
    for (int k = 0; k < 2; k++) {
      const int c = kid[2 * (size_t)dyn[j] + k];
      if (c < 0 || dynj[c] >= 0) continue;
      // the strand that starts at row c (its chain's first)
      for (const auto& [g, s] : edge_at)
        if (strands[s].first == c) {
          f[2 * n] = (uint16_t)strands[s].edge;
          if (strands[s].top) f[2 * n + 1] = (uint16_t)strands[s].node;
        }
      n++;
    }
    const int p = par[dyn[j]];
    f[4] = (uint16_t)(p >= 0 ? dynj[p] : 0xFFFF);
  }
  if (P.npub > 0xFFFF || nt + 1 + P.nd > 0xFFFF || (int64_t)G * C * T + P.nd > INT32_MAX) {
    why = "too large";
    return false;
  }
  return true;
}

// The kernel's phases in its order, with arrays in place of registers and LDS.
void resident_solve_host(const ResPlanHost& P, const double* b, const double* dyn_diag, double* x) {
  constexpr int C = kResC;
  const int G = P.G, T = P.T, nt = P.nt;
  const size_t U = (size_t)G * T;
  std::vector<double> r(U * C, 0.0), rr(U * C, 0.0), below(U, 0.0), xin(U, 0.0);
  for (int i = 0; i < P.N; i++)
    if (P.slot[i] < (int64_t)U * C) r[P.slot[i]] = b[i];
  auto uco = [&](int a, size_t u) { return P.uco[(size_t)a * U + u]; };
  std::vector<double> pub(P.npub, 0.0), dO(nt + 1, 0.0), din(nt + 1, 0.0), dX(nt + 1 + P.nd, 0.0);
  std::vector<std::vector<double>> X(G), In(G);
  for (int g = 0; g < G; g++) {
    const int np = P.ginfo[4 * g], nh = P.ginfo[4 * g + 1];
    std::vector<double> o(T, 0.0), O(T + 1, 0.0);
    In[g].assign(T, 0.0);
    X[g].assign(T + 1, 0.0);
    for (int t = 0; t < T; t++) {
      auto at = [&](int k) { return ((size_t)g * C + k) * T + t; };
      double acc = r[at(C - 1)];
      for (int k = C - 2; k >= 0; k--) acc = P.F[at(k + 1)] * acc + r[at(k)];
      o[t] = P.F[at(0)] * acc;
    }
    auto piece = [&](int t) { return (int)(P.uinf[3 * ((size_t)g * T + t)] & 0x3FF); };
    auto pos = [&](int t) { return (int)((P.uinf[3 * ((size_t)g * T + t)] >> 10) & 63); };
    auto len = [&](int t) { return (int)((P.uinf[3 * ((size_t)g * T + t)] >> 16) & 127); };
    for (int t = T - 1; t >= 0; t--) {
      if (piece(t) == kResNone) continue;
      if (pos(t) + 1 < len(t)) {
        below[(size_t)g * T + t] = o[t + 1];
        o[t] += uco(kUZ, (size_t)g * T + t) * o[t + 1];
      }
      if (pos(t) == 0) O[piece(t)] = o[t];
    }
    for (int h = 1; h < nh; h++)
      for (int p = 0; p < np; p++) {
        const uint16_t* f = &P.pinf[8 * ((size_t)g * T + p)];
        if (f[3] != h) continue;
        In[g][p] = O[f[0]] + O[f[1]];
        O[p] += P.pz[(size_t)g * T + p] * In[g][p];
      }
    std::vector<double> q(T, 0.0), scan(T, 0.0);
    for (int t = 0; t < T; t++) {
      auto at = [&](int k) { return ((size_t)g * C + k) * T + t; };
      const size_t u = (size_t)g * T + t;
      double acc = piece(t) == kResNone ? 0.0 : below[u] + uco(kUBelow, u) * In[g][piece(t)];
      acc += r[at(C - 1)];
      rr[at(C - 1)] = acc;
      for (int k = C - 2; k >= 0; k--) rr[at(k)] = acc = P.F[at(k + 1)] * acc + r[at(k)];
      double v = P.I[at(0)] * rr[at(0)];
      for (int k = 1; k < C; k++) v = P.F[at(k)] * v + P.I[at(k)] * rr[at(k)];
      q[t] = v;
      if (piece(t) == kResNone) continue;
      if (pos(t) > 0) {
        scan[t] = q[t - 1];
        q[t] += uco(kUZ, u) * q[t - 1];
      }
      if (pos(t) + 1 == len(t)) X[g][piece(t)] = q[t];
    }
    for (int p = 0; p < np; p++) {  // by descending height
      const uint16_t* f = &P.pinf[8 * ((size_t)g * T + p)];
      X[g][p] += P.pz[(size_t)g * T + p] * X[g][f[2]];
      if (f[4]) pub[f[4]] = O[p];
      if (f[5]) pub[f[5]] = X[g][p];
    }
    for (int t = 0; t < T; t++) {
      const size_t u = (size_t)g * T + t;
      if (piece(t) == kResNone) continue;
      xin[u] = scan[t] + uco(kUAbove, u) * X[g][P.uinf[3 * u + 2] >> 16];
    }
  }
  for (int j = 0; j < nt; j++) {
    const uint16_t* f = &P.tinf[6 * (size_t)j];
    din[j] = (pub[f[0]] + dO[f[1]]) + (pub[f[2]] + dO[f[3]]);
    dO[j] = P.tz[j] * din[j];
  }
  std::vector<double> dd(P.nd), dr(P.nd);
  for (int j = 0; j < P.nd; j++) {
    const uint16_t* f = &P.dinf[6 * (size_t)j];
    dd[j] = dyn_diag[j] - P.dyn_s[j];
    dr[j] = b[P.dyn_row[j]] + (pub[f[0]] + dO[f[1]]) + (pub[f[2]] + dO[f[3]]);
  }
  for (int j = 0; j < P.nd; j++) {
    const int p = P.dinf[6 * (size_t)j + 4];
    if (p == 0xFFFF) continue;
    const double f = P.dyn_u[j] / dd[j];
    dd[p] -= f * P.dyn_u[j];
    dr[p] -= f * dr[j];
  }
  for (int j = P.nd - 1; j >= 0; j--) {
    const int p = P.dinf[6 * (size_t)j + 4];
    dX[nt + 1 + j] = (dr[j] - (p == 0xFFFF ? 0.0 : P.dyn_u[j] * dX[nt + 1 + p])) / dd[j];
    x[P.dyn_row[j]] = dX[nt + 1 + j];
  }
  for (int j = nt - 1; j >= 0; j--) {
    const uint16_t* f = &P.tinf[6 * (size_t)j];
    dX[j] = P.te[j] * din[j] + P.tz[j] * (dX[f[4]] + pub[f[5]]);
  }
  std::vector<double> xs(U * C, 0.0);
  for (int g = 0; g < G; g++)
    for (int t = 0; t < T; t++) {
      auto at = [&](int k) { return ((size_t)g * C + k) * T + t; };
      const size_t u = (size_t)g * T + t;
      const uint32_t w1 = P.uinf[3 * u + 1], w2 = P.uinf[3 * u + 2];
      const double di = din[w2 & 0xFFFF];
      const double xu = xin[u] + uco(kUCum, u) * (dX[w1 & 0xFFFF] + pub[w1 >> 16]) +
                        uco(kUEin, u) * di;
      double acc = uco(kUBin, u) * di;
      for (int k = C - 1; k >= 0; k--) {
        rr[at(k)] += acc;
        acc *= P.F[at(k)];
      }
      double v = P.F[at(0)] * xu + P.I[at(0)] * rr[at(0)];
      xs[at(0)] = v;
      for (int k = 1; k < C; k++) xs[at(k)] = v = P.F[at(k)] * v + P.I[at(k)] * rr[at(k)];
    }
  for (int i = 0; i < P.N; i++)
    if (P.slot[i] < (int64_t)U * C) x[i] = xs[P.slot[i]];
}

}  // namespace nrt

extern "C" int nrt_test_resident_solve_host(int N, const int32_t* rowptr, const int32_t* col,
                                            const double* val, const double* b,
                                            const int32_t* hh_row, int nhh, int T, double* x,
                                            int32_t* info, char* why, int why_len) {
  using namespace nrt;
  std::vector<int32_t> par(N, -1), hh(hh_row, hh_row + nhh);
  std::vector<double> D(N, 0), U(N, 0), W(N, 0);
  for (int i = 0; i < N; i++)
    for (int k = rowptr[i]; k < rowptr[i + 1]; k++) {
      if (col[k] == i) D[i] = val[k];
      else if (col[k] < i) {
        par[i] = col[k];
        U[i] = val[k];
      }
    }
  for (int i = 0; i < N; i++)
    for (int k = rowptr[i]; k < rowptr[i + 1]; k++)
      if (col[k] > i) {
        if (par[col[k]] != i) return 4;
        W[col[k]] = val[k];
      }
  ResPlanHost P;
  std::string s;
  const bool ok = build_resident_plan(N, par, D, U, W, hh, T, P, s);
  if (why && why_len > 0) {
    std::strncpy(why, s.c_str(), (size_t)why_len - 1);
    why[why_len - 1] = 0;
  }
  if (!ok) return 7;
  std::vector<double> dd(P.nd);
  for (int j = 0; j < P.nd; j++) dd[j] = D[P.dyn_row[j]];
  resident_solve_host(P, b, dd.data(), x);
  int nh = 0, np = 0;
  for (int g = 0; g < P.G; g++) {
    nh = std::max(nh, P.ginfo[4 * g + 1]);
    np = std::max(np, P.ginfo[4 * g]);
  }
  const int32_t out[8] = {P.G, P.nt, P.nth, P.npub, P.rounds, nh, np, P.nd};
  if (info) std::memcpy(info, out, sizeof(out));
  return 0;
}
