// stmtdesc.hpp -- the descriptor a round kernel is generated from (or interprets), and its limits.
#pragma once

namespace exh {

constexpr int MAXT = 16;    // tables plus linear forms per statement
constexpr int MAXV = 8;     // linear forms per statement
constexpr int MAXVT = 4;    // tables per linear form
constexpr int MAXG = 16;    // table groups per statement
constexpr int MAXDEG = 6;   // tables per group
constexpr int MAXEV = 6;    // evaluation points per group
constexpr int MAXTERMS = 4; // groups that share accumulators
constexpr int MAXACC = 36;  // accumulators (group, point) per statement
constexpr int MAXX = 7;     // largest evaluation point
constexpr int BLOCK = 256;  // threads per workgroup

// A statement as the kernels see it: G groups, group g the product of the deg[g] factors tab[g][..],
// evaluated at the nev[g] points ev[g][..]; accumulators are numbered group by group, point by point, a group that
// follows another (lead) having none of its own.
// Factor t < T is table t; factor T + v is the linear form sum_k vcoef[v][k] * table vtab[v][k] + vconst[v]
// (vcoef canonical and, for the kernels' products, in Montgomery form in vcoefm).
struct StmtDesc {
  int T, G, nacc, maxx;
  int deg[MAXG];
  int tab[MAXG][MAXDEG];
  int nev[MAXG];
  int ev[MAXG][MAXEV];
  int NV;
  int vn[MAXV];
  int vtab[MAXV][MAXVT];
  unsigned vcoef[MAXV][MAXVT], vcoefm[MAXV][MAXVT];
  unsigned vconst[MAXV];
  // the first group with group g's accumulators (g itself, or one whose products g's are added to: at most MAXTERMS groups
  // of one coefficient and degree, one after the other), and the first of those accumulators
  int lead[MAXG];
  int acc[MAXG];
};

#if defined(__HIPCC__)
#define EXH_DESC_FN __host__ __device__
#else
#define EXH_DESC_FN
#endif

// no group behind g shares g's accumulators (those that do follow one another)
template <class Desc>
EXH_DESC_FN constexpr bool group_is_last(const Desc &d, int g) {
  return !(g + 1 < d.G && g + 1 < MAXG && d.lead[g + 1 < MAXG ? g + 1 : g] == d.lead[g]);
}
// the most groups that share an accumulator
template <class Desc>
EXH_DESC_FN constexpr int desc_terms(const Desc &d) {
  int m = 1;
  for (int g = 0; g < d.G; g++) {
    int n = 0;
    for (int h = g; h < d.G; h++) n += d.lead[h] == g ? 1 : 0;
    m = n > m ? n : m;
  }
  return m;
}
// the largest number of factors in a group
template <class Desc>
EXH_DESC_FN constexpr int desc_maxdeg(const Desc &d) {
  int m = 1;
  for (int g = 0; g < d.G; g++) m = d.deg[g] > m ? d.deg[g] : m;
  return m;
}

// ---- the slots of the base-field sweep that serves rounds 0 and 1 (the kernels and their generator agree here)
// the index of X among group g's evaluation points, or -1
template <class Desc>
EXH_DESC_FN constexpr int ev_index(const Desc &d, int g, int x) {
  int at = -1;
  for (int e = 0; e < MAXEV; e++)
    if (e < d.nev[g] && d.ev[g][e] == x) at = e;
  return at;
}
// per group: nev * (deg + 1) slots of round 1, then nev extras unless X = 1 is an evaluation point anyway; a group that
// follows another has none of its own
template <class Desc>
EXH_DESC_FN constexpr int group_slots(const Desc &d, int g) {
  return d.lead[g] != g ? 0 : d.nev[g] * (d.deg[g] + 1) + (ev_index(d, g, 1) < 0 ? d.nev[g] : 0);
}
template <class Desc>
EXH_DESC_FN constexpr int node_slots(const Desc &d) {
  int n = 0;
  for (int g = 0; g < d.G; g++) n += group_slots(d, g);
  return n;
}

// The pairs of factors that the sweep takes as quadratics, where a row of slots costs fewer products that way and their
// values stay small: one of three factors, two of four, in the first groups that have them (each is eighteen registers).
constexpr int MAXQUADS = 4;
template <class Desc>
EXH_DESC_FN constexpr int group_quads(const Desc &d, int g) {
  return d.maxx > 4 ? 0 : d.deg[g] == 4 ? 2 : d.deg[g] == 3 ? 1 : 0;
}
// those of group g's that are taken, and the first one's number
template <class Desc>
EXH_DESC_FN constexpr int first_quad(const Desc &d, int g) {
  int n = 0;
  for (int h = 0; h < g; h++) n += n + group_quads(d, h) <= MAXQUADS ? group_quads(d, h) : 0;
  return n;
}
template <class Desc>
EXH_DESC_FN constexpr int sweep_quads(const Desc &d, int g) {
  return first_quad(d, g) + group_quads(d, g) <= MAXQUADS ? group_quads(d, g) : 0;
}

// the launches per round of the base-field sweep for degree D and the slots each takes: the slots are split
// evenly over launches of at most NODES_CAP4 (F_p^4) or NODES_CAP8 (F_p^8) slots, a slot taking D registers of sums; no
// launches when the slot sums do not fit the accumulators' buffers.  A launch repeats the tables' part of the work, so that at
// F_p^4 one takes all slots there can be.  Four tables of 2^24, one launch and two, us: 24 slots 106 and 144, 32 slots 106 and
// 152; eight tables of 2^22, 32 slots, 48 and 60.  At F_p^8 24 slots have been measured (nodes_kernel), more have not.
constexpr int NODES_CAP4 = MAXACC, NODES_CAP8 = 24;
template <class Desc>
EXH_DESC_FN constexpr int nodes_slots_per_pass(const Desc &d, int D) {
  int slots = node_slots(d), cap = D == 4 ? NODES_CAP4 : NODES_CAP8, passes = (slots + cap - 1) / cap;
  return (slots + passes - 1) / passes;
}
// Wavefronts a SIMD: two where 256 registers hold what a lane has of a launch's slots (D sums and a word of digits each), its
// tables (eight words fetched ahead each), their lines and linear forms' (twelve) and its quadratics.  Tables of 2^24, us of the
// sweep by one wavefront a SIMD and by two (the words by this count): F_p^8, three tables, 15 slots 92 and 83 (213), 19 slots
// 95 and 85 (249), 23 slots 103 and 193 (285); four tables, twice 16 slots 185 and 208 (260), 24 slots 123 and 284 (336);
// F_p^4, four tables, 32 slots 107 and 161 (276); twelve tables of 2^20, 8 slots, 35 and 43 (280).
template <class Desc>
EXH_DESC_FN constexpr int sweep_waves(const Desc &d, int D, int slots) {
  int words = slots * (D + 1) + 8 * d.T + 12 * (d.T + d.NV);
  for (int g = 0; g < d.G; g++) words += 18 * sweep_quads(d, g);
  return words > 256 ? 1 : 2;
}
template <class Desc>
EXH_DESC_FN constexpr int nodes_launches(const Desc &d, int D) {
  int slots = node_slots(d), cap = D == 4 ? NODES_CAP4 : NODES_CAP8;
  return (slots + cap - 1) / cap;
}

}  // namespace exh
