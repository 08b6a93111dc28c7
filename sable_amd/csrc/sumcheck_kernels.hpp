// sumcheck_kernels.hpp -- the sumcheck prover's round kernel for gfx950, generated per statement.
//
// One launch does, for every pair i of the tables being summed,
//   [FOLD]  bind the previous round's variable: read four entries per table, write the two folded
//           entries lo + r (hi - lo) (src/sumcheck.lisp:84-104), and use them as the pair (or bind two
//           or three variables of the base tables at once, src/sumcheck.lisp:496-510);
//   sums    for every group g of the statement (a product of tables) and each of its evaluation
//           points X:  acc[g, X] += LOW[l] * prod_{t in g} line_t(X),  line_t(X) = lo + X (hi - lo),
//           i = h |LOW| + l  (src/sumcheck.lisp:230-257), in lazily reduced 64-bit accumulators;
//   then reduces the accumulators over the workgroup (cross-lane, then LDS), multiplies by HIGH[h]
//   and writes one partial per workgroup.  A second small kernel adds the partials.
//
// The statement is a compile-time descriptor (StmtDesc) when the kernel was generated for it, or a
// run-time one interpreted by the same code (the fallback for statements without a generated kernel).
// Tables, weights and outputs are canonical residues; the sums come out scaled by a power of 1/R
// (R = 2^32) that the host removes: a group of degree d carries R^-d.
#pragma once
// (a run-time compilation of these kernels has the runtime's declarations built in and no host headers)
#if !defined(__HIPCC_RTC__)
#include <hip/hip_runtime.h>

#include <stddef.h>
#include <type_traits>
#endif

#include "dev_transcript.hpp"
#include "field.hpp"
#include "stmtdesc.hpp"

namespace exh {

// StmtDesc and the limits MAXT, MAXG, ... come from stmtdesc.hpp
constexpr int MAXROUNDS = 48;  // rounds of one device-driven sumcheck (a count of them fits six bits)
constexpr int MAXPTS = 7;      // wire points of a device-driven round message
constexpr int MAXTAIL = 16;    // rounds the tail kernel can take
constexpr int OWN_VARS = 10;   // variables behind the first of a session whose one launch builds its weight tables
// A round's LOW table takes all variables behind the round's when they are no more than these, and HIGH is one entry then:
// what the heap of such a session's weights stands on.
constexpr int LOW_VARS = 13;
static_assert(OWN_VARS <= LOW_VARS, "the weights that a session's one launch builds have one HIGH entry");

// The control block of a device-driven sumcheck, in device memory: the transcript state, the current
// fold challenge, the launch's completion counter and the logs the host reads back at the end.
struct Ctrl {
  DevB3S tr;
  uint32_t r_mont[8];
  uint32_t round;    // rounds completed
  uint32_t gave_up;  // set by a workgroup of a grid launch whose wait for the others ran out: the proof is void
  uint32_t pad[2];
  uint32_t msg[MAXROUNDS][MAXPTS * 8];
  uint32_t chal[MAXROUNDS][8];
  uint32_t finals[MAXT * 8];  // entry 0 of every table once a single entry is left
};
template <int D>
struct RoundArgs {
  const uint32_t *in[MAXT];  // the tables read: 4 entries per pair when folding, else 2
  uint32_t *out[MAXT];       // folded tables written (after a fold; null after two or three at once: only the sums)
  const uint32_t *low;       // |LOW| = 2^low_bits EXTs
  const uint32_t *high;      // n_high EXTs
  uint32_t *partials;        // [gridDim.x][nacc][D]
  uint64_t n_pairs;          // pairs summed (after the fold)
  uint32_t low_bits;
  uint32_t pairs_per_thread;
  uint32_t deferred;         // every workgroup's pairs share one h: HIGH[h] applied once per workgroup
  uint32_t do_sums;
  uint32_t r_mont[D];        // the fold challenge, times R (host-driven rounds)
  Ctrl *ctrl;                // device-driven rounds: the fold challenge is read from here (else null)
  uint32_t pstride;          // words per workgroup partial (a power of two >= nacc * D)
  // device-driven rounds: the round's sums meet in counted totals and the last workgroup to arrive sends the
  // message and draws the challenge itself (see RoundTotals); totals null: one partial row per workgroup
  unsigned long long *totals;  // [groups][pstride], zero before the launch
  uint32_t *arrivals;          // workgroups that have added their sums, zero before the launch
  uint32_t groups, points, spin_limit;
  const uint32_t *mtilde, *c0;  // the round's message map and constant terms
  const uint32_t *consts;       // a statement in direct form: its constant slots (EXTs, Montgomery form)
};

// How the workgroups of a streaming launch finish a round without another launch.  Every workgroup adds its sums
// into the totals of its group (workgroup w: group w % groups) with integer atomics that also count the
// contribution in the word's top 16 bits, then takes a ticket; the workgroup with the last ticket polls the words
// until each carries its group's full count -- the data travels inside the atomics, so no fence is needed and
// nobody reads memory another workgroup wrote with plain stores -- and goes on to the message, the transcript step
// and the next challenge, which the next launch reads from the control block.
struct RoundTotals {
  unsigned long long *totals;
  uint32_t *arrivals;
  uint32_t groups, pstride, spin_limit;
};
constexpr int TOTALS_POLLS = 8;  // words a thread of the elected workgroup polls: groups * width <= 8 * BLOCK

// The rounds below 2^18 pairs, with the tables resident in LDS: no global memory round trip separates a
// round's sums, its transcript step and its fold.  With one workgroup (the last rounds) everything
// stays on one compute unit; with a grid (the rounds before them) every workgroup keeps a contiguous
// slice of every table, the round's sums meet in global totals (integer atomics that count their
// contributions), and every workgroup runs the same transcript step, so each knows the next challenge.
// The grid must be resident at once: the host launches at most one workgroup per compute unit.
constexpr uint32_t TAIL_LDS_BYTES = 32768;        // LDS given to the tables of the one-workgroup launch
constexpr uint32_t SLICE_LDS_BYTES = 128 * 1024;  // and to a workgroup's slices in the grid launch
template <int D>
struct TailArgs {
  const uint32_t *in[MAXT];  // tables of `entries` entries each; base (stride 1) when in_base
  uint32_t *out;             // where the folded tables go: table t at t * final_entries * D
  const uint32_t *weights;   // base of the weight tables
  uint64_t low_off[MAXTAIL], high_off[MAXTAIL];  // in EXTs, per round
  uint32_t low_bits[MAXTAIL];
  uint32_t entries;          // per table, over all workgroups
  uint32_t in_base;
  uint32_t first_fold;       // fold by ctrl's challenge while loading
  uint32_t rounds;           // rounds summed here; a fold follows each
  uint32_t first_round;      // index of the first of them
  uint32_t capacity;         // entries per table in a workgroup's LDS
  uint32_t lds_bytes;        // T * capacity * D * 4
  uint32_t points;
  Ctrl *ctrl;
  const uint32_t *mtilde;
  const uint32_t *c0;        // [rounds][points][D]
  unsigned long long *totals;  // grid launch: [rounds][groups][pstride] counted sums, zeroed by the host
  uint32_t pstride;
  uint32_t groups;           // workgroup w adds into group w % groups
  uint32_t spin_limit;       // polls of a total before giving up
  // the last launch of a device-driven loop (one workgroup): it ends by copying the control block into pinned
  // host memory and raising host_log[host_flag_at] to host_seq, so that the host needs neither a copy nor a wait
  // on the stream to read the logs (null: it does both)
  uint32_t *host_log;
  uint32_t host_flag_at, host_seq;
  const uint32_t *consts;  // a statement in direct form: its constant slots (EXTs, Montgomery form)
  // A session whose every round runs in this one launch builds its weight tables itself (`own`), in LDS behind the
  // tables (no set-up launch): `factors` holds (r_v R, (1 - r_v) R) for the eq point's n_vars <= OWN_VARS + 1 variables.
  // They are one heap of 2^n_vars entries.  Entries [2^s, 2^(s + 1)) are the products over the last s variables, and the LOW
  // table of the round before those; low_bits is s in that round, so that its HIGH table is one entry, and entry 0, which is
  // one, serves every round as such.  Without an eq point (factors null) all entries are ones; with block weights (block_high)
  // the HIGH entries are those, read from `weights`.
  const uint32_t *factors;
  uint32_t n_vars, own, block_high;
  uint32_t valid;  // entries that the tables in memory hold, zeros beyond them (0: all of them; unfolded extension tables)
  // ... and brings its constants itself: staged_words words from pinned host memory to staged_dst, where the control block,
  // the message map, the factors and the block weights are then read (null: they are there already)
  const uint32_t *staged;
  uint32_t *staged_dst;
  uint32_t staged_words;
};

template <int D>
__device__ __forceinline__ Ext<D> load_ext(const uint32_t *p) {
  Ext<D> e;
  if constexpr (D == 4) {
    uint4 v = *reinterpret_cast<const uint4 *>(p);
    e.c[0] = v.x, e.c[1] = v.y, e.c[2] = v.z, e.c[3] = v.w;
  } else {
    uint4 v = *reinterpret_cast<const uint4 *>(p), u = *reinterpret_cast<const uint4 *>(p + 4);
    e.c[0] = v.x, e.c[1] = v.y, e.c[2] = v.z, e.c[3] = v.w;
    e.c[4] = u.x, e.c[5] = u.y, e.c[6] = u.z, e.c[7] = u.w;
  }
  return e;
}
template <int D>
__device__ __forceinline__ void store_ext(uint32_t *p, const Ext<D> &e) {
  *reinterpret_cast<uint4 *>(p) = make_uint4(e.c[0], e.c[1], e.c[2], e.c[3]);
  if constexpr (D == 8) *reinterpret_cast<uint4 *>(p + 4) = make_uint4(e.c[4], e.c[5], e.c[6], e.c[7]);
}

// lo + r (hi - lo) for base values: r_mont * (hi - lo) is exact, lo joins coordinate 0
template <int D>
__device__ __forceinline__ Ext<D> fold_base(uint32_t lo, uint32_t hi, const Ext<D> &r_mont) {
  Ext<D> o = ext_scale_mont<D>(r_mont, fsub(hi, lo));
  o.c[0] = fadd(o.c[0], lo);
  return o;
}
template <int D>
__device__ __forceinline__ Ext<D> fold_ext(const Ext<D> &lo, const Ext<D> &hi, const Ext<D> &r_mont) {
  // r is the second operand: its tripled wrap coefficients are the same for every entry of the launch
  return ext_add<D>(lo, ext_mul_mont<D>(ext_sub<D>(hi, lo), r_mont));
}

// ---- the per-pair work: all groups at all their points.  V is uint32_t (base mode) or Ext<D>.
template <int D>
__device__ __forceinline__ uint32_t v_add(uint32_t a, uint32_t b) { return fadd(a, b); }
template <int D>
__device__ __forceinline__ Ext<D> v_add(const Ext<D> &a, const Ext<D> &b) { return ext_add<D>(a, b); }
template <int D>
__device__ __forceinline__ uint32_t v_sub(uint32_t a, uint32_t b) { return fsub(a, b); }
template <int D>
__device__ __forceinline__ Ext<D> v_sub(const Ext<D> &a, const Ext<D> &b) { return ext_sub<D>(a, b); }
template <int D>
__device__ __forceinline__ uint32_t v_mul(uint32_t a, uint32_t b) { return mont_mul(a, b); }
template <int D>
__device__ __forceinline__ Ext<D> v_mul(const Ext<D> &a, const Ext<D> &b) { return ext_mul_mont<D>(a, b); }
template <int D>
__device__ __forceinline__ void v_weigh(Acc96 *acc, const Ext<D> &w, uint32_t v) { ext_scale_acc<D>(acc, w, v); }

// integer multiples and integer offsets, for the linear forms
template <int D>
__device__ __forceinline__ uint32_t v_scale(uint32_t a, uint32_t c, uint32_t c_mont) {
  return c == 1 ? a : c == P - 1 ? fneg(a) : mont_mul(a, c_mont);
}
template <int D>
__device__ __forceinline__ Ext<D> v_scale(const Ext<D> &a, uint32_t c, uint32_t c_mont) {
  Ext<D> o;
#pragma unroll
  for (int k = 0; k < D; k++) o.c[k] = v_scale<D>(a.c[k], c, c_mont);
  return o;
}
template <int D>
__device__ __forceinline__ uint32_t v_offset(uint32_t a, uint32_t k) { return fadd(a, k); }
template <int D>
__device__ __forceinline__ Ext<D> v_offset(Ext<D> a, uint32_t k) {
  a.c[0] = fadd(a.c[0], k);
  return a;
}

// helpers of the weighted first factor (never reached with base values)
template <int D, class V>
__device__ __forceinline__ V v_of(const Ext<D> &w) {
  if constexpr (std::is_same<V, uint32_t>::value)
    return w.c[0];
  else
    return w;
}
template <int D>
__device__ __forceinline__ void v_mul_acc(Acc96 *acc, uint32_t a, uint32_t b) { acc_mad(acc[0], a, b); }
template <int D>
__device__ __forceinline__ void v_mul_acc(AccLazy *acc, const Ext<D> &a, const Ext<D> &b) { ext_mul_acc<D>(acc, a, b); }

// A statement too wide for accumulators per table group comes in direct form: its descriptor's type carries an
// evaluator of the written form (generated code) and a flag, and the accumulators are the wire points.
template <class T>
struct is_direct {
  template <class U>
  static char test(decltype(U::direct) *);
  template <class U>
  static long test(...);
  static constexpr bool value = sizeof(test<T>(nullptr)) == sizeof(char);
};

// The accumulators of a pair's words: sums of products of extension elements, or of a weight and a base value (whose two
// instructions a word the 96-bit sum is cheaper for); a statement in direct form evaluates in the extension either way.
template <class V, class Desc>
struct AccOf {
  typedef typename std::conditional<std::is_same<V, uint32_t>::value && !is_direct<Desc>::value, Acc96, AccLazy>::type type;
};

// The pair's contribution for a statement in direct form: the tables' lines in Montgomery form (so that sums and
// products of any shape stay in one scale), the form evaluated at each wire point X = 0, 2, 3, ..., and w times
// that value added to the point's accumulator.  The loop over the points is kept a loop: the evaluator is long,
// and one copy of it per kernel keeps compile times and code size in hand; the accumulators stay in registers
// because each is named by a constant inside the switch.
template <int D, class V, class Desc, int PARTS, int PART>
__device__ __forceinline__ void accumulate_direct(const Desc &d, const V *lo, const V *hi, const Ext<D> &w,
                                                  AccLazy (*acc)[D], const uint32_t *kc) {
  Ext<D> at0[MAXT], slope[MAXT];
#pragma unroll
  for (int t = 0; t < MAXT; t++)
    if (t < d.T) {
      if constexpr (std::is_same<V, uint32_t>::value) {
        at0[t] = ext_lift<D>(mont_mul(lo[t], R2));
        slope[t] = ext_lift<D>(mont_mul(fsub(hi[t], lo[t]), R2));
      } else {
        at0[t] = ext_scale_mont<D>(lo[t], R2);
        slope[t] = ext_scale_mont<D>(ext_sub<D>(hi[t], lo[t]), R2);
      }
    }
#pragma unroll 1
  for (int k = PART; k < d.nacc; k += PARTS) {
    const uint32_t x_mont = mont_mul(k == 0 ? 0u : (uint32_t)k + 1u, R2);
    Ext<D> t[MAXT];
#pragma unroll
    for (int i = 0; i < MAXT; i++)
      if (i < d.T) t[i] = ext_add<D>(at0[i], ext_scale_mont<D>(slope[i], x_mont));
    const Ext<D> f = Desc::template eval<D>(t, kc);
    switch (k) {
      case 0: ext_mul_acc<D>(acc[0], f, w); break;
      case 1: ext_mul_acc<D>(acc[1], f, w); break;
      case 2: ext_mul_acc<D>(acc[2], f, w); break;
      case 3: ext_mul_acc<D>(acc[3], f, w); break;
      case 4: ext_mul_acc<D>(acc[4], f, w); break;
      default: ext_mul_acc<D>(acc[5], f, w); break;
    }
  }
}

// With PARTS > 1 only the accumulators a with a % PARTS == PART are computed (a compile-time constant: with the
// part as a run-time value, uniform as it is, the compiler folds the parts' branches into one path that indexes
// the accumulators by it, and they move from registers to scratch memory): the last rounds, with a pair per lane
// and lanes to spare, give each of a workgroup's wavefronts a share of a pair's accumulators, so that a round
// waits for a quarter of the products.
template <int D, class V, class Desc, int PARTS, int PART, class Acc>
__device__ __forceinline__ void accumulate_groups(const Desc &d, const V *lo, const V *hi, const Ext<D> &w, Acc (*acc)[D]) {
  V cur[MAXT], slope[MAXT];
#pragma unroll
  for (int t = 0; t < MAXT; t++)
    if (t < d.T) {
      cur[t] = lo[t];
      slope[t] = v_sub<D>(hi[t], lo[t]);
    }
  // the linear forms are lines too: value at 0 from the tables' values at 0 plus the offset, slope
  // from the tables' slopes
#pragma unroll
  for (int v = 0; v < MAXV; v++)
    if (v < d.NV) {
      V c0 = v_scale<D>(cur[d.vtab[v][0]], d.vcoef[v][0], d.vcoefm[v][0]);
      V s0 = v_scale<D>(slope[d.vtab[v][0]], d.vcoef[v][0], d.vcoefm[v][0]);
#pragma unroll
      for (int k = 1; k < MAXVT; k++)
        if (k < d.vn[v]) {
          c0 = v_add<D>(c0, v_scale<D>(cur[d.vtab[v][k]], d.vcoef[v][k], d.vcoefm[v][k]));
          s0 = v_add<D>(s0, v_scale<D>(slope[d.vtab[v][k]], d.vcoef[v][k], d.vcoefm[v][k]));
        }
      cur[d.T + v] = v_offset<D>(c0, d.vconst[v]);
      slope[d.T + v] = s0;
    }
  // A group evaluated at three points or more carries the weight on its first factor: w * factor is a
  // line too (two products per pair), and each point then needs one product fewer.  Extension values
  // only: in the base field the products are cheap and the weight is the one extension operation.
  constexpr bool EXT = !std::is_same<V, uint32_t>::value;
  V wcur[MAXG], wslope[MAXG];
#pragma unroll
  for (int g = 0; g < MAXG; g++)
    if (g < d.G && EXT && d.nev[g] >= 3 && d.deg[g] >= 2) {
      wcur[g] = v_mul<D>(cur[d.tab[g][0]], v_of<D, V>(w));
      wslope[g] = v_mul<D>(slope[d.tab[g][0]], v_of<D, V>(w));
    }
#pragma unroll
  for (int x = 0; x <= MAXX; x++) {
    if (x <= d.maxx) {
      if (x >= 1) {
#pragma unroll
        for (int t = 0; t < MAXT; t++) {
          if (x == 1 && t < d.T)
            cur[t] = hi[t];
          else if (t < d.T + d.NV)
            cur[t] = v_add<D>(cur[t], slope[t]);
        }
#pragma unroll
        for (int g = 0; g < MAXG; g++)
          if (g < d.G && EXT && d.nev[g] >= 3 && d.deg[g] >= 2) wcur[g] = v_add<D>(wcur[g], wslope[g]);
      }
      AccLazy sum[D];  // (the unreduced sum of the products of groups that share an accumulator, which follow one another)
      V total;
#pragma unroll
      for (int g = 0; g < MAXG; g++) {
        if (g < d.G) {
          const bool pre = EXT && d.nev[g] >= 3 && d.deg[g] >= 2, first = d.lead[g] == g, last = group_is_last(d, g);
          const bool shared = EXT && !pre && d.deg[g] >= 2 && !(first && last);
#pragma unroll
          for (int k = 0; k < MAXEV; k++) {
            if (k < d.nev[g]) {
              const int a = d.acc[g] + k;
              if (d.ev[g][k] == x && (PARTS == 1 || a % PARTS == PART)) {
                // the product of the factors but the last; the last goes with the accumulation or the sum
                V prod = pre ? wcur[g] : cur[d.tab[g][0]];
#pragma unroll
                for (int j = 1; j < MAXDEG; j++)
                  if (j < d.deg[g] - (pre || shared ? 1 : 0)) prod = v_mul<D>(prod, cur[d.tab[g][j]]);
                if constexpr (EXT) {
                  if (shared) {
                    if (first) {
#pragma unroll
                      for (int c = 0; c < D; c++) acc_zero(sum[c]);
                    }
                    ext_mul_acc<D>(sum, prod, cur[d.tab[g][d.deg[g] - 1]]);
                    if (last) {
#pragma unroll
                      for (int c = 0; c < D; c++) total.c[c] = mont_reduce4(sum[c].v);
                    }
                  } else {
                    total = pre || first ? prod : v_add<D>(total, prod);
                  }
                  if (pre || last) v_mul_acc<D>(acc[a], total, pre ? cur[d.tab[g][d.deg[g] - 1]] : v_of<D, V>(w));
                } else {
                  total = first ? prod : v_add<D>(total, prod);
                  if (last) v_weigh<D>(acc[a], w, total);
                }
              }
            }
          }
        }
      }
    }
  }
}

// A product of four factors, as two products of two: factors 0 and 1 (with the weight on factor 0) and factors 2 and 3 are
// quadratics in X, known from their values at 0 and 1 and their coefficient of X^2 -- a pair costs twelve products where a
// factor at a time takes fourteen (2867 instructions for 3135 at F_p^8), and the first quadratic needs the first tables alone.
// Registers are what it must not cost: with 25 words of it spilled the bind by three took 740 us, 559 with two.
// (`h`: which two)
template <class Desc>
__device__ __forceinline__ bool product_of_four(const Desc &d) {
  return d.G == 1 && d.deg[0] == 4 && d.nev[0] == 4;
}
// the last table that factors 0 and 1 are made of
template <class Desc>
__device__ __forceinline__ int first_half_table(const Desc &d) {
  int last = 0;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int f = d.tab[0][j];
    if (f < d.T) {
      last = f > last ? f : last;
    } else {
#pragma unroll
      for (int k = 0; k < MAXVT; k++)
        if (k < d.vn[f - d.T]) last = d.vtab[f - d.T][k] > last ? d.vtab[f - d.T][k] : last;
    }
  }
  return last;
}
template <int D, class Desc>
__device__ __forceinline__ void factor_line(const Desc &d, int f, const Ext<D> *lo, const Ext<D> *hi, Ext<D> &at0, Ext<D> &slope) {
  at0 = ext_zero<D>(), slope = ext_zero<D>();
#pragma unroll
  for (int t = 0; t < MAXT; t++)
    if (t < d.T && f == t) at0 = lo[t], slope = ext_sub<D>(hi[t], lo[t]);
#pragma unroll
  for (int v = 0; v < MAXV; v++)
    if (v < d.NV && f == d.T + v) {
#pragma unroll
      for (int k = 0; k < MAXVT; k++)
        if (k < d.vn[v]) {
          const int t = d.vtab[v][k];
          const Ext<D> a = v_scale<D>(lo[t], d.vcoef[v][k], d.vcoefm[v][k]);
          const Ext<D> b = v_scale<D>(ext_sub<D>(hi[t], lo[t]), d.vcoef[v][k], d.vcoefm[v][k]);
          at0 = k == 0 ? a : ext_add<D>(at0, a), slope = k == 0 ? b : ext_add<D>(slope, b);
        }
      at0 = v_offset<D>(at0, d.vconst[v]);
    }
}
template <int D>
struct Quadratic {
  Ext<D> at0, at1, square;  // values at 0 and 1, coefficient of X^2
};
template <int D, class Desc>
__device__ __forceinline__ Quadratic<D> quadratic(const Desc &d, int h, const Ext<D> *lo, const Ext<D> *hi, const Ext<D> &w) {
  Ext<D> a, da, b, db;
  factor_line<D>(d, d.tab[0][2 * h], lo, hi, a, da);
  factor_line<D>(d, d.tab[0][2 * h + 1], lo, hi, b, db);
  if (h == 0) a = ext_mul_mont<D>(a, w), da = ext_mul_mont<D>(da, w);
  Quadratic<D> q;
  q.at0 = ext_mul_mont<D>(a, b);
  q.square = ext_mul_mont<D>(da, db);
  q.at1 = ext_mul_mont<D>(ext_add<D>(a, da), ext_add<D>(b, db));
  return q;
}
template <int D, class Desc>
__device__ __forceinline__ void accumulate_quadratics(const Desc &d, const Quadratic<D> &p, const Quadratic<D> &q, AccLazy (*acc)[D]) {
  Ext<D> x = p.at0, y = q.at0, dx = ext_sub<D>(p.at1, p.at0), dy = ext_sub<D>(q.at1, q.at0);
  const Ext<D> ddx = ext_add<D>(p.square, p.square), ddy = ext_add<D>(q.square, q.square);
#pragma unroll
  for (int at = 0; at <= MAXX; at++) {
    if (at <= d.maxx) {
      if (at == 1) {
        x = p.at1, y = q.at1;
      } else if (at > 1) {
        dx = ext_add<D>(dx, ddx), dy = ext_add<D>(dy, ddy);
        x = ext_add<D>(x, dx), y = ext_add<D>(y, dy);
      }
#pragma unroll
      for (int k = 0; k < MAXEV; k++)
        if (k < d.nev[0] && d.ev[0][k] == at) ext_mul_acc<D>(acc[d.acc[0] + k], x, y);
    }
  }
}

template <int D, class V, class Desc, int PARTS = 1, int PART = 0, class Acc>
__device__ __forceinline__ void accumulate_pair(const Desc &d, const V *lo, const V *hi, const Ext<D> &w,
                                                Acc (*acc)[D], const uint32_t *kc = nullptr) {
  if constexpr (is_direct<Desc>::value)
    accumulate_direct<D, V, Desc, PARTS, PART>(d, lo, hi, w, acc, kc);
  else
    accumulate_groups<D, V, Desc, PARTS, PART>(d, lo, hi, w, acc);
}

// A workgroup barrier that orders LDS traffic only: what the threads of a workgroup hand each other in these
// kernels lives in LDS, and a full barrier would also wait for every global access in flight (the weights fetched
// a round ahead, the rows on their way to the host).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// cross-lane sum of a canonical value over the 64 lanes of a wavefront: four DPP butterfly steps inside
// each row of 16 lanes (no LDS traffic), then the four row sums through read-lane
#define EXH_DPP(v, ctrl) ((uint32_t)__builtin_amdgcn_update_dpp(0, (int)(v), (ctrl), 0xf, 0xf, false))
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  v = fadd(v, EXH_DPP(v, 0xB1));   // quad_perm [1,0,3,2]
  v = fadd(v, EXH_DPP(v, 0x4E));   // quad_perm [2,3,0,1]
  v = fadd(v, EXH_DPP(v, 0x141));  // row_half_mirror
  v = fadd(v, EXH_DPP(v, 0x140));  // row_mirror
  uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)v, 0), b = (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)v, 32), d = (uint32_t)__builtin_amdgcn_readlane((int)v, 48);
  return fadd(fadd(a, b), fadd(c, d));
}

// eq((r0, .., r_(F-1)), b) for b < 2^F, F = 2 to 4 (bit k of b goes with r_k), in Montgomery form: the weights that bind
// the first F variables of a base table at once, entry <- sum_b e[b] * T[2^F x + b] (BIND-PREFIX, src/sumcheck.lisp:496-510).
// Of challenges 0 to F - 1 (the last one also lies in ctrl->r_mont), a coefficient a lane, into e in powers of w: every
// workgroup forms them for itself, and as straight code on values that are the same for all lanes the 2 or 6 products run on
// the scalar unit, some 1,200 dependent instructions at D = 8 and F = 2 before a workgroup's first pair.  All threads call.
template <int D, int F>
__device__ __forceinline__ void bind_weights_lds(const Ctrl *ctrl, uint32_t *e) {
  __shared__ uint32_t r[F][2 * D];  // the challenges in powers of w, times R; then their triples
  const uint32_t tid = threadIdx.x, k = tid % D;
  if (tid < (uint32_t)(F * D)) {
    const uint32_t v = to_mont(ctrl->chal[tid / D][brev_bits<D>(k)]);
    r[tid / D][k] = v, r[tid / D][D + k] = times3(v);
    if (tid < (uint32_t)D) {
      const uint32_t one = k == 0 ? R1 : 0u;
      e[D + k] = v, e[k] = fsub(one, v);  // bound by r_0 alone: r_0 and 1 - r_0
    }
  }
#pragma unroll
  for (int f = 1; f < F; f++) {  // e[b + 2^f] = e[b] r_f, e[b] -= that
    __syncthreads();
    uint32_t at = 0, v = 0, rest = 0;
    if (tid < (uint32_t)(D << f)) {
      at = tid / D * D;
      uint64_t t = 0;
#pragma unroll
      for (uint32_t i = 0; i < (uint32_t)D; i++) {
        const uint32_t j = (k - i) & (D - 1);
        if (i >= 4 && i % 2 == 0) t = mont_lazy(t);
        t += (uint64_t)e[at + i] * r[f][i > k ? D + j : j];
      }
      v = mont_reduce4(t), rest = fsub(e[at + k], v);
    }
    __syncthreads();
    if (tid < (uint32_t)(D << f)) e[at + k] = rest, e[(D << f) + at + k] = v;
  }
  __syncthreads();
}
template <int D, int F>
struct BindWeights {
  Ext<D> e[1 << F];
};
// the words end up in scalar registers
template <int D, int F>
__device__ __forceinline__ BindWeights<D, F> bind_weights(const Ctrl *ctrl) {
  __shared__ uint32_t e[(1 << F) * D];
  bind_weights_lds<D, F>(ctrl, e);
  BindWeights<D, F> w;
#pragma unroll
  for (int b = 0; b < 1 << F; b++)
#pragma unroll
    for (int c = 0; c < D; c++) w.e[b].c[c] = (uint32_t)__builtin_amdgcn_readfirstlane((int)e[b * D + brev(c, D)]);
  return w;
}
// sum_b e[b] * v[b], exact: one reduction per coordinate
template <int D, int F>
__device__ __forceinline__ Ext<D> bind(const BindWeights<D, F> &w, const uint32_t *v) {
  Ext<D> o;
#pragma unroll
  for (int c = 0; c < D; c++) {
    uint64_t t = 0;
#pragma unroll
    for (int b = 0; b < 1 << F; b++) {
      if (b >= 4 && b % 2 == 0) t = mont_lazy(t);
      t += (uint64_t)w.e[b].c[c] * v[b];
      if (b >= 4 && b % 2 == 0) keep_sum(t);
    }
    o.c[c] = mont_reduce4(t);
  }
  return o;
}

// ---- folds of extension elements of degree 8 on the matrix cores.  A folded entry's coordinates are fixed combinations, the
// same for every entry of a launch, of the words it comes from: out[c] = sum_k M[c][k] in[k] mod p, of the two entries' 16
// words when an extension table is folded (1 - r and r times the powers of w), of 2^F words when F variables of a base table
// are bound at once.  Both sides are written in signed bytes.  A table word is four digits, in[k] = sum_j v_j 2^(8 j); a
// coefficient is the digits of each of M[c][k] 2^(8 j) mod p; and out[c] is congruent to sum_i 2^(8 i) of its row i's sum,
// over k and j, of digit_i(M[c][k] 2^(8 j)) v_j, an exact 32-bit sum: 32 rows, 32 entries a product.  The left operand is made
// once by a workgroup and stays in registers; the right one is the tables' words as they lie in memory, sixteen bytes a lane;
// what is left to the vector units is two instructions for the digits of a word read and eight to put four digit sums together
// (digit_sums_value), 12 a coordinate of a fold where a product and the subtraction and addition about it are 25.
// Four tables of 2^26, with the quadratics of accumulate_quadratics: the rounds bound by two and by three challenges 973 -> 862
// and 620 -> 559 us (469 where it writes nothing), by four 415, the largest fold round 440 -> 420 (1.6 GB, 3.8 TB/s).
// At F_p^4, where those 25 are 17, the rounds took as long one way as the other: 78.8 and 83.3 us, 62.3 and 62, 48.8 and 48.7.
constexpr uint32_t DIGIT_BIAS = 0x80808080u;
// the word whose bytes are the signed digits of a canonical value
EXH_HD uint32_t signed_digits(uint32_t v) { return (v + DIGIT_BIAS) ^ DIGIT_BIAS; }
#if defined(__HIPCC__)
typedef int digit_sums __attribute__((ext_vector_type(4)));
typedef int digit_sums16 __attribute__((ext_vector_type(16)));
// sum_i 2^(8 i) d_i mod p, canonical, for |d_i| <= 2^20 (64 products of signed bytes): with a = d_0 + 2^8 d_1 and
// b = d_2 + 2^8 d_3 within 2^28.01 the quotient's estimate from b alone leaves less than 0.64 p.
__device__ __forceinline__ uint32_t digit_sums_value(int d0, int d1, int d2, int d3) {
  const int a = d0 + d1 * 256, b = d2 + d3 * 256;
  const int q = (int)(((int64_t)b * 132104 + 0x80000000ll) >> 32);  // b 2^16 / p, rounded: 132104 = rint(2^48 / p)
  const uint32_t r = ((uint32_t)b << 16) + (uint32_t)a - (uint32_t)q * P;
  return umin32(r, r + P);
}

// FOLDS = 1: an extension table folded by one challenge; 2 to 4: base tables bound at once.  A wavefront's 64 pairs go in two
// batches of 32; the results have a lane hold four coordinates of an entry, and exchanges between the lanes' halves bring a
// pair's words to its own lane.
template <int FOLDS>
struct FoldMap {
  static constexpr int WORDS = FOLDS == 1 ? 16 : 1 << FOLDS;  // of memory, per folded entry
  static constexpr int PARTS = WORDS / 4;                     // quads a lane holds of a batch (a pair's 2 WORDS, by two lanes)
  digit_sums op[2];
};
// The map of a launch: of the challenge r_mont (FOLDS = 1), or of challenges 0 to FOLDS - 1.  All threads call.
template <int FOLDS>
__device__ __forceinline__ FoldMap<FOLDS> fold_map(const Ext<8> &r_mont, const Ctrl *ctrl) {
  constexpr int D = 8;
  typedef FoldMap<FOLDS> Map;
  __shared__ uint32_t e[FOLDS == 1 ? D : D << FOLDS];  // the challenge in tower order, or a bind's weights in powers of w
  __shared__ uint4 rows[Map::WORDS * D];               // coordinate c's four rows of word k at k * D + c
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  if constexpr (FOLDS == 1) {
    if (tid == 0) {
#pragma unroll
      for (int q = 0; q < D; q++) e[q] = r_mont.c[q];
    }
    __syncthreads();
  } else {
    bind_weights_lds<D, FOLDS>(ctrl, e);
  }
  if (tid < (uint32_t)(Map::WORDS * D)) {
    const uint32_t k = tid / D, to = brev_bits<D>(tid % D), up = brev_bits<D>(k % D);
    uint32_t v;  // M[c][k] R
    if constexpr (FOLDS == 1) {
      const uint32_t from = brev_bits<D>((to - up) & (D - 1));
      v = e[from];
      if (k < (uint32_t)D) v = fsub(from == 0 ? R1 : 0u, v);
      if (to < up) v = times3(v);
    } else {
      v = e[k * D + to];
    }
    uint32_t dig[4], row[4] = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; j++) dig[j] = signed_digits(mont_mul(v, 1u << (8 * j)));
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) row[i] |= (dig[j] >> (8 * i) & 255u) << (8 * j);
    rows[tid] = make_uint4(row[0], row[1], row[2], row[3]);
  }
  __syncthreads();
  // this lane's row of the left operand is digit i of coordinate c, so that a lane of the result has coordinates 4 g + 0 .. 3
  const uint32_t i = lane & 3, c = 4 * (lane >> 2 & 1) + ((lane & 31) >> 3), g = lane >> 5;
  auto digits = [&](uint32_t k) { return (int)reinterpret_cast<const uint32_t *>(rows)[(k * D + c) * 4 + i]; };
  Map m;
#pragma unroll
  for (int t = 0; t < 4; t++) {
    if constexpr (FOLDS == 2) {  // a product holds the pair: its first half is the first entry's, its second half the other's
      m.op[0][t] = g == 0 ? digits(t) : 0;
      m.op[1][t] = g == 0 ? 0 : digits(t);
    } else {  // an entry's words fill a product, or two
      m.op[0][t] = digits(4 * g + t);
      m.op[1][t] = Map::WORDS == 16 ? digits(8 + 4 * g + t) : 0;
    }
  }
  return m;
}
// the words of a wavefront's pairs base .. base + 63 as the products take them; pairs beyond `last` are `last` again
template <int FOLDS>
__device__ __forceinline__ void fetch_mapped(const uint32_t *in, uint64_t base, uint32_t last, uint4 *raw) {
  typedef FoldMap<FOLDS> Map;
  const uint32_t lane = threadIdx.x & 63, n = lane % 32, g = lane / 32;
  const char *const from = reinterpret_cast<const char *>(in + base * (2 * Map::WORDS));  // (the same for all lanes)
#pragma unroll
  for (int b = 0; b < 2; b++) {
    uint32_t at = umin32(32 * b + n, last) * (8 * Map::WORDS) + 16 * g;
    asm("" : "+v"(at));  // (an offset from a scalar address, not one of many addresses kept in vector registers)
#pragma unroll
    for (int part = 0; part < Map::PARTS; part++)
      raw[b * Map::PARTS + part] = *reinterpret_cast<const uint4 *>(from + at + part * 32);
  }
}
// and the pair of this lane from them
template <int FOLDS>
__device__ __forceinline__ void pair_mapped(const FoldMap<FOLDS> &m, const uint4 *raw, Ext<8> &lo, Ext<8> &hi) {
  auto words = [](const uint4 &q) {
    return digit_sums{(int)signed_digits(q.x), (int)signed_digits(q.y), (int)signed_digits(q.z), (int)signed_digits(q.w)};
  };
  digit_sums16 zero;
#pragma unroll
  for (int q = 0; q < 16; q++) zero[q] = 0;
  uint32_t v[2][2][4];  // [entry][batch][coordinate % 4]
#pragma unroll
  for (int b = 0; b < 2; b++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      digit_sums16 x;
      if constexpr (FoldMap<FOLDS>::WORDS == 16) {
        x = __builtin_amdgcn_mfma_i32_32x32x32_i8(m.op[0], words(raw[4 * b + 2 * h]), zero, 0, 0, 0);
        x = __builtin_amdgcn_mfma_i32_32x32x32_i8(m.op[1], words(raw[4 * b + 2 * h + 1]), x, 0, 0, 0);
      } else {
        x = __builtin_amdgcn_mfma_i32_32x32x32_i8(m.op[FOLDS == 2 ? h : 0], words(raw[FOLDS == 2 ? b : 2 * b + h]), zero, 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < 4; q++) v[h][b][q] = digit_sums_value(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
    }
  // the halves of the lanes hold coordinates 0 to 3 and 4 to 7 of a batch's entries
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const auto s = __builtin_amdgcn_permlane32_swap(v[0][0][q], v[0][1][q], false, false);
    const auto t = __builtin_amdgcn_permlane32_swap(v[1][0][q], v[1][1][q], false, false);
    lo.c[q] = s[0], lo.c[4 + q] = s[1], hi.c[q] = t[0], hi.c[4 + q] = t[1];
  }
}
#endif

// the pair (lo, hi) of every table at pair index i, folding first when FOLD
template <int D, bool IN_BASE, bool FOLD, class V, class Desc>
__device__ __forceinline__ void load_pair(const Desc &d, const uint32_t *const *in, uint32_t *const *out, uint64_t i,
                                          const Ext<D> &r, V *lo, V *hi) {
#pragma unroll
  for (int t = 0; t < MAXT; t++) {
    if (t < d.T) {
      if constexpr (FOLD && IN_BASE) {
        uint4 e = *reinterpret_cast<const uint4 *>(in[t] + 4 * i);
        lo[t] = fold_base<D>(e.x, e.y, r);
        hi[t] = fold_base<D>(e.z, e.w, r);
      } else if constexpr (FOLD) {
        const uint32_t *p = in[t] + 4 * i * D;
        lo[t] = fold_ext<D>(load_ext<D>(p), load_ext<D>(p + D), r);
        hi[t] = fold_ext<D>(load_ext<D>(p + 2 * D), load_ext<D>(p + 3 * D), r);
      } else if constexpr (IN_BASE) {
        uint2 e = *reinterpret_cast<const uint2 *>(in[t] + 2 * i);
        lo[t] = e.x;
        hi[t] = e.y;
      } else {
        const uint32_t *p = in[t] + 2 * i * D;
        lo[t] = load_ext<D>(p);
        hi[t] = load_ext<D>(p + D);
      }
      if constexpr (FOLD) {
        store_ext<D>(out[t] + 2 * i * D, lo[t]);
        store_ext<D>(out[t] + (2 * i + 1) * D, hi[t]);
      }
    }
  }
}

// The same in two steps, so that a table's loads can be issued ahead of their arithmetic: the words as they lie in memory
// (QUADS 16-byte quads per table), then the pair from them.  FOLDS: the folds before the pair, 0 or 1, or 2 or 3 of base
// tables at once by the bind weights.
template <int D, bool IN_BASE, int FOLDS>
constexpr int raw_quads() {
  return IN_BASE ? (FOLDS == 4 ? 8 : FOLDS == 3 ? 4 : FOLDS == 2 ? 2 : 1) : FOLDS == 1 ? D : D / 2;
}
template <int D, bool IN_BASE, int FOLDS, int Q>
__device__ __forceinline__ void fetch_raw(const uint32_t *in, uint64_t i, uint4 *raw) {
  if constexpr (FOLDS == 0 && IN_BASE) {
    uint2 e = *reinterpret_cast<const uint2 *>(in + 2 * i);
    raw[0] = make_uint4(e.x, e.y, 0u, 0u);
  } else {
    // words per pair: 16 (three folds), 8 (two), 4 (base, folding), 4 D (extension, folding), 2 D (extension)
    const uint4 *p = reinterpret_cast<const uint4 *>(in) + (uint64_t)Q * i;
#pragma unroll
    for (int q = 0; q < Q; q++) raw[q] = p[q];
  }
}
template <int D>
__device__ __forceinline__ Ext<D> ext_from_quads(const uint4 *q) {
  Ext<D> e;
  e.c[0] = q[0].x, e.c[1] = q[0].y, e.c[2] = q[0].z, e.c[3] = q[0].w;
  if constexpr (D == 8) e.c[4] = q[1].x, e.c[5] = q[1].y, e.c[6] = q[1].z, e.c[7] = q[1].w;
  return e;
}
template <int D, bool IN_BASE, int FOLDS, class V>
__device__ __forceinline__ void pair_from_raw(const uint4 *raw, const Ext<D> &r, V &lo, V &hi,
                                              const BindWeights<D, FOLDS >= 2 ? FOLDS : 2> *bw) {
  if constexpr (FOLDS >= 2) {
    constexpr int H = FOLDS == 3 ? 2 : 1;  // quads per entry
    uint32_t v[8 * H];
#pragma unroll
    for (int q = 0; q < 2 * H; q++) v[4 * q] = raw[q].x, v[4 * q + 1] = raw[q].y, v[4 * q + 2] = raw[q].z, v[4 * q + 3] = raw[q].w;
    lo = bind<D>(*bw, v);
    hi = bind<D>(*bw, v + 4 * H);
  } else if constexpr (FOLDS == 1 && IN_BASE) {
    lo = fold_base<D>(raw[0].x, raw[0].y, r);
    hi = fold_base<D>(raw[0].z, raw[0].w, r);
  } else if constexpr (FOLDS == 1) {
    constexpr int E = D / 4;  // quads per element
    lo = fold_ext<D>(ext_from_quads<D>(raw), ext_from_quads<D>(raw + E), r);
    hi = fold_ext<D>(ext_from_quads<D>(raw + 2 * E), ext_from_quads<D>(raw + 3 * E), r);
  } else if constexpr (IN_BASE) {
    lo = raw[0].x;
    hi = raw[0].y;
  } else {
    constexpr int E = D / 4;
    lo = ext_from_quads<D>(raw);
    hi = ext_from_quads<D>(raw + E);
  }
}

// A lane's values meet those of the lane that differs from it in lane bit M: x and y become, in the lanes with the
// bit clear, the two lanes' values of the first, in the others those of the second.  Bits 5 and 4 take one exchange of
// half registers; for the others the value the partner keeps is fetched by a permutation within a row of 16: the
// opposite lane of a group of 8 for bit 2 (so bits 0 and 1 come after it: until then all of a group's lanes still hold
// the same words), eight lanes on for bit 3, within quads for bits 1 and 0.  None goes through LDS.
template <int M>
__device__ __forceinline__ uint32_t lane_partner(uint32_t v) {
  static_assert(M == 1 || M == 2 || M == 4 || M == 8, "bits within a row");
  return M == 1 ? EXH_DPP(v, 0xB1) : M == 2 ? EXH_DPP(v, 0x4E) : M == 4 ? EXH_DPP(v, 0x141) : EXH_DPP(v, 0x128);
}
template <int M>
__device__ __forceinline__ uint32_t lane_sum(uint32_t v) {  // v plus the partner's v
  if constexpr (M >= 16) {
    const auto p = M == 32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false) : __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return fadd(p[0], p[1]);
  } else {
    return fadd(v, lane_partner<M>(v));
  }
}
template <int M>
__device__ __forceinline__ uint32_t lane_halve(uint32_t x, uint32_t y) {  // the sum of x (bit clear) or of y (bit set)
  if constexpr (M >= 16) {
    const auto p = M == 32 ? __builtin_amdgcn_permlane32_swap(x, y, false, false) : __builtin_amdgcn_permlane16_swap(x, y, false, false);
    return fadd(p[0], p[1]);
  } else {
    const bool upper = (threadIdx.x & M) != 0;
    return fadd(upper ? y : x, lane_partner<M>(upper ? x : y));
  }
}

// The wavefront's sums of W = 8, 16 or 32 values per lane, value k given by val(k): the values are halved over lane
// bits 5, 4, 3, .. until each lane holds one (about 2 W operations instead of the 6 W of a tree per value), then summed
// over the bits that are left.  Lane l ends with the sum of value transposed_word<W>(l); val is called for two values
// at a time, so only W / 2 are live at once.
template <int W>
__device__ __forceinline__ uint32_t transposed_word(uint32_t lane) {
  const uint32_t b5 = (lane >> 5) & 1, b4 = (lane >> 4) & 1, b3 = (lane >> 3) & 1, b2 = (lane >> 2) & 1, b1 = (lane >> 1) & 1;
  return W == 32 ? 16 * b5 + 8 * b4 + 4 * b3 + 2 * b2 + b1 : W == 16 ? 8 * b5 + 4 * b4 + 2 * b3 + b2 : 4 * b5 + 2 * b4 + b3;
}
template <int W>
__device__ __forceinline__ bool transposed_writer(uint32_t lane) {  // one lane per value
  return (lane & (64 / W - 1)) == 0;
}
template <int W, class F>
__device__ __forceinline__ uint32_t wave_sums_transposed(F val) {
  static_assert(W == 8 || W == 16 || W == 32, "three to five halvings");
  uint32_t a[W / 2];
#pragma unroll
  for (int k = 0; k < W / 2; k++) {
    const uint32_t x = val(k), y = val(k + W / 2);
    a[k] = lane_halve<32>(x, y);
  }
#pragma unroll
  for (int k = 0; k < W / 4; k++) a[k] = lane_halve<16>(a[k], a[k + W / 4]);
#pragma unroll
  for (int k = 0; k < W / 8; k++) a[k] = lane_halve<8>(a[k], a[k + W / 8]);
  if constexpr (W >= 16) {
#pragma unroll
    for (int k = 0; k < W / 16; k++) a[k] = lane_halve<4>(a[k], a[k + W / 16]);
  } else {
    a[0] = lane_sum<4>(a[0]);
  }
  a[0] = W == 32 ? lane_halve<2>(a[0], a[1 % (W / 2)]) : lane_sum<2>(a[0]);
  return lane_sum<1>(a[0]);
}

// accumulator words [first, first + W) of the lane, reduced mod p (zero beyond the statement's), summed
// over the wavefront and left in lds_row[first ..]
template <int D, int W, class Desc, class Acc>
__device__ __forceinline__ void chunk_sums(const Desc &d, Acc (*acc)[D], int first, uint32_t *lds_row) {
  const uint32_t total = wave_sums_transposed<W>([&](int k) -> uint32_t {
    const int o = first + k;
    return o < d.nacc * D ? acc_reduce(acc[o / D][o % D]) : 0u;
  });
  const uint32_t l = threadIdx.x & 63, o = first + transposed_word<W>(l);
  if (transposed_writer<W>(l) && o < (uint32_t)d.nacc * D) lds_row[o] = total;
}

// The workgroup's sums of every accumulator, reduced mod p, into sums[nacc * D] (LDS); all threads call.
// TRANSPOSED picks the cross-lane scheme: the transposing reduction is the shorter path (the latency-bound
// LDS-resident rounds use it), one tree per value keeps fewer registers live (the streaming round kernels,
// whose occupancy it would cost, use that).
template <int D, bool TRANSPOSED, class Desc, class Acc>
__device__ __forceinline__ void block_sums(const Desc &d, Acc (*acc)[D], uint32_t (*lds)[MAXACC * D],
                                           uint32_t *sums) {
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if constexpr (TRANSPOSED) {
    if (d.nacc * D <= 8)
      chunk_sums<D, 8>(d, acc, 0, lds[wave]);
    else if (d.nacc * D <= 16)
      chunk_sums<D, 16>(d, acc, 0, lds[wave]);
    else {
#pragma unroll
      for (int first = 0; first < MAXACC * D; first += 32)
        if (first < d.nacc * D) chunk_sums<D, 32>(d, acc, first, lds[wave]);
    }
  } else {
#pragma unroll
    for (int a = 0; a < MAXACC; a++) {
      if (a < d.nacc) {
#pragma unroll
        for (int c = 0; c < D; c++) {
          uint32_t v = wave_sum(acc_reduce(acc[a][c]));
          if (lane == 0) lds[wave][a * D + c] = v;
        }
      }
    }
  }
  lds_barrier();
  for (uint32_t o = tid; o < (uint32_t)d.nacc * D; o += BLOCK) {
    uint32_t v = lds[0][o];
#pragma unroll
    for (int wv = 1; wv < BLOCK / 64; wv++) v = fadd(v, lds[wv][o]);
    sums[o] = v;
  }
  lds_barrier();
}

// The wavefront's sums of the accumulators a = PART, PART + PARTS, ... (the ones accumulate_pair<.., PARTS> fills
// on the wavefront that has this part), reduced mod p, into sums[a * D ..] (LDS).  Every word of sums is written
// by one wavefront.
template <int D, int PART, int PARTS, int W, class Desc>
__device__ __forceinline__ void part_chunk_sums(const Desc &d, AccLazy (*acc)[D], int first, int count, uint32_t *sums) {
  const uint32_t total = wave_sums_transposed<W>([&](int k) -> uint32_t {
    const int o = first + k, q = o / D;
    return PARTS * q + PART < MAXACC && q < count ? acc_reduce(acc[(PARTS * q + PART) % MAXACC][o % D]) : 0u;
  });
  const uint32_t l = threadIdx.x & 63, o = first + transposed_word<W>(l);
  if (transposed_writer<W>(l) && o < (uint32_t)count * D) sums[(PARTS * (o / D) + PART) * D + o % D] = total;
}
template <int D, int PART, int PARTS, class Desc>
__device__ __forceinline__ void part_wave_sums(const Desc &d, AccLazy (*acc)[D], uint32_t *sums) {
  const int count = (d.nacc - PART + PARTS - 1) / PARTS;  // accumulators of this part
  if (count <= 0) return;
  if (count * D <= 8)
    part_chunk_sums<D, PART, PARTS, 8>(d, acc, 0, count, sums);
  else if (count * D <= 16)
    part_chunk_sums<D, PART, PARTS, 16>(d, acc, 0, count, sums);
  else {
#pragma unroll
    for (int first = 0; first < ((MAXACC + PARTS - 1) / PARTS) * D; first += 32)
      if (first < count * D) part_chunk_sums<D, PART, PARTS, 32>(d, acc, first, count, sums);
  }
}

// From the round's accumulator sums (LDS, scaled as the kernels leave them) to the round message, through the
// transcript, to the next challenge: rows = mtilde * sums + c0 (ROUND-MESSAGE, src/sumcheck.lisp:313-317), send =
// absorb the rows (src/transcript.lisp:116-128), r = challenge (src/transcript.lisp:174-176).  The workgroup's first
// wavefront does it alone: the message's words lie across its lanes and go from there straight into the transcript's
// pending block, with no barrier and no trip through LDS in between.
struct EpilogueLds {
  alignas(16) uint32_t prod[MAXPTS * MAXACC * 8];  // the totals' words of the groups, before they are added up
  uint32_t chal[8];
  uint32_t r_mont[8];
  uint32_t ring[RING_WORDS];
  // staged copies (filled by the caller when it passes staged = true)
  uint32_t state[sizeof(DevB3S) / 4];
  uint32_t round;
  alignas(16) uint32_t mtilde[MAXPTS * MAXACC * 8];
  alignas(16) uint32_t c0[MAXPTS * 8];
};

// Which part of the message a lane computes: word o = lane / parts (row o / D, coordinate o % D), and of its sum over
// the accumulators every parts-th term from `part` on; parts is as large as the message leaves lanes for, up to 8.
template <int D>
struct MessageLane {
  uint32_t o, part, parts;
  uint32_t at[D];  // the word of an accumulator's sum that goes with coordinate w^i of the map's element, or of its triple
};
constexpr uint32_t TRIPLED = MAXACC * 8;  // sums[TRIPLED + o] = 3 sums[o]: the products that wrap, w^D = 3
template <int D>
__device__ __forceinline__ MessageLane<D> message_lane(uint32_t points) {
  const uint32_t lane = threadIdx.x & 63, words = points * D;
  MessageLane<D> ml;
  ml.parts = words <= 8 ? 8 : words <= 16 ? 4 : words <= 32 ? 2 : 1;
  ml.o = lane / ml.parts, ml.part = lane % ml.parts;
  const uint32_t c = ml.o % D, e = D == 8 ? __brev(c) >> 29 : __brev(c) >> 30;
#pragma unroll
  for (int i = 0; i < D; i++) {
    const uint32_t j = (e - i) & (D - 1), tower = D == 8 ? __brev(j) >> 29 : __brev(j) >> 30;
    ml.at[i] = tower + ((uint32_t)i > e ? TRIPLED : 0u);
  }
  return ml;
}

// the lane's message word (every lane of a word's group has it); sums with their triples, mtilde and c0 in LDS
template <int D>
__device__ __forceinline__ uint32_t round_message_word(const uint32_t *sums, uint32_t nacc, uint32_t points,
                                                       const uint32_t *mtilde, const uint32_t *c0, const MessageLane<D> &ml) {
  const uint32_t o = ml.o < points * D ? ml.o : points * D - 1;
  uint64_t t = 0;
  for (uint32_t a = ml.part; a < nacc; a += ml.parts) {
    const Ext<D> m = load_ext<D>(mtilde + (size_t)((o / D) * nacc + a) * D);
#pragma unroll
    for (int i = 0; i < D; i++) {
      if (i % 2 == 0) t = mont_lazy(t);
      t += (uint64_t)m.c[brev(i, D)] * sums[a * D + ml.at[i]];
    }
  }
  uint32_t v = mont_reduce4(t);
  if (ml.parts >= 2) v = fadd(v, EXH_DPP(v, 0xB1));
  if (ml.parts >= 4) v = fadd(v, EXH_DPP(v, 0x4E));
  if (ml.parts >= 8) v = fadd(v, EXH_DPP(v, 0x141));
  return fadd(v, c0[o]);
}

// the triples beside the sums (the first wavefront)
__device__ __forceinline__ void triple_sums(uint32_t *sums, uint32_t width) {
  for (uint32_t o = threadIdx.x & 63; o < width; o += 64) sums[TRIPLED + o] = times3(sums[o]);
  __builtin_amdgcn_wave_barrier();
}

// The first wavefront's step: send the message whose words the lanes hold (what the last squeeze left to absorb and
// the message's length go first, unless `prefixed` says that they went already), draw the challenge into e->chal and,
// times R, e->r_mont (LDS), call `ready`, then log both.  What this squeeze leaves to absorb stays in `pending`.
template <int D, class Lds, class F>
__device__ __forceinline__ void transcript_step(RunB3S &tr, Ctrl *ctrl, uint32_t round, uint32_t points, Lds *e,
                                                const MessageLane<D> &ml, uint32_t word, PendingAppend &pending,
                                                bool prefixed, bool log, F ready) {
  const uint32_t lane = threadIdx.x & 63, words = points * D;
  if (!prefixed) rb3s_flush(tr, pending, words);
  for (uint32_t base = 0; base < words; base += 16) {  // sixteen words at a time, a word's bytes shared by its lanes
    const uint32_t o = ml.o - base;
    if (ml.o >= base && o < 16 && ml.o < words) {
      if (ml.parts >= 4) {
        if (ml.part < 4) rb3s_put_byte(tr, 4 * o + ml.part, word >> (8 * ml.part));
      } else if (ml.parts == 2) {
        rb3s_put_byte(tr, 4 * o + 2 * ml.part, word >> (16 * ml.part));
        rb3s_put_byte(tr, 4 * o + 2 * ml.part + 1, word >> (16 * ml.part + 8));
      } else {
        rb3s_put_word(tr, 4 * o, word);
      }
    }
    rb3s_advance(tr, 4 * (words - base < 16 ? words - base : 16));
  }
  dev_challenge(
      tr, D,
      [&](uint32_t at, uint32_t v) {
        e->chal[at] = v;
        e->r_mont[at] = to_mont(v);
      },
      ready, &pending);
  if (log) {
    if (ml.part == 0 && ml.o < words) ctrl->msg[round][ml.o] = word;
    if (lane < (uint32_t)D) ctrl->chal[round][lane] = e->chal[lane], ctrl->r_mont[lane] = e->r_mont[lane];
  }
}

// (all threads of the workgroup may call; the first wavefront works)
template <int D>
__device__ __forceinline__ void round_epilogue(Ctrl *ctrl, uint32_t *sums, uint32_t nacc, uint32_t points,
                                               const uint32_t *mtilde, const uint32_t *c0, EpilogueLds *e,
                                               bool staged = false) {
  const uint32_t tid = threadIdx.x;
  if (tid < 64) {
    const uint32_t round = staged ? e->round : ctrl->round;
    RunB3S tr;
    PendingAppend pending{0, 0, 0};
    rb3s_load(tr, e->ring, staged ? reinterpret_cast<const DevB3S *>(e->state) : &ctrl->tr);
    const MessageLane<D> ml = message_lane<D>(points);
    triple_sums(sums, nacc * D);
    const uint32_t word = round_message_word<D>(sums, nacc, points, mtilde, c0, ml);
    transcript_step<D>(tr, ctrl, round, points, e, ml, word, pending, false, true, [] {});
    rb3s_flush(tr, pending);
    rb3s_store(tr, &ctrl->tr);
    if (tid == 0) ctrl->round = round + 1;
  }
}

// All threads of the workgroup call with its sums (canonical, `width` words) in `mine` (LDS).  True in the one
// workgroup that arrived last, which then holds the sums over all workgroups in `sums` (LDS, width words);
// *ok is false when a word did not complete within the spin limit.  scratch: groups * width words of LDS.
// A launch may add only the words [add_first, add_first + add_count) (the passes of the base-field sweep share one
// set of totals, a pass per range of words); the workgroup whose ticket is last_ticket is the elected one.
// G: the workgroups that add to every word (the launch's grid, or the part of it that sums).
__device__ __forceinline__ bool add_and_elect(const RoundTotals &rt, const uint32_t *mine, uint32_t width,
                                              uint32_t *scratch, uint32_t *sums, bool *ok, uint32_t add_first,
                                              uint32_t add_count, uint32_t last_ticket, uint32_t G) {
  __shared__ uint32_t ticket;
  const uint32_t tid = threadIdx.x, wg = blockIdx.x, NG = rt.groups;
  for (uint32_t o = add_first + tid; o < add_first + add_count; o += blockDim.x)
    __hip_atomic_fetch_add(rt.totals + (size_t)(wg % NG) * rt.pstride + o, ((unsigned long long)1 << 48) + mine[o],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (tid == 0) ticket = __hip_atomic_fetch_add(rt.arrivals, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  *ok = true;
  if (ticket != last_ticket) return false;
  // every word this thread answers for is requested before any is looked at (one trip to memory for all), from a
  // clamped address so that no load hangs on a condition
  const uint32_t nwords = NG * width;
  unsigned long long v[TOTALS_POLLS];
  uint32_t pending = 0;
#pragma unroll
  for (int k = 0; k < TOTALS_POLLS; k++)
    if (tid + k * blockDim.x < nwords) pending |= 1u << k;
  uint32_t polls = 0;
  int complete = 1;
  while (pending) {
#pragma unroll
    for (int k = 0; k < TOTALS_POLLS; k++) {
      const uint32_t u = tid + k * blockDim.x, at = u < nwords ? u : 0;
      v[k] = __hip_atomic_load(rt.totals + (size_t)(at / width) * rt.pstride + at % width, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int k = 0; k < TOTALS_POLLS; k++) {
      const uint32_t u = tid + k * blockDim.x, g = u / width;
      const uint32_t expect = (G - g + NG - 1) / NG;  // workgroups w < G with w % NG == g
      if (((pending >> k) & 1u) && (uint32_t)(v[k] >> 48) == expect) {
        scratch[u] = f_canonical((double)(v[k] & (((unsigned long long)1 << 48) - 1)));  // exact below 2^53
        pending &= ~(1u << k);
      }
    }
    if (pending) {
      if (++polls > rt.spin_limit) {
        complete = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  if (!__syncthreads_and(complete)) {
    *ok = false;
    return true;
  }
  for (uint32_t o = tid; o < width; o += blockDim.x) {
    uint32_t t = 0;
    for (uint32_t g = 0; g < NG; g++) t = fadd(t, scratch[g * width + o]);
    sums[o] = t;
  }
  __syncthreads();
  return true;
}

// One workgroup's share of a round: pairs [block * tile, (block + 1) * tile) with tile = BLOCK *
// pairs_per_thread, folded first when FOLD, summed into the workgroup's partial row.
constexpr int FETCH_QUADS = 16;  // 16-byte quads of tables' words that a lane holds ahead of their arithmetic
template <int D>
struct RoundShape {
  const uint32_t *low, *high;
  uint64_t n_pairs;
  uint32_t low_bits, pairs_per_thread;
  bool deferred, do_sums;
  // device-driven rounds (totals non-null): see RoundTotals
  RoundTotals totals;
  uint32_t points;
  const uint32_t *mtilde, *c0;
  Ctrl *ctrl;
  const uint32_t *consts;
};

// what goes through fold_map (a base table's fold by one challenge, a product a coordinate, does not)
constexpr bool folds_mapped(int D, bool in_base, int folds) { return D == 8 && (folds >= 2 || (folds == 1 && !in_base)); }

template <int D, bool IN_BASE, int FOLDS, class Desc, bool GENERATED = false>
__device__ __forceinline__ void round_core(const Desc &d, const uint32_t *const *in, uint32_t *const *out,
                                           const RoundShape<D> &sh, const Ext<D> &r, uint32_t block,
                                           uint32_t *partial_row, const BindWeights<D, FOLDS >= 2 ? FOLDS : 2> *bw = nullptr,
                                           const FoldMap<FOLDS == 0 ? 1 : FOLDS> *map = nullptr) {
  constexpr bool BASE_MODE = IN_BASE && FOLDS == 0;  // the pair's values are base-field
  using V = typename std::conditional<BASE_MODE, uint32_t, Ext<D>>::type;
  const uint32_t tid = threadIdx.x;
  const uint64_t tile = (uint64_t)BLOCK * sh.pairs_per_thread;
  const uint64_t tile_start = (uint64_t)block * tile;
  const uint64_t low_mask = ((uint64_t)1 << sh.low_bits) - 1;

  typename AccOf<V, Desc>::type acc[MAXACC][D];
#pragma unroll
  for (int a = 0; a < MAXACC; a++)
#pragma unroll
    for (int c = 0; c < D; c++) acc_zero(acc[a][c]);

  // With a statement known at compile time a table's words are fetched well before their arithmetic (two workgroups per
  // compute unit leave the registers for it, and too few wavefronts to hide the loads behind one another): SLOTS tables'
  // words are held, table t in slot t % SLOTS, and a slot is filled again as soon as its words are used, with the next
  // table that goes there -- of this pair, or of the next one, whose first SLOTS tables then arrive under the sums.
  // (64 registers of words: two tables at a time of extension elements at D = 8, four at D = 4, all of them in base tables.
  // Without it, at D = 8, a table's loads waited behind the store of the table before: the largest fold round of a
  // four-table statement, 1.6 GB, took 530 us, 440 this way; more or fewer slots, 32 or 96 registers, make no difference
  // beyond the runs'.  Whole pairs held twice are 96 registers for three tables at D = 4 and spill for eight; fold rounds of
  // three tables and 2^21, 2^20 and 2^19 pairs one behind the other 149, 77.1 and 43.2 us that way with the arithmetic of
  // then, 147, 74.6 and 40.6 now.  (Behind the bind by three, the first of its kernel in a proof, a fold round of 2^19 pairs
  // takes 49 us with either way of fetching.)
  // A lane without a next pair fetches the tile's first one: a load under a condition would have to be merged with
  // what the slot held as soon as it is issued.  Left out by a condition on the pair's number, which is the same for all
  // lanes, that round takes 49.2 us for 48.6, and the fold rounds of four tables at D = 8 399 for 229 on average.)
  // The interpreter, and a statement in direct form, which is wide and calls its evaluator in a loop, keep the plain order.
  constexpr bool AHEAD = GENERATED && !is_direct<Desc>::value;
  if constexpr (AHEAD && folds_mapped(D, IN_BASE, FOLDS)) {
    // (the products take a wavefront's pairs together: its lanes stay together, and those beyond the last pair neither store
    // nor sum)
    constexpr int Q = raw_quads<D, IN_BASE, FOLDS>(), SLOTS = FETCH_QUADS / Q < MAXT ? FETCH_QUADS / Q : MAXT;
    const bool store = FOLDS == 1 || out[0] != nullptr;
    uint4 raw[SLOTS][Q];
    const uint32_t lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint64_t first = tile_start + wave * 64 < sh.n_pairs ? tile_start + wave * 64 : tile_start;
    auto last_of = [&](uint64_t base) { return sh.n_pairs - base < 64 ? (uint32_t)(sh.n_pairs - base) - 1 : 63u; };
#pragma unroll
    for (int t = 0; t < SLOTS; t++)
      if (t < d.T) fetch_mapped<FOLDS>(in[t], first, last_of(first), raw[t]);
    for (uint32_t k = 0; k < sh.pairs_per_thread; k++) {
      const uint64_t base = tile_start + (uint64_t)k * BLOCK + wave * 64;
      if (base >= sh.n_pairs) break;
      const uint64_t next = k + 1 < sh.pairs_per_thread && base + BLOCK < sh.n_pairs ? base + BLOCK : first;
      const uint32_t last = last_of(base), next_last = last_of(next);
      Ext<D> w;
      if (sh.do_sums) {
        w = load_ext<D>(sh.low + ((uint32_t)(base + lane) & (uint32_t)low_mask) * D);
        if (!sh.deferred) w = ext_mul_mont<D>(w, load_ext<D>(sh.high + ((base + umin32(lane, last)) >> sh.low_bits) * D));
      }
      V lo[MAXT], hi[MAXT];
      Quadratic<D> half;
#pragma unroll
      for (int t = 0; t < MAXT; t++)
        if (t < d.T) {
          pair_mapped<FOLDS>(*map, raw[t % SLOTS], lo[t], hi[t]);
          if (t + SLOTS < d.T)
            fetch_mapped<FOLDS>(in[t + SLOTS < MAXT ? t + SLOTS : 0], base, last, raw[t % SLOTS]);
          else
            fetch_mapped<FOLDS>(in[t % SLOTS], next, next_last, raw[t % SLOTS]);
          if (store && lane <= last) {
            char *const to = reinterpret_cast<char *>(out[t] + base * (2 * D));
            uint32_t at = lane * (8 * D);
            asm("" : "+v"(at));
            store_ext<D>(reinterpret_cast<uint32_t *>(to + at), lo[t]);
            store_ext<D>(reinterpret_cast<uint32_t *>(to + at + 4 * D), hi[t]);
          }
          // (what the first tables give by themselves, while the others' words arrive)
          if (sh.do_sums && product_of_four(d) && t == first_half_table(d)) half = quadratic<D>(d, 0, lo, hi, w);
        }
      if (sh.do_sums && lane <= last) {
        if (product_of_four(d))
          accumulate_quadratics<D>(d, half, quadratic<D>(d, 1, lo, hi, w), acc);
        else
          accumulate_pair<D, V>(d, lo, hi, w, acc, sh.consts);
      }
    }
  } else if constexpr (AHEAD) {
    constexpr int Q = raw_quads<D, IN_BASE, FOLDS>(), SLOTS = FETCH_QUADS / Q < MAXT ? FETCH_QUADS / Q : MAXT;
    const bool store = FOLDS == 1 || (FOLDS >= 2 && out[0] != nullptr);
    uint4 raw[SLOTS][Q];
    const uint64_t first = tile_start + tid < sh.n_pairs ? tile_start + tid : tile_start;
#pragma unroll
    for (int t = 0; t < SLOTS; t++)
      if (t < d.T) fetch_raw<D, IN_BASE, FOLDS, Q>(in[t], first, raw[t]);
    for (uint32_t k = 0; k < sh.pairs_per_thread; k++) {
      const uint64_t i = tile_start + (uint64_t)k * BLOCK + tid;
      if (i >= sh.n_pairs) break;
      const uint64_t next = k + 1 < sh.pairs_per_thread && i + BLOCK < sh.n_pairs ? i + BLOCK : tile_start;
      Ext<D> w;
      if (sh.do_sums) w = load_ext<D>(sh.low + (i & low_mask) * D);
      V lo[MAXT], hi[MAXT];
#pragma unroll
      for (int t = 0; t < MAXT; t++)
        if (t < d.T) {
          pair_from_raw<D, IN_BASE, FOLDS, V>(raw[t % SLOTS], r, lo[t], hi[t], bw);
          if (t + SLOTS < d.T)
            fetch_raw<D, IN_BASE, FOLDS, Q>(in[t + SLOTS < MAXT ? t + SLOTS : 0], i, raw[t % SLOTS]);
          else
            fetch_raw<D, IN_BASE, FOLDS, Q>(in[t % SLOTS], next, raw[t % SLOTS]);
          if constexpr (FOLDS > 0) {
            if (store) {
              store_ext<D>(out[t] + 2 * i * D, lo[t]);
              store_ext<D>(out[t] + (2 * i + 1) * D, hi[t]);
            }
          }
        }
      if (sh.do_sums) {
        if (!sh.deferred) w = ext_mul_mont<D>(w, load_ext<D>(sh.high + (i >> sh.low_bits) * D));
        accumulate_pair<D, V>(d, lo, hi, w, acc, sh.consts);
      }
    }
  } else {
    for (uint32_t k = 0; k < sh.pairs_per_thread; k++) {
      const uint64_t i = tile_start + (uint64_t)k * BLOCK + tid;
      if (i >= sh.n_pairs) break;
      V lo[MAXT], hi[MAXT];
      load_pair<D, IN_BASE, FOLDS == 1, V, Desc>(d, in, out, i, r, lo, hi);
      if (sh.do_sums) {
        Ext<D> w = load_ext<D>(sh.low + (i & low_mask) * D);
        if (!sh.deferred) w = ext_mul_mont<D>(w, load_ext<D>(sh.high + (i >> sh.low_bits) * D));
        accumulate_pair<D, V>(d, lo, hi, w, acc, sh.consts);
      }
    }
  }
  if (!sh.do_sums) return;

  __shared__ uint32_t lds[BLOCK / 64][MAXACC * D];
  __shared__ uint32_t sums[2 * TRIPLED];
  // a device-driven round: what the elected workgroup's serial part reads from memory (the transcript's state, the
  // message map, the constant terms) is requested by every workgroup here, ahead of the reduction that hides the
  // trip; the one elected later finds it in its LDS
  constexpr int PRE = (MAXPTS * MAXACC * 8 + BLOCK - 1) / BLOCK;
  uint32_t pre_map[PRE], pre_c0 = 0, pre_state = 0, pre_round = 0;
  if (sh.totals.totals) {
    const uint32_t map_words = sh.points * (uint32_t)d.nacc * D;
#pragma unroll
    for (int k = 0; k < PRE; k++) {
      const uint32_t u = tid + k * BLOCK;
      pre_map[k] = sh.mtilde[u < map_words ? u : 0];
    }
    pre_c0 = sh.c0[tid < sh.points * D ? tid : 0];
    pre_state = reinterpret_cast<const uint32_t *>(&sh.ctrl->tr)[tid < sizeof(DevB3S) / 4 ? tid : 0];
    pre_round = sh.ctrl->round;
  }
  block_sums<D, false>(d, acc, lds, sums);
  Ext<D> s;
  if (tid < (uint32_t)d.nacc) {
#pragma unroll
    for (int c = 0; c < D; c++) s.c[c] = sums[tid * D + c];
    if (sh.deferred) s = ext_mul_mont<D>(s, load_ext<D>(sh.high + (tile_start >> sh.low_bits) * D));
  }
  if (!sh.totals.totals) {
    if (tid < (uint32_t)d.nacc) store_ext<D>(partial_row + tid * D, s);
    return;
  }
  // the device-driven round: totals, and in the last workgroup to arrive the message and the challenge
  __shared__ EpilogueLds epi;
  __syncthreads();
  if (tid < (uint32_t)d.nacc) {
#pragma unroll
    for (int c = 0; c < D; c++) sums[tid * D + c] = s.c[c];
  }
  {
    const uint32_t map_words = sh.points * (uint32_t)d.nacc * D;
#pragma unroll
    for (int k = 0; k < PRE; k++)
      if (tid + k * BLOCK < map_words) epi.mtilde[tid + k * BLOCK] = pre_map[k];
    if (tid < sh.points * D) epi.c0[tid] = pre_c0;
    if (tid < sizeof(DevB3S) / 4) epi.state[tid] = pre_state;
    if (tid == 0) epi.round = pre_round;
  }
  __syncthreads();
  bool ok;
  const uint32_t width = (uint32_t)d.nacc * D;
  if (!add_and_elect(sh.totals, sums, width, epi.prod, sums, &ok, 0, width, gridDim.x - 1, gridDim.x)) return;
  if (!ok) {
    if (tid == 0) __hip_atomic_store(&sh.ctrl->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  round_epilogue<D>(sh.ctrl, sums, (uint32_t)d.nacc, sh.points, epi.mtilde, epi.c0, &epi, true);
}

template <int D, bool IN_BASE, int FOLDS, class Desc, bool GENERATED = false>
__device__ __forceinline__ void round_body(const Desc &d, const RoundArgs<D> &args) {
  RoundShape<D> sh{args.low, args.high, args.n_pairs, args.low_bits, args.pairs_per_thread, args.deferred != 0,
                   args.do_sums != 0, RoundTotals{args.totals, args.arrivals, args.groups, args.pstride, args.spin_limit},
                   args.points, args.mtilde, args.c0, args.ctrl, args.consts};
  uint32_t *const partial_row = args.partials + (uint64_t)blockIdx.x * args.pstride;
  Ext<D> r = ext_zero<D>();
  if constexpr (FOLDS == 1) {
    const uint32_t *rp = args.ctrl ? args.ctrl->r_mont : args.r_mont;
#pragma unroll
    for (int c = 0; c < D; c++) r.c[c] = rp[c];
  }
  if constexpr (GENERATED && !is_direct<Desc>::value && folds_mapped(D, IN_BASE, FOLDS)) {
    const FoldMap<FOLDS> map = fold_map<FOLDS>(r, args.ctrl);
    round_core<D, IN_BASE, FOLDS, Desc, GENERATED>(d, args.in, args.out, sh, r, blockIdx.x, partial_row, nullptr, &map);
  } else if constexpr (FOLDS >= 2) {
    const BindWeights<D, FOLDS> bw = bind_weights<D, FOLDS>(args.ctrl);
    round_core<D, true, FOLDS, Desc, GENERATED>(d, args.in, args.out, sh, r, blockIdx.x, partial_row, &bw);
  } else {
    round_core<D, IN_BASE, FOLDS, Desc, GENERATED>(d, args.in, args.out, sh, r, blockIdx.x, partial_row);
  }
}

// The round's second launch when the device drives the loop: one workgroup adds the partials, forms the
// message, runs the transcript and leaves the next challenge in ctrl.  (A last-workgroup-done scheme
// inside the round kernel needs a device-scope fence per workgroup, which on this part writes back the
// XCD's whole L2 and costs more than a launch.)
// sums[o] = sum over the workgroups' partial rows of word o (o < width <= blockDim.x): thread t takes column
// t % width of the rows t / width, t / width + groups, ... with groups = blockDim.x / width, so that all
// threads share the rows whatever the row stride; sixteen loads in flight per thread.
// All threads of the workgroup call; scratch holds blockDim.x words.
__device__ __forceinline__ void sum_partials(const uint32_t *partials, uint32_t nblocks, uint32_t ps, uint32_t width,
                                             uint32_t *scratch, uint32_t *sums) {
  const uint32_t tid = threadIdx.x, nthreads = blockDim.x;
  const uint32_t groups = width ? nthreads / width : 0, col = width ? tid % width : 0, row0 = width ? tid / width : 0;
  // sixteen loads in flight per thread and trip to memory, the last batch's rows beyond the end masked off (a loop
  // over single rows behind full batches would be a trip to memory per row)
  uint32_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (row0 < groups) {
    const uint32_t *p = partials + col;
    for (uint32_t b = row0; b < nblocks; b += 16 * groups) {
      uint32_t x[16];
#pragma unroll
      for (int q = 0; q < 16; q++) {
        const uint32_t row = b + q * groups;
        x[q] = row < nblocks ? p[(uint64_t)row * ps] : 0u;
      }
#pragma unroll
      for (int q = 0; q < 16; q++) v[q & 7] = fadd(v[q & 7], x[q]);
    }
  }
  __syncthreads();
  scratch[tid] = fadd(fadd(fadd(v[0], v[1]), fadd(v[2], v[3])), fadd(fadd(v[4], v[5]), fadd(v[6], v[7])));
  __syncthreads();
  if (tid < width) {
    uint32_t total = scratch[tid];
    for (uint32_t g = 1; g < groups; g++) total = fadd(total, scratch[g * width + tid]);
    sums[tid] = total;
  }
  __syncthreads();
}

struct EpilogueArgs {
  const uint32_t *partials;
  uint32_t nblocks, pstride, nacc, points;
  const uint32_t *mtilde, *c0;
  Ctrl *ctrl;
};

constexpr int EPI_BLOCK = 1024;

template <int D>
__global__ __launch_bounds__(EPI_BLOCK) void epilogue_kernel(EpilogueArgs args) {
  __shared__ uint32_t scratch[EPI_BLOCK];
  __shared__ uint32_t sums[2 * TRIPLED];
  __shared__ EpilogueLds epi;
  const uint32_t tid = threadIdx.x, width = args.nacc * D, ps = args.pstride;
  // everything the serial part needs from global memory is requested first, so that its latency
  // overlaps the partial sums: the transcript state, the message map and the constant terms
  if (tid < sizeof(DevB3S) / 4) epi.state[tid] = reinterpret_cast<const uint32_t *>(&args.ctrl->tr)[tid];
  if (tid == 64) epi.round = args.ctrl->round;
  for (uint32_t u = tid; u < args.points * width; u += EPI_BLOCK) epi.mtilde[u] = args.mtilde[u];
  for (uint32_t u = tid; u < args.points * D; u += EPI_BLOCK) epi.c0[u] = args.c0[u];
  sum_partials(args.partials, args.nblocks, ps, width, scratch, sums);
  round_epilogue<D>(args.ctrl, sums, args.nacc, args.points, epi.mtilde, epi.c0, &epi, true);
}

// A small round's sums on one wavefront: the accumulators PART, PART + 4, ... of the lane's pair, summed over the
// wavefront into sums (LDS).  The accumulators are this function's own, so that they live in registers.
template <int D, int PART, int PARTS, class Desc>
__device__ __forceinline__ void small_round_sums(const Desc &d, const Ext<D> *lo, const Ext<D> *hi, const Ext<D> &w,
                                                 uint32_t *sums, const uint32_t *kc) {
  AccLazy acc[MAXACC][D];
#pragma unroll
  for (int a = 0; a < MAXACC; a++)
#pragma unroll
    for (int c = 0; c < D; c++) acc_zero(acc[a][c]);
  accumulate_pair<D, Ext<D>, Desc, PARTS, PART>(d, lo, hi, w, acc, kc);
  part_wave_sums<D, PART, PARTS>(d, acc, sums);
}

// A product of an accumulator as a lane walks it in a spread round (see tail_body): its degree (0: the accumulator has no
// such product), its evaluation point, and where in LDS its factors' tables begin.
constexpr int SPREAD_FACTORS = MAXDEG;
constexpr int SPREAD_UNITS = MAXACC + MAXG;  // accumulators times the most products of one, as far as rounds run spread
struct SpreadUnit {
  uint32_t deg, x, table[SPREAD_FACTORS];
};
__device__ __forceinline__ uint32_t lane_bits(uint32_t n) {  // 2^bits: the next power of two from n up
  return n <= 1 ? 0 : 32 - __builtin_clz(n - 1);
}
// An accumulator's products are on lanes of their own (2^term_bits); in the interpreter, where they do not all fit, a lane
// takes them one after the other: a round beyond that costs it 25 us (three products of one coefficient and a table, a proof
// of 2^8 175 us and 237 without, of 2^15 469 and 597; 203 and 552 when every product had an accumulator of its own).  The
// kernels of a statement's own lose by it (three products of two tables, slices of 2^12 33.2 us and 31.6 without).  The lanes
// of an accumulator in the interpreter:
__device__ __forceinline__ uint32_t unit_bits(uint32_t pairs, uint32_t nacc, uint32_t term_bits) {
  const uint32_t bits = lane_bits(pairs) + term_bits;
  return bits > 6 || (nacc << bits) > 192 ? lane_bits(pairs) : bits;
}
template <int M>
struct LaneBit {
  static constexpr int value = M;
};

// A launch of LDS-resident rounds is part of a proof -- the grid of slices, or one workgroup with the last rounds -- or a
// session as a whole in one workgroup, which brings its constants, builds its weight tables and pads its tables.  A
// statement's own kernels are two, one for each: the launches of a chain wait for their instructions, and the parts of a
// proof without the session's code are 2 to 5 % shorter (us, one kernel for both and two: slices of 2^16 50.8 and 49.9, of
// 2^19 at four tables 103.6 and 101.3, of a fraction tree's layers 51.0 and 49.9 on average; a layer's last launch with the
// step behind it 44.2 and 42.5; a session of 2^10 55.8 and 53.6).  Not the grid and the one workgroup behind it as two: its
// instructions then come from memory when the streaming rounds before have used up the caches (last rounds of three tables of
// 2^24 47.5 and 53.4).  EITHER: one kernel for both, where it is compiled at run time; INTERPRETER: for any statement.
enum class Tail { ROUNDS, WHOLE, EITHER, INTERPRETER };

// A workgroup's slice of every table into LDS, MODE: entries of base tables (0), folded on the way in (1), of extension tables
// (2), folded (3).  Every load of a batch is issued before the first is waited for.  With a table's store to LDS between its load
// and the next table's, a launch opened with a trip to memory for each table and 256 entries: with the state and the constants,
// which are asked for beside the tables too, 9,900 cycles for nine tables of four entries and 18,200 for four of 2^10, now 5,700
// and 8,500.  The lanes beyond the slice fetch its last entry again.  `valid`: entries that there are, zeros beyond (0: all).
template <int D, int MODE, class Desc>
__device__ __forceinline__ void load_slice(const Desc &d, const uint32_t *const *in, uint32_t *tables, uint32_t cap, uint64_t first,
                                           uint32_t entries, uint32_t valid, const Ext<D> &r) {
  constexpr int WORDS = (MODE & 1 ? 2 : 1) * (MODE >= 2 ? D : 1), QUADS = (WORDS + 3) / 4;
  constexpr int SLOTS = FETCH_QUADS / QUADS;
  const int chunks = 4 * d.T <= SLOTS ? 4 : 2 * d.T <= SLOTS ? 2 : 1;  // of 256 entries, in a batch
  const uint64_t last = MODE == 2 && valid && valid < first + entries ? valid - 1 : first + entries - 1;
  for (uint32_t base = threadIdx.x; base - threadIdx.x < entries; base += BLOCK * chunks)
#pragma unroll
    for (int t0 = 0; t0 < MAXT; t0 += SLOTS)
      if (t0 < d.T) {
        uint4 raw[SLOTS][QUADS];
#pragma unroll
        for (int s = 0; s < SLOTS; s++) {
          const int t = t0 + s / chunks;
          if (t < d.T) {
            uint64_t x = first + base + s % chunks * BLOCK;
            x = x < last ? x : last;
            const uint32_t *p = in[t] + x * WORDS;
            if constexpr (WORDS == 1)
              raw[s][0].x = *p;
            else if constexpr (WORDS == 2) {
              const uint2 e = *reinterpret_cast<const uint2 *>(p);
              raw[s][0].x = e.x, raw[s][0].y = e.y;
            } else {
#pragma unroll
              for (int q = 0; q < QUADS; q++) raw[s][q] = reinterpret_cast<const uint4 *>(p)[q];
            }
          }
        }
#pragma unroll
        for (int s = 0; s < SLOTS; s++) {
          const int t = t0 + s / chunks;
          const uint32_t x = base + s % chunks * BLOCK;
          if (t < d.T && x < entries) {
            Ext<D> v;
            if constexpr (MODE == 0) {
              v = ext_zero<D>();
              v.c[0] = raw[s][0].x;
            } else if constexpr (MODE == 1) {
              v = fold_base<D>(raw[s][0].x, raw[s][0].y, r);
            } else if constexpr (MODE == 2) {
              v = ext_from_quads<D>(raw[s]);
              if (valid && first + x >= valid) v = ext_zero<D>();
            } else {
              v = fold_ext<D>(ext_from_quads<D>(raw[s]), ext_from_quads<D>(raw[s] + D / 4), r);
            }
            store_ext<D>(tables + ((size_t)t * cap + x) * D, v);
          }
        }
      }
}

// What a launch of rounds leaves to a step that follows in the same launch (the first wavefront's transcript, in registers
// and LDS, and the tables).
struct TailEnd {
  RunB3S tr;
  PendingAppend pending{0, 0, 0};
  const uint32_t *tables;  // table t's one entry at t * capacity * D
};

// Load (folding or lifting on the way in) into LDS, then per round sums -> message -> challenge -> fold
// on the slice this workgroup holds: entries [w * E, (w + 1) * E) of every table, E = entries / grid.
// A grid launch ends when its rounds are done and leaves the slices in `out` for the one-workgroup
// launch that follows; that one ends with the finals.
// STEP: a step follows in the launch, which takes the transcript and the finals from `end`; they go nowhere else.  False when
// an earlier launch had given up.
template <int D, Tail KIND, bool STEP = false, class Desc>
__device__ __forceinline__ bool tail_body(const Desc &d, const TailArgs<D> &args, TailEnd &end) {
  extern __shared__ __align__(16) uint32_t tail_tables[];  // [T][capacity][D]
  __shared__ uint32_t lds[BLOCK / 64][MAXACC * D];
  __shared__ uint32_t sums[2 * TRIPLED];
  __shared__ EpilogueLds epi;
  __shared__ uint32_t c0s[MAXTAIL * MAXPTS * D];
  // (a statement in direct form, or with linear forms among its factors, keeps a pair's accumulators on one lane)
  constexpr bool SPREAD = !is_direct<Desc>::value;
  __shared__ SpreadUnit units[SPREAD ? SPREAD_UNITS : 1];
  // (products of an accumulator: as many lanes each as the next power of two)
  const uint32_t term_bits = SPREAD ? lane_bits((uint32_t)desc_terms(d)) : 0;
  constexpr bool SESSION = KIND != Tail::ROUNDS;
  const uint32_t tid = threadIdx.x, cap = args.capacity, G = KIND == Tail::WHOLE ? 1 : gridDim.x,
                 wg = KIND == Tail::WHOLE ? 0 : blockIdx.x;
  const uint32_t width = (uint32_t)d.nacc * D;
  RunB3S &tr = end.tr;
  PendingAppend &pending = end.pending;  // (the first wavefront's)
  end.tables = tail_tables;
  MessageLane<D> ml;
  bool prefixed = false;
  uint32_t entries = (args.first_fold ? args.entries / 2 : args.entries) / G;  // of this workgroup's slice
  const uint32_t my_staged = SESSION && args.staged ? args.staged[tid < args.staged_words ? tid : 0] : 0;
  auto constants = [&] {  // (a trip over the bus for all of them)
    if (SESSION && args.staged) {
      if (tid < args.staged_words) args.staged_dst[tid] = my_staged;
      for (uint32_t u = tid + BLOCK; u < args.staged_words; u += BLOCK) args.staged_dst[u] = args.staged[u];
      __syncthreads();
    }
  };
  // The session's own weight tables (see TailArgs::factors), in LDS behind the tables: the factors, then an element 1, which is
  // every round's HIGH table, then the LOW tables as one heap: 2^s + x is the product over the last s variables as x's bits have
  // it (a session's rounds are few enough that LOW takes all variables behind the round's), the table of the round before s
  // variables.
  const bool own_weights = SESSION && args.own != 0;
  uint32_t *const own_factors = tail_tables + (size_t)d.T * cap * D;
  uint32_t *const own_tables = own_factors + (size_t)2 * args.n_vars * D;
  auto own_at = [&](uint32_t jj) { return 1u << (args.n_vars - (args.first_round + jj + 1)); };  // in elements
  uint32_t done_rounds;
  {
    // what the rounds need from memory besides the tables is asked for before them and goes to LDS behind them
    Ext<D> r = ext_zero<D>();
    uint32_t my_state = 0, my_map = 0, my_c0 = 0, my_factor = 0;
    const uint32_t map_words = args.points * width, c0_words = args.rounds * args.points * D, factor_words = 2 * args.n_vars * D;
    auto ask = [&] {
      if (args.first_fold) {
#pragma unroll
        for (int c = 0; c < D; c++) r.c[c] = args.ctrl->r_mont[c];
      }
      my_state = reinterpret_cast<const uint32_t *>(&args.ctrl->tr)[tid < sizeof(DevB3S) / 4 ? tid : 0];
      my_map = args.mtilde[tid < map_words ? tid : 0], my_c0 = args.c0[tid < c0_words ? tid : 0];
      if (own_weights && args.factors) my_factor = args.factors[tid < factor_words ? tid : 0];
      done_rounds = args.ctrl->round;
    };
    const bool early = !(SESSION && args.staged);
    if (early) ask();
    const uint64_t first = (uint64_t)wg * entries;
    if constexpr (KIND == Tail::INTERPRETER) {
      for (int t = 0; t < d.T; t++)
        for (uint32_t x = tid; x < entries; x += BLOCK) {
          const uint64_t gx = first + x;  // index after the fold on the way in
          const uint32_t *in = args.in[t];
          Ext<D> v;
          if (args.in_base) {
            if (args.first_fold) {
              uint2 e = *reinterpret_cast<const uint2 *>(in + 2 * gx);
              v = fold_base<D>(e.x, e.y, r);
            } else {
              v = ext_zero<D>();
              v.c[0] = in[gx];
            }
          } else if (args.first_fold) {
            v = fold_ext<D>(load_ext<D>(in + 2 * gx * D), load_ext<D>(in + (2 * gx + 1) * D), r);
          } else if (SESSION && args.valid && gx >= args.valid) {
            v = ext_zero<D>();
          } else {
            v = load_ext<D>(in + gx * D);
          }
          store_ext<D>(tail_tables + ((size_t)t * cap + x) * D, v);
        }
    } else if (args.in_base) {
      if (args.first_fold)
        load_slice<D, 1>(d, args.in, tail_tables, cap, first, entries, 0, r);
      else
        load_slice<D, 0>(d, args.in, tail_tables, cap, first, entries, 0, r);
    } else if (args.first_fold) {
      load_slice<D, 3>(d, args.in, tail_tables, cap, first, entries, 0, r);
    } else {
      load_slice<D, 2>(d, args.in, tail_tables, cap, first, entries, SESSION ? args.valid : 0, r);
    }
    constants();
    if (!early) ask();
    if (tid < sizeof(DevB3S) / 4) epi.state[tid] = my_state;
    if (tid < map_words) epi.mtilde[tid] = my_map;
    for (uint32_t u = tid + BLOCK; u < map_words; u += BLOCK) epi.mtilde[u] = args.mtilde[u];
    if (tid < c0_words) c0s[tid] = my_c0;
    for (uint32_t u = tid + BLOCK; u < c0_words; u += BLOCK) c0s[u] = args.c0[u];
    if (own_weights && args.factors) {
      if (tid < factor_words) own_factors[tid] = my_factor;
      for (uint32_t u = tid + BLOCK; u < factor_words; u += BLOCK) own_factors[u] = args.factors[u];
    }
  }
  __syncthreads();
  if (tid < 64) {
    rb3s_load(tr, epi.ring, reinterpret_cast<const DevB3S *>(epi.state));
    ml = message_lane<D>(args.points);
  }
  if (done_rounds != args.first_round) return false;  // an earlier launch gave up: leave the count as it is
  static_assert(SPREAD_UNITS <= 64 && BLOCK == 256, "the units are made by the last wavefront's lanes");
  if (const uint32_t u = tid - 192; SPREAD && tid >= 192 && ((uint32_t)d.nacc << term_bits) <= (uint32_t)SPREAD_UNITS &&
                                    u < ((uint32_t)d.nacc << term_bits)) {
    const uint32_t a = u >> term_bits, term = u & ((1u << term_bits) - 1);
    units[u].deg = 0, units[u].x = 0;
    for (int j = 0; j < SPREAD_FACTORS; j++) units[u].table[j] = 0;
    uint32_t met = 0;  // the accumulator's products so far
    for (int g = 0; g < d.G; g++)
      if (a >= (uint32_t)d.acc[g] && a < (uint32_t)(d.acc[g] + d.nev[g]) && met++ == term) {
        units[u].deg = (uint32_t)d.deg[g], units[u].x = (uint32_t)d.ev[g][a - (uint32_t)d.acc[g]];
        for (int j = 0; j < SPREAD_FACTORS; j++)
          units[u].table[j] = (uint32_t)d.tab[g][j < d.deg[g] ? j : 0] * cap * D;
      }
  }
  if (own_weights) {
    // The heap's entries of up to five variables, and beside them, on another wavefront, the products over the variables before
    // those five (below a factor R: `parts`, a heap as well); every other entry is a product of one of each.  An entry by
    // itself is a chain of up to nine products of 1,100 cycles and a search for its table: the weights of a session of 2^10 took
    // 20,000 cycles that way, 3,750 this way, of 2^6 5,000 and 1,850.
    constexpr uint32_t LAST = 5;
    __shared__ Ext<D> parts[2 << (OWN_VARS - LAST)];
    const uint32_t vars = args.n_vars - 1, late = vars < LAST ? vars : LAST, before = vars - late;
    auto product = [&](uint32_t from, uint32_t bits, uint32_t x) {  // over variables [from, from + bits), times R; bits >= 1
      auto factor = [&](uint32_t b) { return load_ext<D>(own_factors + ((size_t)(from + b) * 2 + (x >> b & 1 ? 0 : 1)) * D); };
      Ext<D> e = factor(0);
      for (uint32_t b = 1; b < bits; b++) e = ext_mul_mont<D>(e, factor(b));
      return e;
    };
    if (!args.factors) {
      for (uint32_t u = tid; u < 2u << vars; u += BLOCK) store_ext<D>(own_tables + (size_t)u * D, ext_lift<D>(1));
    } else if (tid >= 64 && tid < 128) {
      const uint32_t u = tid - 64, bits = u == 0 ? 0 : 31 - __builtin_clz(u);
      if (u < 2u << late)
        store_ext<D>(own_tables + (size_t)u * D, bits == 0 ? ext_lift<D>(1)  // (the exact product)
                                                           : ext_scale_mont<D>(product(args.n_vars - bits, bits, u - (1u << bits)), 1u));
    } else if (tid >= 128 && tid < 192) {
      const uint32_t u = tid - 128, bits = u == 0 ? 0 : 31 - __builtin_clz(u);
      if (bits > 0 && u < 2u << before) parts[u] = product(args.n_vars - late - bits, bits, u - (1u << bits));
    }
    __syncthreads();
    for (uint32_t u = (2u << late) + tid; args.factors && u < 2u << vars; u += BLOCK) {
      const uint32_t bits = 31 - __builtin_clz(u), x = u - (1u << bits), s = bits - late;
      const Ext<D> rest = load_ext<D>(own_tables + (size_t)((1u << late) + (x >> s)) * D);
      store_ext<D>(own_tables + (size_t)u * D, ext_mul_mont<D>(parts[(1u << s) + (x & ((1u << s) - 1))], rest));
    }
    __syncthreads();
  }
  // the weight factors of this thread's first pair of a round, fetched one round ahead
  Ext<D> wl = ext_zero<D>(), wh = ext_zero<D>();
  // (a round of at most 64 pairs runs with a pair per lane on all four wavefronts, each computing a share of the
  // pair's accumulators)
  const uint32_t lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  // (every thread loads, from a clamped index: a load under a condition has to be merged with the old value as soon
  // as it is issued, which turns the prefetch into a wait for memory at the end of every round)
  auto load_weight = [&](uint32_t jj, uint64_t i) {
    if (own_weights) {
      wl = load_ext<D>(own_tables + (size_t)(own_at(jj) + (uint32_t)(i & (((uint64_t)1 << args.low_bits[jj]) - 1))) * D);
      wh = args.block_high ? load_ext<D>(args.weights + (args.high_off[jj] + (i >> args.low_bits[jj])) * D)
                           : load_ext<D>(own_tables);
      return;
    }
    wl = load_ext<D>(args.weights + (args.low_off[jj] + (i & (((uint64_t)1 << args.low_bits[jj]) - 1))) * D);
    wh = load_ext<D>(args.weights + (args.high_off[jj] + (i >> args.low_bits[jj])) * D);
  };
  auto fetch_weight = [&](uint32_t jj, uint32_t pairs) {
    const uint32_t me = pairs <= 64 ? lane : tid;
    load_weight(jj, (uint64_t)wg * pairs + (me < pairs ? me : pairs - 1));
  };
  // A fold of `count` outputs by r, in place: the lanes run in lockstep, so every read of a chunk of 64 comes before
  // its writes, and those land below what later chunks read.  `spread`: wavefronts 1 to 3, an output per lane (a
  // table's outputs in as many lanes as the next power of two, so in one wavefront); else a table per wavefront.
  auto fold_small = [&](const Ext<D> &r, uint32_t count, bool spread) {
    if (spread) {
      const uint32_t u = tid - 64, bits = lane_bits(count), t = u >> bits, x = u & ((1u << bits) - 1);
      if (tid >= 64 && t < (uint32_t)d.T && x < count) {
        const uint32_t *p = tail_tables + ((size_t)t * cap + 2 * x) * D;
        const Ext<D> folded = fold_ext<D>(load_ext<D>(p), load_ext<D>(p + D), r);
        store_ext<D>(tail_tables + ((size_t)t * cap + x) * D, folded);
      }
      return;
    }
#pragma unroll
    for (int t = 0; t < MAXT; t++)
      if (t < d.T && (uint32_t)((t + 1) & 3) == wave) {  // (the first wavefront, late from the transcript, last)
        for (uint32_t x = lane; x < count; x += 64) {
          const uint32_t *p = tail_tables + ((size_t)t * cap + 2 * x) * D;
          const Ext<D> folded = fold_ext<D>(load_ext<D>(p), load_ext<D>(p + D), r);
          store_ext<D>(tail_tables + ((size_t)t * cap + x) * D, folded);
        }
      }
  };
  // Rounds whose (accumulator, pair) units fit the 192 lanes of wavefronts 1 to 3 run spread: a unit per lane, which
  // walks the accumulator's factors (their tables and its evaluation point come from LDS) instead of every wavefront
  // computing a third of the accumulators of a pair per lane; a unit is a few products where a third of a GKR layer's
  // accumulators is four, and the sum over the pairs halves its words over the lanes first.
  // (with several blocks the pairs are no power of two: a unit's lanes are the next one)
  // 192 is what three wavefronts hold: a round beyond that takes the shares below.  With the rule and without it, us:
  // the interpreter gains most (six groups, n = 12: 497 and 683; one group of six factors, n = 10: 428 and 767), the
  // kernels of a statement's own are about even (a launch over GKR layers: one lookup 28.2 and 27.6, two 34.2 and 34.7,
  // three 52.6 and 53.4 with the glue, 57.0 and 51.2 without; over the blocks of two lookups 21.5 and 25.3).
  // (WALK: see unit_bits.)
  constexpr bool WALK = KIND == Tail::INTERPRETER;
  auto spreads = [&](uint32_t pairs) {
    uint32_t bits = lane_bits(pairs) + term_bits;
    if constexpr (WALK) bits = unit_bits(pairs, (uint32_t)d.nacc, term_bits);
    return SPREAD && BLOCK == 256 && d.NV == 0 && bits <= 6 && ((uint32_t)d.nacc << bits) <= 192 &&
           ((uint32_t)d.nacc << term_bits) <= (uint32_t)SPREAD_UNITS;
  };
  uint32_t unit_a = 0, unit_lane = 0, unit_pair = 0, unit_deg = 0, unit_x = 0, unit_table[SPREAD_FACTORS];
  Ext<D> unit_w = ext_zero<D>();
  // a lane's unit of a round and its weight, which wait for nothing that the round before computes
  auto prepare_unit = [&](uint32_t jj, uint32_t pairs) {
    const uint32_t u = tid < 64 ? 0 : tid - 64;
    // (an accumulator's lanes: the pairs of its first product, of its second, ...)
    uint32_t pair_bits = lane_bits(pairs), bits = pair_bits + term_bits;
    if constexpr (WALK) bits = unit_bits(pairs, (uint32_t)d.nacc, term_bits);
    unit_a = u >> bits, unit_lane = u & ((1u << bits) - 1), unit_pair = unit_lane & ((1u << pair_bits) - 1);
    const SpreadUnit &unit = units[unit_a < (uint32_t)d.nacc ? (unit_a << term_bits) + (unit_lane >> pair_bits) : 0];
    unit_deg = unit.deg, unit_x = unit.x;
    const bool on = unit_pair < pairs && unit_deg != 0;  // (a lane without a pair takes the last one with no weight)
#pragma unroll
    for (int j = 0; j < SPREAD_FACTORS; j++) unit_table[j] = unit.table[j];
    const uint64_t i = (uint64_t)wg * pairs + (on ? unit_pair : pairs - 1);
    const uint32_t *low = own_weights ? own_tables + (size_t)own_at(jj) * D : args.weights + args.low_off[jj] * D;
    const uint32_t *high = own_weights && !args.block_high ? own_tables : args.weights + args.high_off[jj] * D;
    const Ext<D> l = load_ext<D>(low + (i & (((uint64_t)1 << args.low_bits[jj]) - 1)) * D);
    const Ext<D> h = load_ext<D>(high + (i >> args.low_bits[jj]) * D);
    unit_w = ext_scale_mont<D>(ext_mul_mont<D>(l, h), on ? R2 : 0u);  // (times R for the product that takes it in below)
  };
  // the round's sums from the units (wavefronts 1 to 3), with their triples
  auto unit_sums = [&](uint32_t pairs) {
    const int maxx = d.maxx, maxdeg = desc_maxdeg(d);
    auto factor = [&](uint32_t table) {  // the factor's line at the unit's evaluation point
      const uint32_t *p = tail_tables + table + 2 * (unit_pair < pairs ? unit_pair : pairs - 1) * D;
      const Ext<D> lo = load_ext<D>(p), hi = load_ext<D>(p + D);
      Ext<D> v;
#pragma unroll
      for (int c = 0; c < D; c++) {
        const uint32_t slope = fsub(hi.c[c], lo.c[c]);
        uint32_t at = unit_x >= 1 ? hi.c[c] : lo.c[c], next = hi.c[c];
#pragma unroll
        for (int x = 2; x <= MAXX; x++)
          if (x <= maxx) {
            next = fadd(next, slope);
            at = unit_x >= (uint32_t)x ? next : at;
          }
        v.c[c] = at;
      }
      return v;
    };
    Ext<D> f = factor(unit_table[0]);
#pragma unroll
    for (int j = 1; j < SPREAD_FACTORS; j++)
      if (j < maxdeg) {
        if ((uint32_t)j < unit_deg) f = ext_mul_mont<D>(f, factor(unit_table[j]));
      }
    if constexpr (WALK) {
      if (unit_bits(pairs, (uint32_t)d.nacc, term_bits) < lane_bits(pairs) + term_bits &&
          unit_a < (uint32_t)d.nacc)  // (of one degree and one evaluation point)
        for (uint32_t term = 1; term < 1u << term_bits; term++) {
          const SpreadUnit &unit = units[(unit_a << term_bits) + term];
          if (unit.deg == 0) break;
          Ext<D> g = factor(unit.table[0]);
          for (uint32_t j = 1; j < unit.deg; j++) g = ext_mul_mont<D>(g, factor(unit.table[j]));
          f = ext_add<D>(f, g);
        }
    }
    f = ext_mul_mont<D>(f, unit_w);
    // Over the pairs, the low lane bits of a unit: the words are halved as long as there are several.  Bit 2 comes first:
    // its partner is the opposite lane of a group of 8, which still holds the same words then (see lane_partner).
    uint32_t lanes = 1u << (lane_bits(pairs) + term_bits);
    if constexpr (WALK) lanes = 1u << unit_bits(pairs, (uint32_t)d.nacc, term_bits);
    uint32_t v[D], word = 0, count = D, keys = 0;
#pragma unroll
    for (int c = 0; c < D; c++) v[c] = f.c[c];
    auto step = [&](auto bit) {
      constexpr int M = decltype(bit)::value;
      if (lanes <= (uint32_t)M) return;
      auto halve = [&](auto half) {
        constexpr int H = decltype(half)::value;
#pragma unroll
        for (int k = 0; k < H; k++) v[k] = lane_halve<M>(v[k], v[k + H]);
        word = 2 * word + ((lane & M) ? 1 : 0), count = H, keys |= M;
      };
      if constexpr (M <= 4) {
        if (D == 8 && count == 8)
          halve(LaneBit<D / 2>{});
        else if (count == 4)
          halve(LaneBit<2>{});
        else if (count == 2)
          halve(LaneBit<1>{});
        else
          v[0] = lane_sum<M>(v[0]);
      } else {
        v[0] = lane_sum<M>(v[0]);
      }
    };
    step(LaneBit<4>{}), step(LaneBit<1>{}), step(LaneBit<2>{}), step(LaneBit<8>{}), step(LaneBit<16>{}), step(LaneBit<32>{});
    if (tid >= 64 && unit_a < (uint32_t)d.nacc && (unit_lane & ~keys) == 0) {
#pragma unroll
      for (int k = 0; k < D; k++)
        if (k < (int)count) {
          const uint32_t o = unit_a * D + word * count + k;
          sums[o] = v[k], sums[TRIPLED + o] = times3(v[k]);
        }
    }
  };
  if (spreads(entries / 2)) {
    __syncthreads();  // (the units and the session's own weights)
    if (tid >= 64) prepare_unit(0, entries / 2);
  } else {
    fetch_weight(0, entries / 2);
  }
  __syncthreads();
  for (uint32_t jj = 0; jj < args.rounds; jj++) {
    const uint32_t pairs = entries / 2;
    const bool small = pairs <= 64 && BLOCK == 256, spread = spreads(pairs), more = jj + 1 < args.rounds;
    const bool next_spread = more && spreads(pairs / 2);
    {  // the round's sums
      if (spread) {
        // the first wavefront, which ran the transcript, meanwhile absorbs what the last squeeze left to absorb and
        // the length of the message to come (a compression every other round): nobody waits for that any more
        if (wave == 0)
          rb3s_flush(tr, pending, args.points * D), prefixed = true;
        else
          unit_sums(pairs);
        lds_barrier();
      } else if (small) {  // each wavefront its own share of the pair's accumulators, in code of its own
        Ext<D> lo[MAXT], hi[MAXT];
        const uint32_t at = lane < pairs ? lane : 0;
#pragma unroll
        for (int t = 0; t < MAXT; t++)
          if (t < d.T) {
            const uint32_t *p = tail_tables + ((size_t)t * cap + 2 * at) * D;
            lo[t] = load_ext<D>(p);
            hi[t] = load_ext<D>(p + D);
          }
        Ext<D> ww = ext_mul_mont<D>(wl, wh);
        if (lane >= pairs) ww = ext_zero<D>();  // lanes without a pair add nothing
        if (more && !next_spread) fetch_weight(jj + 1, pairs / 2);
        // three wavefronts share the accumulators; the first as above
        if (wave == 0)
          rb3s_flush(tr, pending, args.points * D), prefixed = true;
        else if (wave == 1)
          small_round_sums<D, 0, 3>(d, lo, hi, ww, sums, args.consts);
        else if (wave == 2)
          small_round_sums<D, 1, 3>(d, lo, hi, ww, sums, args.consts);
        else
          small_round_sums<D, 2, 3>(d, lo, hi, ww, sums, args.consts);
        lds_barrier();
      } else {
        AccLazy acc[MAXACC][D];
#pragma unroll
        for (int a = 0; a < MAXACC; a++)
#pragma unroll
          for (int c = 0; c < D; c++) acc_zero(acc[a][c]);
        for (uint32_t i = tid; i < pairs; i += BLOCK) {
          Ext<D> lo[MAXT], hi[MAXT];
#pragma unroll
          for (int t = 0; t < MAXT; t++)
            if (t < d.T) {
              const uint32_t *p = tail_tables + ((size_t)t * cap + 2 * i) * D;
              lo[t] = load_ext<D>(p);
              hi[t] = load_ext<D>(p + D);
            }
          if (i >= BLOCK) load_weight(jj, (uint64_t)wg * pairs + i);  // beyond the prefetched pair
          accumulate_pair<D, Ext<D>>(d, lo, hi, ext_mul_mont<D>(wl, wh), acc, args.consts);
        }
        if (more && !next_spread) fetch_weight(jj + 1, pairs / 2);
        block_sums<D, true>(d, acc, lds, sums);
      }
      if (G > 1) {
        // The round's sums over all workgroups.  Each workgroup adds its sums into its group's totals,
        // one integer atomic per word that also counts the contribution in the word's top 16 bits; a
        // word whose count equals the group's size is complete, so readers poll the words themselves:
        // nothing else is exchanged (the tables live in LDS), and no fence or separate barrier is needed.
        // Groups keep the atomics on one address few.
        const uint32_t NG = args.groups, gsize = G / NG;
        unsigned long long *totals = args.totals + (size_t)jj * NG * args.pstride;
        for (uint32_t o = tid; o < width; o += BLOCK)
          __hip_atomic_fetch_add(totals + (size_t)(wg % NG) * args.pstride + o, ((unsigned long long)1 << 48) + sums[o],
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int complete = 1;
        for (uint32_t u = tid; u < NG * width; u += BLOCK) {
          const unsigned long long *word = totals + (size_t)(u / width) * args.pstride + u % width;
          unsigned long long v;
          uint32_t polls = 0;
          while (((v = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >> 48) != gsize) {
            if (++polls > args.spin_limit) {  // the grid is not all there: give up, the host sees the round count
              complete = 0;
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
          epi.prod[u] = f_canonical((double)(v & (((unsigned long long)1 << 48) - 1)));  // exact below 2^53
        }
        if (!__syncthreads_and(complete)) {
          // leave a mark: the others may have seen this workgroup's sums and go on to publish the rounds, but
          // its slice is never written
          if (tid == 0) __hip_atomic_store(&args.ctrl->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          return true;
        }
        for (uint32_t o = tid; o < width; o += BLOCK) {
          uint32_t v = 0;
          for (uint32_t g = 0; g < NG; g++) v = fadd(v, epi.prod[g * width + o]);
          sums[o] = v, sums[TRIPLED + o] = times3(v);
        }
        lds_barrier();
      }
    }
    {  // the message, the challenge, the fold
      // The first wavefront goes on alone, up to the barrier at which the others, which meanwhile prepare what of the
      // next round they can, wait for the challenge; it finishes the transcript's step behind that barrier.
      if (wave == 0) {
        if (G == 1 && !spread) triple_sums(sums, width);
        const uint32_t word = round_message_word<D>(sums, (uint32_t)d.nacc, args.points, epi.mtilde,
                                                    c0s + (size_t)jj * args.points * D, ml);
        transcript_step<D>(tr, args.ctrl, args.first_round + jj, args.points, &epi, ml, word, pending, prefixed, wg == 0,
                           [] { lds_barrier(); });
        prefixed = false;
      } else {
        if (next_spread) prepare_unit(jj + 1, pairs / 2);
        lds_barrier();
      }
      Ext<D> r;
#pragma unroll
      for (int c = 0; c < D; c++) r.c[c] = epi.r_mont[c];
      if (small) {
        fold_small(r, pairs, ((uint32_t)d.T << lane_bits(pairs)) <= 192);
        lds_barrier();
      }
      // fold in place, 256 entries at a time in ascending order: a chunk's reads come before its writes,
      // and its writes land below everything a later chunk reads
      for (uint32_t base = 0; base < pairs && !small; base += BLOCK) {
        const uint32_t x = base + tid;
        Ext<D> folded[MAXT];
        if (x < pairs) {
#pragma unroll
          for (int t = 0; t < MAXT; t++)
            if (t < d.T) {
              const uint32_t *p = tail_tables + ((size_t)t * cap + 2 * x) * D;
              folded[t] = fold_ext<D>(load_ext<D>(p), load_ext<D>(p + D), r);
            }
        }
        lds_barrier();
        if (x < pairs) {
#pragma unroll
          for (int t = 0; t < MAXT; t++)
            if (t < d.T) store_ext<D>(tail_tables + ((size_t)t * cap + x) * D, folded[t]);
        }
        lds_barrier();
      }
    }
    entries = pairs;
  }
  const bool delivers = !STEP && args.host_log && G == 1;
  if (STEP || delivers) __syncthreads();  // (the logs' stores are done before other wavefronts read them)
#pragma unroll
  for (int t = 0; t < MAXT; t++)
    if (t < d.T)
      for (uint32_t x = tid; x < entries; x += BLOCK)
        store_ext<D>(args.out + (((size_t)t * G + wg) * entries + x) * D,
                     load_ext<D>(tail_tables + ((size_t)t * cap + x) * D));
  if (STEP) return true;
  const uint32_t done = args.first_round + args.rounds;
  if (G == 1 && entries == 1 && tid < (uint32_t)d.T * D) {  // the finals travel with the logs
    const uint32_t v = tail_tables[(size_t)(tid / D) * cap * D + tid % D];
    args.ctrl->finals[tid] = v;
    if (delivers) args.host_log[offsetof(Ctrl, finals) / 4 + tid] = v;
  }
  if (tid < 64) {
    rb3s_flush(tr, pending);
    if (wg == 0) {
      // (by way of LDS: with the state stored twice, the compiler reloads a spilled pair of registers -- its 64-bit counter, in the
      // kernel of a wide statement -- into an odd one, which it then refuses)
      rb3s_store(tr, reinterpret_cast<DevB3S *>(epi.state));
      __builtin_amdgcn_wave_barrier();
      if (tid < sizeof(DevB3S) / 4) {
        reinterpret_cast<uint32_t *>(&args.ctrl->tr)[tid] = epi.state[tid];
        if (delivers) args.host_log[tid] = epi.state[tid];
      }
      if (tid == 0) args.ctrl->round = done;
      if (tid == 0 && delivers) args.host_log[offsetof(Ctrl, round) / 4] = done;
    }
  } else if (delivers) {
    // The other wavefronts bring what the rounds filled of the logs -- points * D words of a round's message, D of its
    // challenge -- and the mark of a grid that gave up, every word through the L2 (this workgroup wrote some of them a moment
    // ago, other launches the rest), while the first one ends the transcript and sends its state itself.
    const uint32_t mw = args.points * D, messages = done * mw, total = messages + done * D + 1;
    const uint32_t *words = reinterpret_cast<const uint32_t *>(args.ctrl);
    constexpr uint32_t TRIP = 4, LANES = BLOCK - 64;
    for (uint32_t base = tid - 64; base < total; base += TRIP * LANES) {
      uint32_t at[TRIP], w[TRIP];
#pragma unroll
      for (uint32_t k = 0; k < TRIP; k++) {
        const uint32_t u = base + k * LANES, c = u - messages;
        at[k] = u < messages    ? (uint32_t)(offsetof(Ctrl, msg) / 4) + u / mw * (MAXPTS * 8) + u % mw
                : u < total - 1 ? (uint32_t)(offsetof(Ctrl, chal) / 4) + c / D * 8 + c % D
                                : (uint32_t)(offsetof(Ctrl, gave_up) / 4);
        w[k] = __hip_atomic_load(words + at[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
#pragma unroll
      for (uint32_t k = 0; k < TRIP; k++)
        if (base + k * LANES < total) args.host_log[at[k]] = w[k];
    }
  }
  if (delivers) {
    __threadfence_system();
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(args.host_log + args.host_flag_at, args.host_seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  return true;
}

// ---- rounds 0 and 1 from one sweep of the base tables.  A pair of round 1 is four base entries per table:
// the value at (X0, X1) is bilinear in them, u(X1) + X0 v(X1) with base-field u, v.  A group of degree d is
// therefore a polynomial of degree d in X0 with base-field coefficients at every X1, and the kernel sums,
// weighted by round 1's weights, its values on a grid ("slots"):
//   (point e, node m):  X1 = the group's e-th evaluation point, X0 = m in 0..d     -- round 1, whose epilogue
//                       interpolates in X0 at the challenge r0,
//   (extra e):          X1 = 1, X0 = the e-th evaluation point                     -- round 0: its sum at X0 is
//                       eq(w1, 0) * slot(X1 = 0, X0) + eq(w1, 1) * slot(X1 = 1, X0), the weight of variable 1
//                       being the one factor round 0's weights have beyond round 1's.
// All products are base-field; no folded table is written; rounds 2 and 3 read the base tables.  A launch covers the slots
// [PASS * SPP, (PASS + 1) * SPP) so the accumulators stay in registers.
// The epilogue of that sweep, both rounds by one workgroup: slot sums -> round 0's accumulator sums -> its
// message, through the transcript, to r0 -> the Lagrange basis at r0 -> round 1's accumulator sums -> its
// message and r1.  The statement's shape comes as run-time arrays.
struct NodesEpilogueArgs {
  EpilogueArgs e;            // c0 points at round 0's rows, round 1's follow
  const uint32_t *eq1;       // eq(w1, 1) and eq(w1, 0) as two elements, Montgomery form; null: both weights 1
  uint32_t groups, slots;
  uint32_t deg[MAXG], nev[MAXG];
  uint8_t ev[MAXG][MAXEV];
  uint32_t inv_den[(MAXDEG + 1) * (MAXDEG + 1)];  // [deg][m]: 1 / prod_{q != m, q <= deg} (m - q), Montgomery form
};

template <int D>
struct NodesArgs {
  const uint32_t *in[MAXT];  // base tables
  // round 1's weights in three factors: the pair index's low four bits (16 EXTs), the bits from there to low_bits in digit
  // form (SWEEP_* below), and HIGH for the rest (null: ones; the weights of blocks shorter than a tile are in the digits)
  const uint32_t *columns, *digits, *high;
  uint64_t n_pairs;          // pairs of round 1, four base entries each: a multiple of BLOCK
  uint32_t low_bits, pairs_per_thread;  // a workgroup's tile stays within 2^low_bits pairs
  // the slot sums of all passes meet in one set of counted totals (slot s at word s * D), and the last workgroup
  // of the last pass to arrive runs the two rounds' epilogue itself (see RoundTotals)
  RoundTotals totals;
  uint32_t passes;
  NodesEpilogueArgs epi;
};

// A 64-bit accumulator of 32 x 32-bit products kept below p 2^32 by a conditional subtraction of p from its high
// word after every product: acc < p 2^32, the product of a canonical weight and a residue below 2^32 is below
// p 2^32 as well, so the sum is below 2^64, and min(hi, hi - p) brings it back (hi < p: hi - p wraps above hi).
__device__ __forceinline__ void lazy_mad(uint64_t &acc, uint32_t w, uint32_t v) {
  acc = mont_lazy((uint64_t)w * v + acc);
}
__device__ __forceinline__ uint32_t lazy_reduce(uint64_t acc) {
  Acc96 a;
  a.lo = acc, a.hi = 0;
  return acc_reduce(a);
}

// The sweep's weighted sums are matrix products.  A wavefront's step is 128 pairs: lane n + 16 g takes pairs 64 t + 16 g + n
// (t = 0, 1), so that column n holds the pairs whose index ends in n, and along a column only the index above the low four
// bits varies: sum over k of mid[k] v[k][n] for all sixteen columns at once, with the sixteen columns' own weights applied
// once a workgroup.  In bytes: a value is written in four signed digits v = sum_j v_j 2^(8 j), a weight's coordinate w as the
// four digits of each of w 2^(8 j) mod p, and w v is congruent to sum_i 2^(8 i) sum_j digit_i(w 2^(8 j)) v_j, so that row
// (coordinate, i) of the product's result, an exact 32-bit sum, is that coordinate's i-th digit sum.  Sixteen rows
// at F_p^4 and thirty-two at F_p^8, eight pairs' four bytes along the contraction: v_mfma_i32_16x16x32_i8 with the value's
// word as it is for the right operand and digit words made once per proof (store_sweep_digits) for the left.
// What that takes from the vector units, which bound the sweep: a slot's weighted sum is two instructions a pair (its digits)
// where a multiply-add a coordinate, their reductions and a canonical value are eleven at F_p^4 and nineteen at F_p^8, and
// half the registers, so that F_p^8 needs one pass for the 24 slots of a product of four, not three.  With the quadratics
// below, by the counters: 327 vector instructions a pair for 559 with three tables at F_p^4 (2^24 entries: 100 -> 70 us), 517
// for 1455 with four at F_p^8 (2^26: 860 -> 355 to 385 us).
constexpr int SWEEP_STEP = 128;         // pairs of a wavefront's step
// A digit sum grows by at most 4 * 128 * 128 a pair of its column, a column has a sixteenth of a wavefront's share of the
// tile, and the sums of four digits are put together below 2^54.02.
constexpr int SWEEP_PPT_BITS = 12;
static_assert(((uint64_t)64 / 16 * 4 * 128 * 128) << SWEEP_PPT_BITS <= (uint64_t)1 << 30, "a digit sum stays within 2^30");
#if defined(__HIPCC__)
// a quarter of weight k's coordinates into place: [k / 8][coordinate / 4][lane (coordinate % 4) * 4 + i + 16 (k % 4)][k / 4 % 2],
// byte j = digit i of w 2^(8 j)
template <int D>
__device__ __forceinline__ void store_sweep_digits(uint32_t *out, uint64_t k, const Ext<D> &e, uint32_t quarter) {
  constexpr uint32_t SHIFT[4] = {R1, (uint32_t)(((uint64_t)R1 << 8) % P), (uint32_t)(((uint64_t)R1 << 16) % P),
                                 (uint32_t)(((uint64_t)R1 << 24) % P)};  // 2^(8 j) R
#pragma unroll
  for (uint32_t tile = 0; tile < D / 4; tile++) {
    const uint32_t w = quarter == 0 ? e.c[4 * tile] : quarter == 1 ? e.c[4 * tile + 1] : quarter == 2 ? e.c[4 * tile + 2]
                                                                                                   : e.c[4 * tile + 3];
    uint32_t dig[4];
#pragma unroll
    for (int j = 0; j < 4; j++) dig[j] = signed_digits(mont_mul(w, SHIFT[j]));
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t word = 0;
#pragma unroll
      for (int j = 0; j < 4; j++) word |= ((dig[j] >> (8 * i)) & 255u) << (8 * j);
      const uint32_t lane = quarter * 4 + i + 16u * (uint32_t)(k & 3);
      out[(((k >> 3) * (D / 4) + tile) * 64 + lane) * 2 + ((k >> 2) & 1)] = word;
    }
  }
}
#endif

// the LDS of the two rounds' epilogue
template <int D>
struct NodesEpilogueLds {
  uint32_t slot_sums[MAXACC * D];
  uint32_t sums[2 * TRIPLED];
  uint32_t basis[(MAXDEG + 1) * (MAXDEG + 1) * D];  // [deg][node]: Lagrange basis at r0, Montgomery form
  // the statement's shape: indexed by lane-dependent values out of the kernel's arguments, every access would be
  // a load from memory with the next one waiting behind it
  uint32_t s_deg[MAXG], s_nev[MAXG], s_inv_den[(MAXDEG + 1) * (MAXDEG + 1)];
  uint8_t s_ev[MAXG][MAXEV];
  EpilogueLds epi;
};

// everything the epilogue reads from memory, into LDS (all threads call; a barrier must follow before use)
template <int D>
__device__ __forceinline__ void nodes_epilogue_stage(const NodesEpilogueArgs &args, NodesEpilogueLds<D> &L) {
  const uint32_t tid = threadIdx.x, nthreads = blockDim.x, points = args.e.points, nacc = args.e.nacc;
  if (tid < MAXG) L.s_deg[tid] = args.deg[tid], L.s_nev[tid] = args.nev[tid];
  if (tid < MAXG * MAXEV) L.s_ev[tid / MAXEV][tid % MAXEV] = args.ev[tid / MAXEV][tid % MAXEV];
  if (tid < (MAXDEG + 1) * (MAXDEG + 1)) L.s_inv_den[tid] = args.inv_den[tid];
  if (tid < sizeof(DevB3S) / 4) L.epi.state[tid] = reinterpret_cast<const uint32_t *>(&args.e.ctrl->tr)[tid];
  for (uint32_t u = tid; u < points * nacc * D; u += nthreads) L.epi.mtilde[u] = args.e.mtilde[u];
  for (uint32_t u = tid; u < points * D; u += nthreads) L.epi.c0[u] = args.e.c0[u];
}

// from the slot sums (L.slot_sums) to both rounds' messages and challenges; all threads of the workgroup call
template <int D>
__device__ __forceinline__ void nodes_epilogue_body(const NodesEpilogueArgs &args, NodesEpilogueLds<D> &L) {
  const uint32_t tid = threadIdx.x, nthreads = blockDim.x, points = args.e.points, nacc = args.e.nacc;
  EpilogueLds &epi = L.epi;
  auto slot = [&](uint32_t index) {
    Ext<D> v;
#pragma unroll
    for (int c = 0; c < D; c++) v.c[c] = L.slot_sums[index * D + c];
    return v;
  };
  auto row_of = [&](uint32_t g, uint32_t x) {  // the index of X among group g's points, or nev
    uint32_t at = L.s_nev[g];
    for (uint32_t e = 0; e < L.s_nev[g]; e++)
      if (L.s_ev[g][e] == x) at = e;
    return at;
  };
  // accumulator tid is point e of group g, whose slots start at `base` (every thread finds its own, so that the
  // accumulators' sums below run side by side on the lanes of one wavefront)
  uint32_t g = 0, e = 0, base = 0;
  bool mine = false;
  {
    uint32_t a = 0;
    for (uint32_t k = 0; k < args.groups && !mine; k++) {
      const uint32_t nev = L.s_nev[k];
      if (tid < a + nev) {
        g = k, e = tid - a, mine = true;
      } else {
        a += nev;
        base += nev * (L.s_deg[k] + 1) + (row_of(k, 1) < nev ? 0 : nev);
      }
    }
  }
  // ---- round 0: accumulator (g, e) = eq(w1, 0) * slot(X1 = 0, node ev_e) + eq(w1, 1) * slot(X1 = 1, node ev_e)
  if (mine) {
    const uint32_t deg = L.s_deg[g], nev = L.s_nev[g], row0 = row_of(g, 0), row1 = row_of(g, 1);
    const uint32_t node = L.s_ev[g][e];
    Ext<D> at0 = slot(base + row0 * (deg + 1) + node);
    Ext<D> at1 = row1 < nev ? slot(base + row1 * (deg + 1) + node) : slot(base + nev * (deg + 1) + e);
    if (args.eq1) {
      at1 = ext_mul_mont<D>(at1, load_ext<D>(args.eq1));
      at0 = ext_mul_mont<D>(at0, load_ext<D>(args.eq1 + D));
    }
    const Ext<D> total = ext_add<D>(at0, at1);
#pragma unroll
    for (int c = 0; c < D; c++) L.sums[tid * D + c] = total.c[c];
  }
  __syncthreads();
  RunB3S tr;
  PendingAppend pending{0, 0, 0};
  MessageLane<D> ml;
  auto send_round = [&](uint32_t round) {  // (the first wavefront)
    triple_sums(L.sums, nacc * D);
    const uint32_t word = round_message_word<D>(L.sums, nacc, points, epi.mtilde, epi.c0, ml);
    transcript_step<D>(tr, args.e.ctrl, round, points, &epi, ml, word, pending, false, true, [] {});
  };
  if (tid < 64) {
    rb3s_load(tr, epi.ring, reinterpret_cast<const DevB3S *>(epi.state));
    ml = message_lane<D>(points);
    send_round(0);
  }
  __syncthreads();
  // ---- round 1: the basis of nodes 0..deg at r0, L_m = prod_{q != m} (r0 - q) / (m - q)
  for (uint32_t u = tid; u < points * D; u += nthreads) epi.c0[u] = args.e.c0[points * D + u];
  if (tid < (MAXDEG + 1) * (MAXDEG + 1)) {
    const uint32_t deg = tid / (MAXDEG + 1), m = tid % (MAXDEG + 1);
    if (deg >= 1 && m <= deg) {
      Ext<D> r0, acc = ext_lift<D>(R1);  // 1 in Montgomery form
#pragma unroll
      for (int c = 0; c < D; c++) r0.c[c] = epi.r_mont[c];
      for (uint32_t q = 0; q <= deg; q++) {
        if (q == m) continue;
        Ext<D> f = r0;
        f.c[0] = fsub(f.c[0], to_mont(q));  // (r0 - q) R
        acc = ext_mul_mont<D>(acc, f);
      }
      acc = ext_scale_mont<D>(acc, L.s_inv_den[tid]);
#pragma unroll
      for (int c = 0; c < D; c++) L.basis[tid * D + c] = acc.c[c];
    }
  }
  __syncthreads();
  // accumulator (g, e) = sum over nodes of basis * slot
  if (mine) {
    const uint32_t deg = L.s_deg[g];
    Ext<D> total = ext_zero<D>();
    for (uint32_t m = 0; m <= deg; m++) {
      Ext<D> lb;
#pragma unroll
      for (int c = 0; c < D; c++) lb.c[c] = L.basis[(deg * (MAXDEG + 1) + m) * D + c];
      total = ext_add<D>(total, ext_mul_mont<D>(lb, slot(base + e * (deg + 1) + m)));
    }
#pragma unroll
    for (int c = 0; c < D; c++) L.sums[tid * D + c] = total.c[c];
  }
  __syncthreads();
  if (tid < 64) {
    send_round(1);
    rb3s_flush(tr, pending);
    rb3s_store(tr, &args.e.ctrl->tr);
    if (tid == 0) args.e.ctrl->round = 2;
  }
}

// the slot sums: lines and products in double precision (field.hpp), weighted sums on the matrix cores (above)
template <int D, int PASS, int SPP, class Desc>
__device__ __forceinline__ void nodes_body(const Desc &d, const NodesArgs<D> &args) {
  // magnitudes, in units of p: a table line's ends < 1, a linear form < 5 (MAXVT terms and the constant),
  // the step between X points < 10, so at X <= 7 a line's end < 65 and its slope < 52, a node's value
  // < 65 + 6 * 52 = 377; a product of two < 377^2 p^2 < 2^80 and its quotient by p < 2^49.
  // A quadratic's reduced values and coefficient are within 0.57 p; at X <= 4 it is within 19 times that, and in X0 <= 4
  // within 19 times that again: 206 p.
  static_assert(MAXVT <= 4 && MAXX <= 7 && MAXDEG <= 6, "the bounds of the double-precision products");
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint64_t tile = (uint64_t)BLOCK * args.pairs_per_thread, tile_start = (uint64_t)blockIdx.x * tile;
  const uint64_t tile_end = tile_start + tile < args.n_pairs ? tile_start + tile : args.n_pairs;
  const uint64_t low_mask = ((uint64_t)1 << args.low_bits) - 1;
  constexpr int TILES = D / 4, STEPS = SWEEP_STEP / 64;
  digit_sums acc[SPP][TILES];
  uint32_t held[SPP];  // the digits of a step's first pairs, until its second ones complete the product's operand
#pragma unroll
  for (int a = 0; a < SPP; a++)
#pragma unroll
    for (int q = 0; q < TILES; q++) acc[a][q] = digit_sums{0, 0, 0, 0};

  // the loads run a step ahead of the arithmetic: few waves fit beside the accumulators
  uint4 ahead[STEPS][MAXT];
  uint2 wahead[TILES];
  const uint64_t first = tile_start + wave * SWEEP_STEP;
  // (a wavefront's step lies in its tile as a whole; behind the last one the first is fetched again, and not used)
  auto fetch = [&](int t, uint64_t base) {
#pragma unroll
    for (int q = 0; q < MAXT; q++)
      if (q < d.T) ahead[t][q] = reinterpret_cast<const uint4 *>(args.in[q] + 4 * (base + 64 * t))[lane];
  };
  auto fetch_digits = [&](uint64_t base) {
    if (args.digits) {
      const uint32_t *const at = args.digits + ((base & low_mask) / SWEEP_STEP) * (TILES * 128);
#pragma unroll
      for (int q = 0; q < TILES; q++) wahead[q] = reinterpret_cast<const uint2 *>(at)[q * 64 + lane];
    }
  };
  // without digits every weight is one: coordinate 0's row i has digit i of 2^(8 j), one at j = i
#pragma unroll
  for (int q = 0; q < TILES; q++)
    wahead[q].x = wahead[q].y = q == 0 && (lane & 15) < 4 ? 1u << (8 * (lane & 15)) : 0u;
  if (first < tile_end) {
#pragma unroll
    for (int t = 0; t < STEPS; t++) fetch(t, first);
    fetch_digits(first);
  }
  for (uint64_t base = first; base < tile_end; base += (BLOCK / 64) * SWEEP_STEP) {
    const uint64_t next = base + (BLOCK / 64) * SWEEP_STEP < tile_end ? base + (BLOCK / 64) * SWEEP_STEP : first;
    uint2 weights[TILES];
#pragma unroll
    for (int q = 0; q < TILES; q++) weights[q] = wahead[q];
    fetch_digits(next);
#pragma unroll
    for (int step_pairs = 0; step_pairs < STEPS; step_pairs++) {
      // per factor: the line in r0 at X = 0 (u0 + r0 v0) and at X = 1 (u1 + r0 v1)
      double cu[MAXT], cv[MAXT], du[MAXT], dv[MAXT], u1[MAXT], v1[MAXT];
#pragma unroll
      for (int t = 0; t < MAXT; t++)
        if (t < d.T) {
          const uint4 e = ahead[step_pairs][t];
          cu[t] = (double)e.x, cv[t] = (double)e.y - cu[t], u1[t] = (double)e.z, v1[t] = (double)e.w - u1[t];
        }
      fetch(step_pairs, next);
#pragma unroll
      for (int v = 0; v < MAXV; v++)
        if (v < d.NV) {  // a linear form of the tables: the same combination of the lines
          double a0 = (double)d.vconst[v], b0 = 0, a1 = a0, b1 = 0;
#pragma unroll
          for (int q = 0; q < MAXVT; q++)
            if (q < d.vn[v]) {
              const int t = d.vtab[v][q];
              a0 += f_scale(cu[t], d.vcoef[v][q]), b0 += f_scale(cv[t], d.vcoef[v][q]);
              a1 += f_scale(u1[t], d.vcoef[v][q]), b1 += f_scale(v1[t], d.vcoef[v][q]);
            }
          cu[d.T + v] = a0, cv[d.T + v] = b0, u1[d.T + v] = a1, v1[d.T + v] = b1;
        }
#pragma unroll
      for (int t = 0; t < MAXT; t++)
        if (t < d.T + d.NV) du[t] = u1[t] - cu[t], dv[t] = v1[t] - cv[t];

      // A group of three or four factors takes two of them (or two and two) as one quadratic in X1 and in X0: nine products
      // give its values at X1 = 0 and 1 and its coefficient of X1^2, each of them at X0 = 0 and 1 and as the coefficient of
      // X0^2, and the others follow by differences; a slot is then one product, where a factor at a time takes two or three.
      double qcur[MAXQUADS][3], qstep[MAXQUADS][3], qtwo[MAXQUADS][3], qnext[MAXQUADS][3];
      int quads_n = 0;
#pragma unroll
      for (int g = 0; g < MAXG; g++)
        if (g < d.G) {
#pragma unroll
          for (int h = 0; h < 2; h++)
            if (h < sweep_quads(d, g)) {
              const int a = d.tab[g][2 * h], b = d.tab[g][2 * h + 1], q = first_quad(d, g) + h;
              const double va[3][3] = {
                  {cu[a], u1[a], du[a]}, {cu[a] + cv[a], u1[a] + v1[a], du[a] + dv[a]}, {cv[a], v1[a], dv[a]}};
              const double vb[3][3] = {
                  {cu[b], u1[b], du[b]}, {cu[b] + cv[b], u1[b] + v1[b], du[b] + dv[b]}, {cv[b], v1[b], dv[b]}};
#pragma unroll
              for (int k = 0; k < 3; k++) {
                qcur[q][k] = f_mul(va[k][0], vb[k][0]);
                qnext[q][k] = f_mul(va[k][1], vb[k][1]);
                const double square = f_mul(va[k][2], vb[k][2]);
                qtwo[q][k] = square + square;
                qstep[q][k] = qnext[q][k] - qcur[q][k];
              }
              quads_n = q + 1;
            }
        }
      int slot = 0;  // numbered group by group (point by point, node by node, then the extras) -- visited X1-major
#pragma unroll
      for (int x = 0; x <= (d.maxx > 1 ? d.maxx : 1); x++) {
        if (x >= 1) {
#pragma unroll
          for (int t = 0; t < MAXT; t++)
            if (t < d.T + d.NV) {
              if (x == 1)
                cu[t] = u1[t], cv[t] = v1[t];
              else
                cu[t] += du[t], cv[t] += dv[t];
            }
#pragma unroll
          for (int q = 0; q < MAXQUADS; q++)
            if (q < quads_n)
#pragma unroll
              for (int k = 0; k < 3; k++) {
                if (x == 1) {
                  qcur[q][k] = qnext[q][k];
                } else {
                  qstep[q][k] += qtwo[q][k];
                  qcur[q][k] += qstep[q][k];
                }
              }
        }
        int base = 0, lead_base = 0;  // first slot of group g, and of the group whose slots it shares
        double shared_sum[MAXDEG + 1];
#pragma unroll
        for (int g = 0; g < d.G; g++) {
          const int e = ev_index(d, g, x);  // an evaluation point's row, or at X1 = 1 the row of extras
          const bool first = d.lead[g] == g, last = group_is_last(d, g);
          if (first) lead_base = base;
          if (e >= 0 || x == 1) {
            // the row's factors at X0 = 0, the quadratics first
            const int quads = sweep_quads(d, g), factors = d.deg[g] - quads, q0 = first_quad(d, g);
            double val[MAXDEG], step[2];
#pragma unroll
            for (int j = 0; j < MAXDEG; j++) {
              if (j < quads)
                val[j] = qcur[q0 + (j & 1)][0], step[j & 1] = qcur[q0 + (j & 1)][1] - val[j];
              else if (j < factors)
                val[j] = cu[d.tab[g][j + quads]];
            }
#pragma unroll
            for (int m = 0; m <= d.deg[g]; m++) {
              if (e >= 0)
                slot = lead_base + e * (d.deg[g] + 1) + m;
              else  // only the nodes that are evaluation points
                slot = ev_index(d, g, m) < 0 ? -1 : lead_base + d.nev[g] * (d.deg[g] + 1) + ev_index(d, g, m);
              if (slot >= PASS * SPP && slot < (PASS + 1) * SPP) {
                double prod = val[0];
#pragma unroll
                for (int j = 1; j < MAXDEG; j++)
                  if (j < factors) prod = f_mul(prod, val[j]);
                shared_sum[m] = first ? prod : shared_sum[m] + prod;  // (groups that share the slot follow one another)
                if (last) {
                  const double total = d.deg[g] == 1 || !first ? f_reduce(shared_sum[m]) : shared_sum[m];
                  const uint32_t digits = f_signed_digits(total);
                  const int at = slot - PASS * SPP;
                  if (step_pairs == 0) {
                    held[at] = digits;
                  } else {
                    const long value = (long)((uint64_t)digits << 32 | held[at]);
#pragma unroll
                    for (int q = 0; q < TILES; q++)
                      acc[at][q] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                          (long)((uint64_t)weights[q].y << 32 | weights[q].x), value, acc[at][q], 0, 0, 0);
                  }
                }
              }
#pragma unroll
              for (int j = 0; j < MAXDEG; j++) {
                if (j < quads) {
                  if (m > 0) step[j & 1] += 2.0 * qcur[q0 + (j & 1)][2];
                  val[j] += step[j & 1];
                } else if (j < factors) {
                  val[j] += cv[d.tab[g][j + quads]];
                }
              }
            }
          }
          base += group_slots(d, g);
        }
      }
      (void)slot;
    }
  }

  // the workgroup's sums of this launch's slots, the columns' weights and HIGH applied once
  constexpr int OWN = (SPP + 3) / 4, WORDS = OWN * D;  // slots and words that a wavefront sees to
  static_assert(BLOCK == 256, "four wavefronts share the slots");
  __shared__ uint32_t by_wave[BLOCK / 64][SPP * TILES][64];
  __shared__ uint32_t lds[BLOCK / 64][(WORDS + 31) / 32 * 32];
  __shared__ NodesEpilogueLds<D> L;
  nodes_epilogue_stage<D>(args.epi, L);  // (the loads' trip hides behind the reduction below)
  // This lane holds coordinates 4 q + g of its column's sums: the sum over a column's coordinates c of w^brev(c) times the
  // column's weight, so of the weight's words moved up by brev(c) powers of w, those that wrap tripled; times R^2, since the
  // digit sums come out over R and the product takes another.
  uint32_t weight[TILES][D];
#pragma unroll
  for (int q = 0; q < TILES; q++) {
    const uint32_t c = 4 * q + (lane >> 4), power = brev_bits<D>(c);
#pragma unroll
    for (int e = 0; e < D; e++) {
      const uint32_t from = brev_bits<D>((brev(e, D) - power) & (D - 1));
      uint32_t v = args.columns ? args.columns[(lane & 15) * D + from] : from == 0 ? 1u : 0u;
      if ((uint32_t)brev(e, D) < power) v = times3(v);
      weight[q][e] = mont_mul(v, R3);
    }
  }
  // the four wavefronts' columns added up, a quarter of the slots by each
#pragma unroll
  for (int a = 0; a < SPP; a++)
#pragma unroll
    for (int q = 0; q < TILES; q++) {
      const digit_sums &v = acc[a][q];
      const int64_t t = (int64_t)v[0] + (int64_t)v[1] * 256 + (int64_t)v[2] * 65536 + (int64_t)v[3] * 16777216;
      by_wave[wave][a * TILES + q][lane] = mont_reduce((uint64_t)(t + (int64_t)((uint64_t)P << 24)));  // (below 2^54.02 + 2^55)
    }
  __syncthreads();
  uint32_t column[OWN][TILES];
#pragma unroll
  for (int a = 0; a < OWN; a++) {
    const uint32_t at = wave * OWN + a;
#pragma unroll
    for (int q = 0; q < TILES; q++) {
      uint32_t v = 0;
      if (at < (uint32_t)SPP) {
        v = by_wave[0][at * TILES + q][lane];
#pragma unroll
        for (int w = 1; w < BLOCK / 64; w++) v = fadd(v, by_wave[w][at * TILES + q][lane]);
      }
      column[a][q] = v;
    }
  }
  {  // and added up across the lanes, 32 words at a time by the transposing reduction
    const uint32_t idx = transposed_word<32>(lane);
#pragma unroll
    for (int first_word = 0; first_word < WORDS; first_word += 32) {
      const uint32_t total = wave_sums_transposed<32>([&](int k) -> uint32_t {
        const int o = first_word + k;
        if (o >= WORDS) return 0u;
        const uint64_t t = (uint64_t)column[o / D][0] * weight[0][o % D];
        if constexpr (TILES == 2) return mont_reduce4(t + (uint64_t)column[o / D][TILES - 1] * weight[TILES - 1][o % D]);
        return mont_reduce(t);
      });
      if (transposed_writer<32>(lane)) lds[wave][first_word + idx] = total;
    }
  }
  __syncthreads();
  const int total = node_slots(d);
  const bool mine = tid < SPP && PASS * SPP + (int)tid < total;
  Ext<D> sum = ext_zero<D>();
  if (mine) {
    // The sums above are of w * (the plain product of the group's factors); the integer kernels' products
    // carry 1/R per multiplication, which the epilogue's constants expect: times R^(1 - degree) here.
    int base = 0, deg = 1;
    for (int g = 0; g < d.G; g++) {
      if (d.lead[g] == g && PASS * SPP + (int)tid >= base) deg = d.deg[g];
      base += group_slots(d, g);
    }
    uint32_t fix = R1;  // mont_mul(v, fix) = v R^(1 - degree)
    for (int q = 1; q < deg; q++) fix = mont_mul(fix, 1u);
#pragma unroll
    for (int c = 0; c < D; c++) {
      sum.c[c] = mont_mul(lds[tid / OWN][tid % OWN * D + c], fix);
    }
    // (the product's 1/R is one that the epilogue's constants expect)
    sum = args.high ? ext_mul_mont<D>(sum, load_ext<D>(args.high + (tile_start >> args.low_bits) * D)) : ext_scale_mont<D>(sum, 1u);
  }
  // the slot sums of all workgroups and passes, and in the last workgroup of the last pass both rounds' epilogue
  if (mine) {
#pragma unroll
    for (int c = 0; c < D; c++) L.sums[(PASS * SPP + tid) * D + c] = sum.c[c];
  }
  __syncthreads();
  const int here = total - PASS * SPP < SPP ? total - PASS * SPP : SPP;  // slots of this pass
  bool ok;
  if (!add_and_elect(args.totals, L.sums, (uint32_t)total * D, L.epi.prod, L.slot_sums, &ok, (uint32_t)(PASS * SPP * D),
                     (uint32_t)(here > 0 ? here : 0) * D, args.passes * gridDim.x - 1, gridDim.x))
    return;
  if (!ok) {
    if (tid == 0) __hip_atomic_store(&args.epi.e.ctrl->gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  nodes_epilogue_body<D>(args.epi, L);
}

// a kernel generated for one statement: S::d is its descriptor, known at compile time
template <int D, bool IN_BASE, bool FOLD, class S>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2))) void round_kernel(RoundArgs<D> args) {
  round_body<D, IN_BASE, FOLD ? 1 : 0, decltype(S::d), true>(S::d, args);
}
template <int D, class S, Tail KIND>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(1, 1))) void tail_kernel(TailArgs<D> args) {
  TailEnd end;
  tail_body<D, KIND>(S::d, args, end);
}
// (the same with half the registers: a statement in direct form at F_p^8 needs more than the 512 either way, and the
// compiler's use of the upper half of the register file for 64-bit values that it also spills has been seen to end
// in registers it then rejects)
template <int D, class S>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2))) void tail_kernel_narrow(TailArgs<D> args) {
  TailEnd end;
  tail_body<D, Tail::EITHER>(S::d, args, end);
}
// base tables folded by the first FOLDS = 2 or 3 (at F_p^8 also 4) challenges at once, see round_core; without tables to write
// (out[0] null) only the sums are taken
template <int D, class S, int FOLDS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2, 2))) void round_kernel_bind(RoundArgs<D> args) {
  round_body<D, true, FOLDS, decltype(S::d), true>(S::d, args);
}
// (24 slots at F_p^8 by one wavefront a SIMD: two passes of twelve with two a SIMD repeat the tables' part of the work, 487 us
// for 356 with four tables of 2^26 and 162 for 123 of 2^24; three tables, 15 slots, two passes and one 114 and 81)
template <int D, class S, int PASS, int SPP>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(sweep_waves(S::d, D, SPP), sweep_waves(S::d, D, SPP)))) void
nodes_kernel(NodesArgs<D> args) {
  nodes_body<D, PASS, SPP>(S::d, args);
}

// the interpreter: the same bodies over a run-time descriptor
template <int D, bool IN_BASE, bool FOLD>
__global__ __launch_bounds__(BLOCK) void round_kernel_interp(RoundArgs<D> args, StmtDesc d) {
  round_body<D, IN_BASE, FOLD ? 1 : 0>(d, args);
}
template <int D>
__global__ __launch_bounds__(BLOCK) void tail_kernel_interp(TailArgs<D> args, StmtDesc d) {
  TailEnd end;
  tail_body<D, Tail::INTERPRETER>(d, args, end);
}

}  // namespace exh
