// gkr.hip -- see gkr.hpp.
#include "gkr.hpp"

#include <string.h>

#include <atomic>
#include <vector>

#include "context.hpp"
#include "forms.hpp"
#include "hostfield.hpp"
#include "prover.hpp"
#include "gkr_glue.hpp"
#include "sumcheck_kernels.hpp"

namespace exh {

constexpr int REDUCE_MAXL = MAXT / 4;  // lookups proved together: four tables each
// the parent of two children: p = p0 q1 + p1 q0, q = q0 q1 (products carry 1/R; multiplying one factor of each product by
// R^2 first makes them exact)
template <int D>
struct Fraction {
  Ext<D> p, q;
};
template <int D>
__device__ __forceinline__ Fraction<D> load_fraction(const uint32_t *p, const uint32_t *q, uint64_t at) {
  return {load_ext<D>(p + at * D), load_ext<D>(q + at * D)};
}
template <int D>
__device__ __forceinline__ Fraction<D> add_fractions(const Fraction<D> &a, const Fraction<D> &b) {
  const Ext<D> q1r = ext_scale_mont<D>(b.q, R2), q0r = ext_scale_mont<D>(a.q, R2);
  return {ext_add<D>(ext_mul_mont<D>(a.p, q1r), ext_mul_mont<D>(b.p, q0r)), ext_mul_mont<D>(a.q, q1r)};
}
template <int D>
__device__ __forceinline__ void store_fraction(uint32_t *p, uint32_t *q, uint64_t at, const Fraction<D> &f) {
  store_ext<D>(p + at * D, f.p);
  store_ext<D>(q + at * D, f.q);
}

// A layer from the one below, parent (b, x) of children (b, x) and (b, x + 2^m), for every lookup (blockIdx.y); TWO: and the
// layer above that, whose parent (b, x) has the parents (b, x) and (b, x + 2^(m-1)): a thread per parent of the last layer.
// Two layers in a launch take the middle one from registers: trees of 2^22 and 2^16 leaves, above the last nine
// layers, 117 us in 20 launches one at a time, 94 in 11.
struct ReduceArgs {
  const uint32_t *p[REDUCE_MAXL], *q[REDUCE_MAXL];
  uint32_t *pp[REDUCE_MAXL][2], *qq[REDUCE_MAXL][2];
  uint32_t m;
  uint64_t n_out;  // parents of the last layer, over all blocks
};
template <int D, bool TWO>
__global__ __launch_bounds__(BLOCK) void gkr_reduce_kernel(ReduceArgs a) {
  const uint64_t o = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  const uint32_t l = blockIdx.y;
  if (o >= a.n_out) return;
  const uint32_t top = TWO ? a.m - 1 : a.m;  // the last layer's
  const uint64_t half = (uint64_t)1 << a.m, b = o >> top, x = o & (((uint64_t)1 << top) - 1), c0 = (b << (a.m + 1)) + x;
  const Fraction<D> f0 = load_fraction<D>(a.p[l], a.q[l], c0), f1 = load_fraction<D>(a.p[l], a.q[l], c0 + half);
  if constexpr (TWO) {
    const uint64_t quarter = half / 2, at = (b << a.m) + x;
    const Fraction<D> f2 = load_fraction<D>(a.p[l], a.q[l], c0 + quarter), f3 = load_fraction<D>(a.p[l], a.q[l], c0 + half + quarter);
    const Fraction<D> g0 = add_fractions<D>(f0, f1), g1 = add_fractions<D>(f2, f3);
    store_fraction<D>(a.pp[l][0], a.qq[l][0], at, g0);
    store_fraction<D>(a.pp[l][0], a.qq[l][0], at + quarter, g1);
    store_fraction<D>(a.pp[l][1], a.qq[l][1], o, add_fractions<D>(g0, g1));
  } else {
    store_fraction<D>(a.pp[l][0], a.qq[l][0], o, add_fractions<D>(f0, f1));
  }
}

// The layers m_top .. 0 of a block of a lookup's tree, in one workgroup (block blockIdx.x of lookup blockIdx.y): layer m
// has 2^m <= BLOCK parents, a thread takes one, and the workgroup's barrier stands between a layer's writes and the next
// one's reads: nobody else reads them in this launch, so they need not leave the compute unit's XCD.  (With a device-wide
// fence every workgroup writes back its L2 behind every layer: blocks of 2^8, 64 of them 47 us and 16.5 without, 1024 of them
// 546 and 13.6; 16384 blocks of 2^4 3860 and 50.)  A launch per layer is 4 us each for a few hundred products; blocks beyond
// what the device holds at once are enough to fill it and leave most of a workgroup idle: 4096 of 2^4 16.6 us here and 8.5 in
// two launches, 16384 50 and 10, but 1024 of 2^8 13.6 here and 18.2 in four launches (REDUCE_TOP_BLOCKS).
constexpr int REDUCE_TOP_LAYERS = 9;     // m_top <= 8: 256 parents
constexpr int REDUCE_TOP_BLOCKS = 2048;  // eight workgroups a compute unit
struct ReduceTopArgs {
  // layer m_top + 1; where the tree over the block index begins, `valid` roots (the others are 0 / 1) that go to pad_p,
  // pad_q with them (else null: every child is there)
  const uint32_t *p[REDUCE_MAXL], *q[REDUCE_MAXL];
  uint32_t *pad_p[REDUCE_MAXL], *pad_q[REDUCE_MAXL];
  uint32_t *pp[REDUCE_MAXL][REDUCE_TOP_LAYERS], *qq[REDUCE_MAXL][REDUCE_TOP_LAYERS];
  int m_top;
  uint32_t valid;
};
template <int D>
__global__ __launch_bounds__(BLOCK) void gkr_reduce_top_kernel(ReduceTopArgs a) {
  static_assert((1 << (REDUCE_TOP_LAYERS - 1)) <= BLOCK, "a thread per parent");
  const uint32_t b = blockIdx.x, l = blockIdx.y;
  const uint32_t *p = a.p[l], *q = a.q[l];
  if (a.pad_p[l]) {
    for (uint32_t o = threadIdx.x; o < 2u << a.m_top; o += BLOCK) {
      store_ext<D>(a.pad_p[l] + o * D, o < a.valid ? load_ext<D>(p + o * D) : ext_zero<D>());
      store_ext<D>(a.pad_q[l] + o * D, o < a.valid ? load_ext<D>(q + o * D) : ext_lift<D>(1));
    }
    __syncthreads();
    p = a.pad_p[l], q = a.pad_q[l];
  }
  for (int m = a.m_top; m >= 0; m--) {
    const uint32_t half = 1u << m, x = threadIdx.x;
    const uint64_t o = ((uint64_t)b << m) + x, c0 = ((uint64_t)b << (m + 1)) + x;
    if (x < half) {
      const Fraction<D> f0 = load_fraction<D>(p, q, c0), f1 = load_fraction<D>(p, q, c0 + half);
      store_fraction<D>(a.pp[l][m], a.qq[l][m], o, add_fractions<D>(f0, f1));
    }
    __syncthreads();
    p = a.pp[l][m], q = a.qq[l][m];
  }
}

static int launch_reduce(int D, int K, int L, bool two, ReduceArgs &a) {
  Context &c = ctx();
  a.n_out = (uint64_t)K << (two ? a.m - 1 : a.m);
  const dim3 grid((uint32_t)((a.n_out + BLOCK - 1) / BLOCK), (uint32_t)L);
  if (D == 4)
    hipLaunchKernelGGL((two ? gkr_reduce_kernel<4, true> : gkr_reduce_kernel<4, false>), grid, dim3(BLOCK), 0, c.stream, a);
  else
    hipLaunchKernelGGL((two ? gkr_reduce_kernel<8, true> : gkr_reduce_kernel<8, false>), grid, dim3(BLOCK), 0, c.stream, a);
  EXH_HIP(hipGetLastError());
  return OK;
}
int gkr_reduce_layer(int D, int K, int m, const uint32_t *p, const uint32_t *q, uint32_t *pp, uint32_t *qq) {
  int status = ctx().require();
  if (status) return status;
  ReduceArgs a;
  memset(&a, 0, sizeof(a));
  a.p[0] = p, a.q[0] = q, a.pp[0][0] = pp, a.qq[0][0] = qq, a.m = (uint32_t)m;
  return launch_reduce(D, K, 1, false, a);
}

// the lower and upper halves of each block, as K contiguous blocks each (HALVES-PER-BLOCK,
// src/gkr.lisp:190-197); only needed when K > 1: with one block the halves are views
// (every vector of a layer in one launch: blockIdx.y picks the vector; the halves of vector i go to
// out + (2 i) n_out D and out + (2 i + 1) n_out D)
struct HalvesArgs {
  const uint32_t *v[MAXT];
  uint32_t *out;
  uint32_t size_bits;
  uint64_t n_out;
};
template <int D>
__global__ __launch_bounds__(BLOCK) void halves_kernel(HalvesArgs a) {
  uint64_t o = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (o >= a.n_out) return;
  const uint32_t *v = a.v[blockIdx.y];
  uint32_t *lower = a.out + (uint64_t)(2 * blockIdx.y) * a.n_out * D, *upper = lower + a.n_out * D;
  uint64_t size = (uint64_t)1 << a.size_bits, b = o >> a.size_bits, x = o & (size - 1);
  store_ext<D>(lower + o * D, load_ext<D>(v + (b * 2 * size + x) * D));
  store_ext<D>(upper + o * D, load_ext<D>(v + (b * 2 * size + size + x) * D));
}

// The same for every layer of a tree at once, in the order in which the tree's one allocation holds them: layer m, from
// n - 1 down to 0, has `vectors` vectors (p and q of each lookup) of K 2^m entries.  The halves of layer l + 1's vector i
// are tables 2 i and 2 i + 1 of layer l's sumcheck, at out + (2 vectors K (2^l - 1) + t K 2^l) D.  blockIdx.y: the vector.
template <int D>
__global__ __launch_bounds__(BLOCK) void all_halves_kernel(const uint32_t *tree, uint32_t *out, uint32_t K, int n,
                                                           uint64_t entries) {
  const uint64_t o = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (o >= entries) return;  // K (2^(n-1) - 1): layers 0 .. n - 2 one after the other
  const uint32_t layer = 31 - __clz((uint32_t)(o / K) + 1), vectors = gridDim.y;
  const uint64_t size = (uint64_t)1 << layer, at = o - K * (size - 1), b = at >> layer, x = at & (size - 1);
  const uint32_t *v = tree + (vectors * K * (((uint64_t)1 << n) - 4 * size) + blockIdx.y * K * 2 * size) * D;
  uint32_t *lower = out + (2 * vectors * K * (size - 1) + 2 * blockIdx.y * K * size) * D;
  store_ext<D>(lower + at * D, load_ext<D>(v + (b * 2 * size + x) * D));
  store_ext<D>(lower + (K * size + at) * D, load_ext<D>(v + (b * 2 * size + size + x) * D));
}

namespace {

int block_bits(int k) {  // src/gkr.lisp:23-25
  int b = 0;
  for (int v = k - 1; v > 0; v >>= 1) b++;
  return b;
}

// LAYER-STATEMENT (src/gkr.lisp:30-41) as a form; with_bw: (* bw statement)
Statement layer_statement(int lookups, bool with_bw) {
  std::string form = "(+";
  std::vector<std::string> tables, constants;
  if (with_bw) tables.push_back("BW");
  for (int l = 0; l < lookups; l++) {
    std::string s = std::to_string(l);
    form += " (* A" + s + " P0-" + s + " Q1-" + s + ") (* A" + s + " P1-" + s + " Q0-" + s + ") (* AL" + s + " Q0-" + s +
            " Q1-" + s + ")";
    for (const char *name : {"P0-", "P1-", "Q0-", "Q1-"}) tables.push_back(name + s);
    constants.push_back("A" + s);
    constants.push_back("AL" + s);
  }
  form += ")";
  if (with_bw) form = "(* BW " + form + ")";
  Statement st;
  compile_statement(form, tables, constants, &st);
  return st;
}

// a_l for each lookup from one challenge stream, then lambda; constants a_l, a_l lambda (:43-51)
void layer_challenges(Transcript &tr, int D, int L, std::vector<uint32_t> &consts, std::vector<hf::E> &as,
                      hf::E &lam) {
  std::vector<uint32_t> raw((size_t)L * D);
  tr.challenges(L, D, raw.data());
  lam.assign(D, 0);
  tr.challenge(D, lam.data());
  consts.assign((size_t)2 * L * D, 0);
  as.clear();
  for (int l = 0; l < L; l++) {
    hf::E a(raw.begin() + (size_t)l * D, raw.begin() + (size_t)(l + 1) * D);
    hf::E al = hf::mul(a, lam);
    memcpy(&consts[(size_t)(2 * l) * D], a.data(), 4 * D);
    memcpy(&consts[(size_t)(2 * l + 1) * D], al.data(), 4 * D);
    as.push_back(a);
  }
}

hf::E layer_claim(int D, const std::vector<hf::E> &as, const hf::E &lam, const std::vector<hf::E> &cp,
                  const std::vector<hf::E> &cq) {  // :53-55
  hf::E acc = hf::zero(D);
  for (size_t l = 0; l < as.size(); l++) acc = hf::add(acc, hf::mul(as[l], hf::add(cp[l], hf::mul(lam, cq[l]))));
  return acc;
}

hf::E fold_pair(const hf::E &lo, const hf::E &hi, const hf::E &r) { return hf::add(lo, hf::mul(r, hf::sub(hi, lo))); }

void next_claims(int D, int L, const uint32_t *finals, const hf::E &tt, std::vector<hf::E> &cp,
                 std::vector<hf::E> &cq) {  // :57-63
  for (int l = 0; l < L; l++) {
    const uint32_t *f = finals + (size_t)(4 * l) * D;
    cp[l] = fold_pair(hf::from(f, D), hf::from(f + D, D), tt);
    cq[l] = fold_pair(hf::from(f + 2 * D, D), hf::from(f + 3 * D, D), tt);
  }
}

hf::E padded_mass(int D, int lk, int K, const std::vector<uint32_t> &rb) {  // :68-71
  std::vector<uint32_t> e = hf::eq_table(rb.data(), lk, D);
  hf::E mass = hf::zero(D);
  for (size_t b = K; b < ((size_t)1 << lk); b++) mass = hf::add(mass, hf::from(&e[b * D], D));
  return mass;
}

std::vector<uint32_t> block_weights(int D, int K, const std::vector<uint32_t> &rb) {  // :73-77
  if (rb.empty()) {
    std::vector<uint32_t> one((size_t)D, 0);
    one[0] = 1;
    return one;
  }
  std::vector<uint32_t> e = hf::eq_table(rb.data(), (int)(rb.size() / D), D);
  e.resize((size_t)K * D);
  return e;
}

int send_finals(Transcript &tr, int D, int ntables, const uint32_t *finals, hf::E &tt) {  // :208-213
  uint64_t dims[2] = {1, (uint64_t)D};
  for (int t = 0; t < ntables; t++) {
    int status = tr.send(finals + (size_t)t * D, 2, dims, nullptr);
    if (status) return status;
  }
  tt.assign(D, 0);
  tr.challenge(D, tt.data());
  return OK;
}

// Frees what it allocated when the proof, or the part of it that the object belongs to, ends.
// (EXACTA_HIP_GKR_BUFFER_LIMIT=<bytes>, for tests: a thread's proof holds no more than that at a time, as if the device
// had no room for more.)
struct DeviceBuffers {
  static thread_local uint64_t live;  // bytes that the thread's objects hold
  uint64_t bytes = 0;
  std::vector<void *> owned;
  ~DeviceBuffers() {
    for (void *p : owned) ctx().pool.release(p);
    live -= bytes;
  }
  uint32_t *alloc(uint64_t words) {
    const char *limit = getenv("EXACTA_HIP_GKR_BUFFER_LIMIT");
    if (limit && live + words * 4 > strtoull(limit, nullptr, 10)) return nullptr;
    void *p = ctx().pool.alloc(words * 4);
    if (!p) return nullptr;
    owned.push_back(p);
    bytes += words * 4, live += words * 4;
    return (uint32_t *)p;
  }
};
thread_local uint64_t DeviceBuffers::live = 0;

constexpr size_t GKR_BW_PIN = 8192, GKR_BW_PIN_WORDS = 1024;  // words of the context's pinned buffer (see below)

// a layer of K blocks can be chained: see gkr_prove_upper
bool blocks_chain(int K, int L, int D) {
  const uint64_t pairs = SumcheckSession::one_workgroup_pairs(4 * L, D), block_pairs = SumcheckSession::one_workgroup_pairs(4 * L + 1, D);
  return K > 1 && K <= GLUE_MAXBLOCKS && (uint64_t)K <= pairs && ((uint64_t)1 << block_bits(K)) / 2 <= block_pairs;
}

// what the chain's sticky word means for the proof (host side)
int chain_outcome(uint32_t failed) {
  if (!failed) return OK;
  set_error("device-error: a chained layer's sumcheck did not complete (a workgroup gave up waiting, or rounds are "
            "missing); the proof is void");
  return E_DEVICE;
}

// PROVE-UPPER's layers, and with several blocks the tree over the block index before them, chained on the device (see
// gkr_glue.hpp): every launch of every sumcheck is enqueued at once, the host waits once and reads the log.
// `held`: the finished layer's last launch (its rounds in one workgroup), not enqueued yet: the step rides on it
// (tail_glue_kernel); empty: the step is a launch of its own.
template <int D>
static int launch_glue(const GlueArgs<D> &a, std::vector<uint8_t> *held = nullptr, const KernelSet *kernels = nullptr) {
  Context &c = ctx();
  if (held && !held->empty() && kernels && kernels->launch_tail_glue) {
    c.prof_begin("tail", a.prev_rounds, 0);
    kernels->launch_tail_glue(held->data(), &a, c.stream);
    c.prof_end();
    held->clear();
    EXH_HIP(hipGetLastError());
    return OK;
  }
  c.prof_begin("gkr_glue", a.n, 0);
  hipLaunchKernelGGL(gkr_glue_kernel<D>, dim3(1), dim3(BLOCK), 0, c.stream, a);
  c.prof_end();
  EXH_HIP(hipGetLastError());
  return OK;
}

// The tables of the layers' sumchecks, on the device: of the tree over the block index (several blocks; lk layers), and of
// the layers in the blocks (n - 1).
struct ChainTables {
  std::vector<const uint32_t *> roots;  // p and q of every lookup
  std::vector<std::vector<const uint32_t *>> top, layers;
};

template <int D>
static int prove_upper_chained(Transcript &tr, int n, int K, int lk, int L, const ChainTables &tables,
                               const std::string &label, uint32_t *out_ri, uint32_t *out_rb, uint32_t *out_cp,
                               uint32_t *out_cq) {
  Context &c = ctx();
  const int NT = 4 * L;
  const Statement st = layer_statement(L, false), st_blk = K > 1 ? layer_statement(L, true) : Statement();
  // The sumchecks in their order, and where each one's messages, challenges and -- unless it is a layer's own with several
  // blocks -- finals and fresh point lie in the log, behind the roots.
  enum Kind { TOP, LAYER, BLOCKS };
  struct Step {
    Kind kind;
    int layer, rounds, points;
    bool finals;
    size_t log_at;
    std::string header;
    const std::vector<const uint32_t *> *tabs;  // (BLOCKS: what the layer's rounds leave)
  };
  std::vector<Step> steps;
  size_t words = (size_t)2 * L * D;
  auto add_step = [&](Kind kind, int layer, const std::string &name, int rounds, int degree, int blocks,
                      const std::vector<const uint32_t *> *tabs) {
    Step s{kind, layer, rounds, degree > 1 ? degree : 1, kind != LAYER || K == 1, words,
           header_bytes(name, rounds, degree, blocks), tabs};
    words += (size_t)rounds * s.points * D + (size_t)rounds * D + (s.finals ? (size_t)NT * D + D : 0);
    steps.push_back(s);
  };
  for (size_t j = 0; j < tables.top.size(); j++) add_step(TOP, (int)j, label + "-top", (int)j, j > 0 ? 2 : 0, 1, &tables.top[j]);
  for (size_t j = 0; j < tables.layers.size(); j++) {
    add_step(LAYER, (int)j, label, (int)j, j > 0 ? 2 : 0, K, &tables.layers[j]);
    if (K > 1) add_step(BLOCKS, (int)j, label + "-blk", lk, st_blk.degree, 1, nullptr);
  }
  for (const Step &s : steps)
    if (s.header.size() > 64) {
      set_error("invalid-parameter: label too long for the chained layers");
      return E_PARAM;
    }
  DeviceBuffers bufs;
  GkrChainState *chain = reinterpret_cast<GkrChainState *>(bufs.alloc((sizeof(GkrChainState) + 3) / 4));
  uint32_t *d_log = bufs.alloc(words), *d_bw = K > 1 ? bufs.alloc((size_t)K * D) : nullptr;
  if (!chain || !d_log || (K > 1 && !d_bw)) {
    set_error("device-out-of-memory: the GKR chain's log");
    return E_NOMEM;
  }
  const DevB3S first = device_state(tr);
  // the log comes to the host as the loop's logs of a single sumcheck do (three copies and a wait on the stream are 40 us)
  const bool deliver = c.host_pinned_dev && !c.profiling && words + sizeof(DevB3S) / 4 + 2 <= PIN_DOWN_WORDS;
  volatile uint32_t *flag = c.host_pinned + PIN_DOWN + words + sizeof(DevB3S) / 4 + 1;
  const std::vector<int> strides(NT + 1, D);
  const std::vector<uint32_t> no_point((size_t)std::max(n, lk) * D, 0), no_consts((size_t)2 * L * D, 0), no_bw((size_t)K * D, 0);
  std::vector<const uint32_t *> blk_tabs(NT + 1, nullptr);
  auto begin_step = [&](SumcheckSession &s, const Step &step) {
    if (step.kind == BLOCKS)
      return s.begin(st_blk, D, lk, blk_tabs.data(), strides.data(), nullptr, nullptr, 1, no_consts.data(), -1, false, true);
    const bool blocks = step.kind == LAYER && K > 1;
    return s.begin(st, D, step.rounds, step.tabs->data(), strides.data(), no_point.data(), blocks ? no_bw.data() : nullptr,
                   blocks ? K : 1, no_consts.data(), step.rounds > 0 ? 2 : 0, false, true);
  };
  int status;
  // the largest sumchecks first, for their buffers alone: the arenas then never grow (and never wait) mid-chain
  for (size_t i = steps.size() - 1, kinds = 0; kinds < 2 && i < steps.size(); i--, kinds++) {
    SumcheckSession widest;
    if ((status = begin_step(widest, steps[i]))) return status;
  }
  if (!tables.top.empty()) {
    SumcheckSession widest;
    if ((status = begin_step(widest, steps[tables.top.size() - 1]))) return status;
  }
  const Ctrl *prev_ctrl = nullptr;
  std::vector<const uint32_t *> prev_tabs;
  const DevB3S unused_state = first;
  // a sumcheck's last launch waits here for the next step, which rides on it (EXACTA_HIP_NO_GKR_FUSE=1: never)
  std::vector<uint8_t> held;
  const KernelSet *held_kernels = nullptr;
  const char *no_fuse = getenv("EXACTA_HIP_NO_GKR_FUSE");
  const bool fuse = !(no_fuse && no_fuse[0] == '1');
  for (size_t i = 0; i <= steps.size(); i++) {  // launch i closes sumcheck i - 1 and opens sumcheck i; the last only closes
    GlueArgs<D> a;
    memset(&a, 0, sizeof(a));
    a.chain = chain, a.L = L, a.NT = NT, a.K = 1;
    if (i == 0) {
      a.close_kind = 1, a.log = d_log, a.start = first;
      for (int t = 0; t < 2 * L; t++) a.tabs[t] = tables.roots[t];
    } else {
      const Step &prev = steps[i - 1];
      a.prev_rounds = prev.rounds, a.prev_points = prev.points, a.log = d_log + prev.log_at;
      if (prev.rounds > 0) {
        a.close_kind = prev.finals ? 2 : 4, a.prev_ctrl = prev_ctrl;
      } else if (prev.finals) {  // no rounds: its finals are its tables' single entries
        a.close_kind = 3;
        for (int t = 0; t < NT; t++) a.tabs[t] = prev_tabs[t];
      }
      if (prev.kind == BLOCKS) a.fin_skip = 1, a.blocks_closed = 1, a.tt_at = prev.layer;
    }
    if (i == steps.size()) {
      if (deliver) {
        if (++c.log_seq == 0) ++c.log_seq;  // 0 is what the flag is reset to
        a.log_all = d_log, a.log_words = (uint32_t)words, a.host_log = c.host_pinned_dev + PIN_DOWN, a.host_seq = c.log_seq;
        *flag = 0;
      }
      if ((status = launch_glue<D>(a, &held, held_kernels))) return status;
      break;
    }
    const Step &step = steps[i];
    a.open = step.kind == BLOCKS ? 2 : 1, a.n = step.rounds, a.header_len = (int)step.header.size();
    for (size_t k = 0; k < step.header.size(); k++) a.header[k / 4] |= (uint32_t)(uint8_t)step.header[k] << (8 * (k % 4));
    if (step.kind != TOP) a.K = K, a.lk = lk, a.bw_table = d_bw;
    if (step.kind == BLOCKS) {
      blk_tabs[0] = d_bw;
      for (int t = 0; t < NT; t++) blk_tabs[t + 1] = prev_tabs[t];
    }
    if (step.rounds == 0) {
      if ((status = launch_glue<D>(a, &held, held_kernels))) return status;
      prev_tabs = *step.tabs;
      continue;
    }
    SumcheckSession s;
    if ((status = begin_step(s, step))) return status;
    std::vector<uint32_t> lagfix;
    std::vector<int> acc_group;
    s.message_map_scalars(&lagfix, &acc_group);
    a.points = s.points, a.nacc = std::max(s.st.nacc, 1), a.c0_words = step.rounds * s.points * D;
    if ((int)lagfix.size() > MAXPTS * MAXACC || !s.setup_deferred || s.points != step.points) {
      set_error("invalid-parameter: layer statement beyond the chained layers' limits");
      return E_PARAM;
    }
    memcpy(a.lagfix, lagfix.data(), lagfix.size() * 4);
    for (int e = 0; e < a.nacc; e++) {
      const Group *g = acc_group[e] >= 0 ? &s.st.groups[acc_group[e]] : nullptr;
      if (!g || g->parts.size() != 1 || g->parts[0].coeff != 1 || g->parts[0].consts.size() != 1 ||
          g->parts[0].consts[0] >= GLUE_MAXCONST) {
        set_error("invalid-parameter: layer statement beyond the chained layers' limits");
        return E_PARAM;
      }
      a.acc_const[e] = (uint8_t)g->parts[0].consts[0];
    }
    a.factors = s.d_weights, a.mtilde = s.d_mtilde, a.c0 = s.d_c0, a.ctrl = s.d_ctrl;
    if (step.kind == LAYER && K > 1) a.bw = s.d_weights + (size_t)2 * step.rounds * D;  // (the block weights follow the factors)
    if (step.kind == BLOCKS) s.valid_entries = (uint64_t)K;
    // (the step that opens this sumcheck rides on the last launch of the one before, when that was held back)
    std::vector<uint8_t> held_now;
    s.chain_hook = [&]() { return launch_glue<D>(a, &held, held_kernels); };
    if (fuse) s.held_tail = &held_now;
    if ((status = s.run_device(unused_state, nullptr, nullptr, nullptr))) return status;
    held.swap(held_now);
    held_kernels = s.kernels;
    prev_ctrl = s.d_ctrl;
    prev_tabs = s.cur;
  }
  // ---- one wait, then the log: polled in pinned memory, where the last step wrote it, or copied
  std::vector<uint32_t> log(words);
  DevB3S last;
  uint32_t failed = 0;
  if (deliver) {
    // (a stream that ends without raising the flag, or is in an error state, ends the polling)
    uint32_t spins = 0;
    while (*flag != c.log_seq)
      if ((++spins & 1023) == 0 && hipStreamQuery(c.stream) != hipErrorNotReady) break;
    if (*flag != c.log_seq) {
      EXH_HIP(hipStreamSynchronize(c.stream));
      if (*flag != c.log_seq) {
        set_error("device-error: the chained layers ended without delivering their log");
        return E_DEVICE;
      }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    const uint32_t *down = c.host_pinned + PIN_DOWN;
    memcpy(log.data(), down, words * 4);
    memcpy(&last, down + words, sizeof(last));
    failed = down[words + sizeof(last) / 4];
  } else {
    EXH_HIP(hipMemcpyAsync(log.data(), d_log, words * 4, hipMemcpyDeviceToHost, c.stream));
    EXH_HIP(hipMemcpyAsync(&last, &chain->tr, sizeof(last), hipMemcpyDeviceToHost, c.stream));
    EXH_HIP(hipMemcpyAsync(&failed, &chain->failed, sizeof(failed), hipMemcpyDeviceToHost, c.stream));
    EXH_HIP(hipStreamSynchronize(c.stream));
  }
  if ((status = chain_outcome(failed))) return status;
  // the messages as they were sent, recorded without hashing them again; the transcript takes the device's state
  uint64_t dims[2] = {2, (uint64_t)D};
  for (int l = 0; l < L; l++)
    if ((status = tr.send(&log[(size_t)l * 2 * D], 2, dims, nullptr, false))) return status;
  const uint32_t *fin = nullptr, *tt = nullptr, *rho = nullptr, *block_rho = nullptr;
  for (const Step &step : steps) {
    const uint32_t *msg = &log[step.log_at], *chal = msg + (size_t)step.rounds * step.points * D;
    (step.kind == BLOCKS ? block_rho : rho) = chal;
    dims[0] = (uint64_t)step.points;
    for (int j = 0; j < step.rounds; j++)
      if ((status = tr.send(msg + (size_t)j * step.points * D, 2, dims, nullptr, false))) return status;
    if (!step.finals) continue;
    fin = chal + (size_t)step.rounds * D;
    tt = fin + (size_t)NT * D;
    dims[0] = 1;
    for (int t = 0; t < NT; t++)
      if ((status = tr.send(fin + (size_t)t * D, 2, dims, nullptr, false))) return status;
  }
  if ((status = adopt_device_state(tr, last))) return status;
  if (out_ri) {
    memcpy(out_ri, rho, (size_t)(n - 2) * D * 4);
    memcpy(out_ri + (size_t)(n - 2) * D, tt, (size_t)D * 4);
  }
  if (out_rb && K > 1) memcpy(out_rb, block_rho, (size_t)lk * D * 4);
  std::vector<hf::E> cp(L), cq(L);
  next_claims(D, L, fin, hf::from(tt, D), cp, cq);
  for (int l = 0; l < L; l++) {
    if (out_cp) memcpy(out_cp + (size_t)l * D, cp[l].data(), 4 * D);
    if (out_cq) memcpy(out_cq + (size_t)l * D, cq[l].data(), 4 * D);
  }
  return OK;
}

}  // namespace

int gkr_prove_upper(Transcript &tr, int n, int K, int L, const uint32_t *const *leaves, const std::string &label,
                    uint32_t *out_ri, uint32_t *out_rb, uint32_t *out_cp, uint32_t *out_cq) {
  Context &c = ctx();
  int status = c.require();
  if (status) return status;
  int D = tr.D, lk = block_bits(K), NT = 4 * L;
  if (L < 1 || NT + 1 > MAXT || n < 0 || n > 30 || K < 1) {
    set_error("invalid-parameter: GKR shape");
    return E_PARAM;
  }
  uint64_t Kp = (uint64_t)1 << lk;
  DeviceBuffers bufs;
  // FRACTION-TREES: every in-block layer, bottom up, kept on the device
  std::vector<std::vector<const uint32_t *>> layers(n + 1, std::vector<const uint32_t *>(2 * L));
  for (int i = 0; i < 2 * L; i++) layers[n][i] = leaves[i];
  // one allocation holds every layer above the leaves: 2 L K (2^n - 1) entries
  if ((status = c.tree.reserve(((((uint64_t)K << n) - K) * 2 * L * D + 64) * 4))) return status;
  uint32_t *next = (uint32_t *)c.tree.ptr;
  // these layers in one launch (-1: none)
  const int m_top = (uint64_t)K * L <= (uint64_t)REDUCE_TOP_BLOCKS ? std::min(n - 1, REDUCE_TOP_LAYERS - 1) : -1;
  for (int m = n - 1; m >= 0; m--)
    for (int l = 0; l < L; l++) {
      uint64_t words = ((uint64_t)K << m) * D;
      uint32_t *pp = next, *qq = next + words;
      next += 2 * words;
      layers[m][2 * l] = pp;
      layers[m][2 * l + 1] = qq;
    }
  for (int m = n - 1; m > m_top;) {
    const bool two = m - 1 > m_top;
    ReduceArgs a;
    memset(&a, 0, sizeof(a));
    a.m = (uint32_t)m;
    for (int l = 0; l < L; l++) {
      a.p[l] = layers[m + 1][2 * l], a.q[l] = layers[m + 1][2 * l + 1];
      for (int k = 0; k < (two ? 2 : 1); k++)
        a.pp[l][k] = const_cast<uint32_t *>(layers[m - k][2 * l]), a.qq[l][k] = const_cast<uint32_t *>(layers[m - k][2 * l + 1]);
    }
    if ((status = launch_reduce(D, K, L, two, a))) return status;
    m -= two ? 2 : 1;
  }
  auto reduce_top = [&](const ReduceTopArgs &a, int blocks) {
    if (D == 4)
      hipLaunchKernelGGL(gkr_reduce_top_kernel<4>, dim3(blocks, L), dim3(BLOCK), 0, c.stream, a);
    else
      hipLaunchKernelGGL(gkr_reduce_top_kernel<8>, dim3(blocks, L), dim3(BLOCK), 0, c.stream, a);
  };
  if (m_top >= 0) {
    ReduceTopArgs a;
    memset(&a, 0, sizeof(a));
    a.m_top = m_top;
    for (int l = 0; l < L; l++) {
      a.p[l] = layers[m_top + 1][2 * l], a.q[l] = layers[m_top + 1][2 * l + 1];
      for (int m = m_top; m >= 0; m--)
        a.pp[l][m] = const_cast<uint32_t *>(layers[m][2 * l]), a.qq[l][m] = const_cast<uint32_t *>(layers[m][2 * l + 1]);
    }
    reduce_top(a, K);
    EXH_HIP(hipGetLastError());
  }
  const char *host_rounds = getenv("EXACTA_HIP_HOST_ROUNDS"), *no_chain = getenv("EXACTA_HIP_NO_GKR_CHAIN");
  const bool chains = L * D <= 12 && 2 * L <= GLUE_MAXCONST && !(host_rounds && host_rounds[0] == '1') &&
                      !(no_chain && no_chain[0] == '1');
  // All layers chained on the device, one wait for the whole proof.  With several blocks as long as a lane holds a block in
  // the step that forms their weights, and the one-workgroup launch the last round's pairs (and the tables over the block
  // index): beyond that a layer is two device-driven sumchecks with a wait each, as below.  That way and this one, us: three
  // blocks of 2^14 and two lookups 1900 and 1310, five of 2^10 1100 and 745, 64 of 2^8 1130 and 830, 33 of 2^10 and three
  // lookups 3900 and 2330.  The chain holds every layer's tables at once, as many bytes as the tree again: where there is no
  // room for them the layers go one at a time as well (nothing has been sent by then), in the largest one's memory, half of
  // that.
  if (chains && n >= 2 && n - 2 <= MAXROUNDS && (K == 1 || blocks_chain(K, L, D))) {
    DeviceBuffers held;
    uint32_t *d_top = K > 1 ? held.alloc(2 * Kp * 2 * L * D) : nullptr;
    uint32_t *d_halves = K > 1 ? held.alloc((uint64_t)NT * K * (((uint64_t)1 << (n - 1)) - 1) * D) : nullptr;
    ChainTables tables;
    auto halves = [&](const std::vector<const uint32_t *> &vectors, uint64_t size) {  // with one block they are views
      std::vector<const uint32_t *> tabs(NT);
      for (int i = 0; i < 2 * L; i++) tabs[2 * i] = vectors[i], tabs[2 * i + 1] = vectors[i] + size * D;
      return tabs;
    };
    if (K == 1) {
      tables.roots = layers[0];
      for (int layer = 0; layer < n - 1; layer++) tables.layers.push_back(halves(layers[layer + 1], (uint64_t)1 << layer));
    } else if (!d_top || !d_halves) {
      status = E_NOMEM;
    } else {
      // the tree over the block index, its lowest layer padded with 0 / 1 (2^lk roots)
      ReduceTopArgs a;
      memset(&a, 0, sizeof(a));
      a.m_top = lk - 1, a.valid = (uint32_t)K;
      std::vector<std::vector<const uint32_t *>> top(lk + 1, std::vector<const uint32_t *>(2 * L));
      for (int l = 0; l < L; l++) {
        a.p[l] = layers[0][2 * l], a.q[l] = layers[0][2 * l + 1];
        for (int m = lk; m >= 0; m--) {
          uint32_t *pp = d_top, *qq = pp + ((uint64_t)D << m);
          d_top = qq + ((uint64_t)D << m);
          (m == lk ? a.pad_p[l] : a.pp[l][m]) = pp, (m == lk ? a.pad_q[l] : a.qq[l][m]) = qq;
          top[m][2 * l] = pp, top[m][2 * l + 1] = qq;
        }
      }
      reduce_top(a, 1);
      EXH_HIP(hipGetLastError());
      tables.roots = top[0];
      for (int j = 0; j < lk; j++) tables.top.push_back(halves(top[j + 1], (uint64_t)1 << j));
      const uint64_t entries = (uint64_t)K * (((uint64_t)1 << (n - 1)) - 1);
      const dim3 grid((uint32_t)((entries + BLOCK - 1) / BLOCK), 2 * L);
      const uint32_t *tree = (const uint32_t *)c.tree.ptr;
      if (D == 4)
        hipLaunchKernelGGL(all_halves_kernel<4>, grid, dim3(BLOCK), 0, c.stream, tree, d_halves, (uint32_t)K, n, entries);
      else
        hipLaunchKernelGGL(all_halves_kernel<8>, grid, dim3(BLOCK), 0, c.stream, tree, d_halves, (uint32_t)K, n, entries);
      EXH_HIP(hipGetLastError());
      for (int layer = 0; layer < n - 1; layer++) {
        const uint64_t n_out = (uint64_t)K << layer;
        std::vector<const uint32_t *> tabs(NT);
        for (int t = 0; t < NT; t++) tabs[t] = d_halves + ((uint64_t)NT * (n_out - K) + t * n_out) * D;
        tables.layers.push_back(tabs);
      }
    }
    if (status == OK)
      status = D == 4 ? prove_upper_chained<4>(tr, n, K, lk, L, tables, label, out_ri, out_rb, out_cp, out_cq)
                      : prove_upper_chained<8>(tr, n, K, lk, L, tables, label, out_ri, out_rb, out_cp, out_cq);
    if (status != E_NOMEM || K == 1) return status;
  }
  if (status == E_NOMEM) {
    (void)hipGetLastError();  // (the refused allocation's)
    c.pool.trim();
    status = OK;
  }
  // With several blocks a layer's halves and the blocks' values after its rounds, in memory that the layers take in turn (a
  // layer's launches are done before the next one's are enqueued); had before anything is sent.
  uint32_t *d_halves = nullptr, *d_blk = nullptr;
  if (K > 1 && n >= 2) {
    d_halves = bufs.alloc(((uint64_t)NT * K << (n - 2)) * D), d_blk = bufs.alloc((uint64_t)(NT + 1) * Kp * D);
    if (!d_halves || !d_blk) {
      set_error("device-out-of-memory: the tables of a layer of several blocks");
      return E_NOMEM;
    }
  }
  // the per-block roots, and the top tree over the block index on the host (2^lk entries)
  std::vector<std::vector<std::vector<uint32_t>>> top(lk + 1, std::vector<std::vector<uint32_t>>(2 * L));
  EXH_HIP(hipStreamSynchronize(c.stream));
  for (int l = 0; l < L; l++) {
    std::vector<uint32_t> p(Kp * D, 0), q(Kp * D, 0);
    EXH_HIP(hipMemcpy(p.data(), layers[0][2 * l], (size_t)K * D * 4, hipMemcpyDeviceToHost));
    EXH_HIP(hipMemcpy(q.data(), layers[0][2 * l + 1], (size_t)K * D * 4, hipMemcpyDeviceToHost));
    for (uint64_t b = K; b < Kp; b++) q[b * D] = 1;  // padded with 0/1
    top[lk][2 * l] = p;
    top[lk][2 * l + 1] = q;
  }
  for (int j = lk - 1; j >= 0; j--)
    for (int l = 0; l < L; l++) {
      uint64_t len = (uint64_t)1 << j;
      const std::vector<uint32_t> &p = top[j + 1][2 * l], &q = top[j + 1][2 * l + 1];
      std::vector<uint32_t> pp(len * D), qq(len * D);
      for (uint64_t b = 0; b < len; b++) {
        hf::E p0 = hf::from(&p[b * D], D), p1 = hf::from(&p[(b + len) * D], D);
        hf::E q0 = hf::from(&q[b * D], D), q1 = hf::from(&q[(b + len) * D], D);
        hf::E np = hf::add(hf::mul(p0, q1), hf::mul(p1, q0)), nq = hf::mul(q0, q1);
        memcpy(&pp[b * D], np.data(), 4 * D);
        memcpy(&qq[b * D], nq.data(), 4 * D);
      }
      top[j][2 * l] = pp;
      top[j][2 * l + 1] = qq;
    }

  Statement st = layer_statement(L, false), st_blk = layer_statement(L, true);
  std::vector<hf::E> cp(L), cq(L), as;
  hf::E lam, tt;
  std::vector<uint32_t> consts, finals((size_t)(NT + 1) * D), rho((size_t)(n + lk + 1) * D);
  std::vector<uint32_t> r, ri;
  uint64_t dims2[2] = {2, (uint64_t)D};
  std::vector<int> strides(NT + 1, D);
  // The top tree is a tree of one block over the block index: its roots and layers are PROVE-UPPER's with one
  // block under the label's "-top", so the chain above serves it as well (one wait instead of one per layer).
  bool top_chained = false;
  if (chains && lk >= 1 && lk - 1 <= MAXROUNDS) {
    // every level of every lookup's top tree in one buffer, one copy
    ChainTables tables;
    std::vector<uint32_t> all;
    std::vector<std::vector<size_t>> at(lk + 1, std::vector<size_t>(2 * L));
    for (int j = 0; j <= lk; j++)
      for (int i = 0; i < 2 * L; i++) {
        at[j][i] = all.size();
        all.insert(all.end(), top[j][i].begin(), top[j][i].end());
      }
    uint32_t *d_top = bufs.alloc(all.size());
    if (!d_top) return E_NOMEM;
    EXH_HIP(hipMemcpyAsync(d_top, all.data(), all.size() * 4, hipMemcpyHostToDevice, c.stream));
    for (int i = 0; i < 2 * L; i++) tables.roots.push_back(d_top + at[0][i]);
    for (int j = 0; j < lk; j++) {
      std::vector<const uint32_t *> tabs(NT);
      for (int i = 0; i < 2 * L; i++) tabs[2 * i] = d_top + at[j + 1][i], tabs[2 * i + 1] = tabs[2 * i] + ((size_t)D << j);
      tables.layers.push_back(tabs);
    }
    r.assign((size_t)lk * D, 0);
    std::vector<uint32_t> ocp((size_t)L * D), ocq((size_t)L * D);
    status = D == 4 ? prove_upper_chained<4>(tr, lk + 1, 1, 0, L, tables, label + "-top", r.data(), nullptr, ocp.data(), ocq.data())
                    : prove_upper_chained<8>(tr, lk + 1, 1, 0, L, tables, label + "-top", r.data(), nullptr, ocp.data(), ocq.data());
    if (status) return status;
    for (int l = 0; l < L; l++) {
      cp[l] = hf::from(&ocp[(size_t)l * D], D);
      cq[l] = hf::from(&ocq[(size_t)l * D], D);
    }
    top_chained = true;
  }
  if (!top_chained) {
    for (int l = 0; l < L; l++) {  // the roots
      uint32_t root[16];
      memcpy(root, top[0][2 * l].data(), 4 * D);
      memcpy(root + D, top[0][2 * l + 1].data(), 4 * D);
      if ((status = tr.send(root, 2, dims2, nullptr))) return status;
      cp[l] = hf::from(root, D);
      cq[l] = hf::from(root + D, D);
    }
  }
  for (int j = 0; j < lk && !top_chained; j++) {  // the top tree, layer by layer
    layer_challenges(tr, D, L, consts, as, lam);
    uint64_t size = (uint64_t)1 << j;
    std::vector<const uint32_t *> tabs(NT);
    for (int l = 0; l < L; l++)
      for (int w = 0; w < 2; w++) {
        uint32_t *d = bufs.alloc(2 * size * D);
        if (!d) return E_NOMEM;
        EXH_HIP(hipMemcpy(d, top[j + 1][2 * l + w].data(), 2 * size * D * 4, hipMemcpyHostToDevice));
        tabs[4 * l + 2 * w] = d;                 // lower half: children b
        tabs[4 * l + 2 * w + 1] = d + size * D;  // upper half: children b + 2^j
      }
    status = sumcheck_prove(tr, j, st, tabs.data(), strides.data(), j > 0 ? r.data() : nullptr, consts.data(),
                            label + "-top", nullptr, 1, j > 0 ? 2 : 0, rho.data(), finals.data(), nullptr);
    if (status) return status;
    if ((status = send_finals(tr, D, NT, finals.data(), tt))) return status;
    next_claims(D, L, finals.data(), tt, cp, cq);
    r.assign(rho.begin(), rho.begin() + (size_t)j * D);
    r.insert(r.end(), tt.begin(), tt.end());
  }
  std::vector<uint32_t> rb = r;
  if (Kp != (uint64_t)K) {
    hf::E mass = padded_mass(D, lk, K, rb);
    for (int l = 0; l < L; l++) cq[l] = hf::sub(cq[l], mass);
  }
  for (int layer = 0; layer < n - 1; layer++) {  // the in-block layers
    layer_challenges(tr, D, L, consts, as, lam);
    std::vector<uint32_t> bw = block_weights(D, K, rb);
    uint64_t size = (uint64_t)1 << layer;
    std::vector<const uint32_t *> tabs(NT);
    if (K == 1) {  // the halves are views
      for (int l = 0; l < L; l++)
        for (int w = 0; w < 2; w++) {
          const uint32_t *v = layers[layer + 1][2 * l + w];
          tabs[4 * l + 2 * w] = v;
          tabs[4 * l + 2 * w + 1] = v + size * D;
        }
    } else {  // one launch splits the layer's 2 L vectors
      const uint64_t n_out = K * size;
      HalvesArgs h;
      memset(&h, 0, sizeof(h));
      h.out = d_halves;
      h.size_bits = (uint32_t)layer, h.n_out = n_out;
      for (int i = 0; i < 2 * L; i++) {
        h.v[i] = layers[layer + 1][i];
        tabs[2 * i] = h.out + (uint64_t)(2 * i) * n_out * D;
        tabs[2 * i + 1] = h.out + (uint64_t)(2 * i + 1) * n_out * D;
      }
      const dim3 grid((uint32_t)((n_out + BLOCK - 1) / BLOCK), (uint32_t)(2 * L));
      if (D == 4)
        hipLaunchKernelGGL(halves_kernel<4>, grid, dim3(BLOCK), 0, c.stream, h);
      else
        hipLaunchKernelGGL(halves_kernel<8>, grid, dim3(BLOCK), 0, c.stream, h);
      EXH_HIP(hipGetLastError());
    }
    // With several blocks the folded tables (one entry per block) stay on the device, zero padded to 2^lk, as the
    // tables of the sumcheck over the block index; the weights, padded alike, go before them in one copy.
    status = sumcheck_prove(tr, layer, st, tabs.data(), strides.data(), layer > 0 ? ri.data() : nullptr,
                            consts.data(), label, bw.data(), K, layer > 0 ? 2 : 0, rho.data(),
                            lk > 0 ? nullptr : finals.data(), nullptr, lk > 0 ? d_blk + Kp * D : nullptr, Kp);
    if (status) return status;
    std::vector<uint32_t> rbn;
    if (lk > 0) {  // bind the block index: the blocks' values and weights, padded with zeros
      std::vector<const uint32_t *> btabs(NT + 1);
      std::vector<uint32_t> bwp(Kp * D, 0);
      memcpy(bwp.data(), bw.data(), (size_t)K * D * 4);
      for (int t = 0; t <= NT; t++) btabs[t] = d_blk + (uint64_t)t * Kp * D;
      // the weights' table: read by the sumcheck's first launch from pinned memory where the host puts it (a part
      // of the context's buffer nothing else uses; the host waits for this sumcheck before it writes there again),
      // or copied beside the blocks' values when it is longer than that part
      if (Kp * D <= GKR_BW_PIN_WORDS && c.host_pinned_dev) {
        memcpy(c.host_pinned + GKR_BW_PIN, bwp.data(), Kp * D * 4);
        btabs[0] = c.host_pinned_dev + GKR_BW_PIN;
      } else {
        EXH_HIP(hipMemcpy(d_blk, bwp.data(), Kp * D * 4, hipMemcpyHostToDevice));
      }
      std::vector<uint32_t> f2((size_t)(NT + 1) * D);
      rbn.assign((size_t)lk * D, 0);
      status = sumcheck_prove(tr, lk, st_blk, btabs.data(), strides.data(), nullptr, consts.data(), label + "-blk",
                              nullptr, 1, -1, rbn.data(), f2.data(), nullptr);
      if (status) return status;
      memcpy(finals.data(), f2.data() + D, (size_t)NT * D * 4);  // bw's final comes first
    }
    if ((status = send_finals(tr, D, NT, finals.data(), tt))) return status;
    next_claims(D, L, finals.data(), tt, cp, cq);
    ri.assign(rho.begin(), rho.begin() + (size_t)layer * D);
    ri.insert(ri.end(), tt.begin(), tt.end());
    rb = rbn;
  }
  if (out_ri && !ri.empty()) memcpy(out_ri, ri.data(), ri.size() * 4);
  if (out_rb && !rb.empty()) memcpy(out_rb, rb.data(), rb.size() * 4);
  for (int l = 0; l < L; l++) {
    if (out_cp) memcpy(out_cp + (size_t)l * D, cp[l].data(), 4 * D);
    if (out_cq) memcpy(out_cq + (size_t)l * D, cq[l].data(), 4 * D);
  }
  EXH_HIP(hipStreamSynchronize(c.stream));
  return OK;
}

int gkr_verify_upper(Transcript &tr, int n, int K, int L, const std::string &label, uint32_t *out_roots,
                     uint32_t *out_ri, uint32_t *out_rb, uint32_t *out_cp, uint32_t *out_cq) {
  int D = tr.D, lk = block_bits(K), NT = 4 * L, status;
  if (L < 1 || NT + 1 > MAXT || n < 0 || K < 1) {
    set_error("invalid-parameter: GKR shape");
    return E_PARAM;
  }
  uint64_t Kp = (uint64_t)1 << lk;
  std::vector<hf::E> cp(L), cq(L), as;
  hf::E lam, tt;
  uint64_t dims2[2] = {2, (uint64_t)D}, dims1[2] = {1, (uint64_t)D};
  for (int l = 0; l < L; l++) {
    uint32_t root[16];
    if ((status = tr.send(nullptr, 2, dims2, root))) return status;
    if (out_roots) memcpy(out_roots + (size_t)l * 2 * D, root, 8 * D);
    cp[l] = hf::from(root, D);
    cq[l] = hf::from(root + D, D);
  }
  Statement st = layer_statement(L, false), st_blk = layer_statement(L, true);
  std::vector<uint32_t> consts, finals((size_t)NT * D), rho((size_t)(n + lk + 1) * D), r, ri, rb;
  uint32_t reduced[8], expected[8];
  auto receive_finals = [&]() -> int {  // :84-89
    for (int t = 0; t < NT; t++) {
      int s = tr.send(nullptr, 2, dims1, &finals[(size_t)t * D]);
      if (s) return s;
    }
    tt.assign(D, 0);
    tr.challenge(D, tt.data());
    return OK;
  };
  for (int j = 0; j < lk; j++) {  // the top tree
    layer_challenges(tr, D, L, consts, as, lam);
    hf::E claim = layer_claim(D, as, lam, cp, cq);
    if ((status = sumcheck_verify(tr, j, st, claim.data(), j > 0 ? r.data() : nullptr, consts.data(), 1,
                                  label + "-top", j > 0 ? 2 : 0, rho.data(), reduced)))
      return status;
    if ((status = receive_finals())) return status;
    evaluate_statement(st, D, finals.data(), consts.data(), expected);
    if (memcmp(reduced, expected, 4 * D)) {
      set_error("verification-failure: gkr-top: layer " + std::to_string(j) + " of the top tree");
      return E_REJECT;
    }
    next_claims(D, L, finals.data(), tt, cp, cq);
    r.assign(rho.begin(), rho.begin() + (size_t)j * D);
    r.insert(r.end(), tt.begin(), tt.end());
  }
  rb = r;
  if (Kp != (uint64_t)K) {
    hf::E mass = padded_mass(D, lk, K, rb);
    for (int l = 0; l < L; l++) cq[l] = hf::sub(cq[l], mass);
  }
  for (int layer = 0; layer < n - 1; layer++) {  // the in-block layers
    layer_challenges(tr, D, L, consts, as, lam);
    std::vector<uint32_t> bw = block_weights(D, K, rb);
    hf::E claim = layer_claim(D, as, lam, cp, cq);
    if ((status = sumcheck_verify(tr, layer, st, claim.data(), layer > 0 ? ri.data() : nullptr, consts.data(), K,
                                  label, layer > 0 ? 2 : 0, rho.data(), reduced)))
      return status;
    std::vector<uint32_t> rbn;
    if (lk > 0) {
      rbn.assign((size_t)lk * D, 0);
      uint32_t red2[8];
      if ((status = sumcheck_verify(tr, lk, st_blk, reduced, nullptr, consts.data(), 1, label + "-blk", -1,
                                    rbn.data(), red2)))
        return status;
      memcpy(reduced, red2, 4 * D);
    }
    if ((status = receive_finals())) return status;
    hf::E weight = hf::zero(D);
    if (K > 1) {  // sum_b bw_b eq(rbn, b)
      std::vector<uint32_t> e = hf::eq_table(rbn.data(), lk, D);
      for (int b = 0; b < K; b++)
        weight = hf::add(weight, hf::mul(hf::from(&bw[(size_t)b * D], D), hf::from(&e[(size_t)b * D], D)));
    } else {
      weight = hf::from(bw.data(), D);
    }
    evaluate_statement(st, D, finals.data(), consts.data(), expected);
    hf::E want = hf::mul(weight, hf::from(expected, D));
    if (memcmp(reduced, want.data(), 4 * D)) {
      set_error("verification-failure: gkr-layer: in-block layer " + std::to_string(layer));
      return E_REJECT;
    }
    next_claims(D, L, finals.data(), tt, cp, cq);
    ri.assign(rho.begin(), rho.begin() + (size_t)layer * D);
    ri.insert(ri.end(), tt.begin(), tt.end());
    rb = rbn;
  }
  if (out_ri && !ri.empty()) memcpy(out_ri, ri.data(), ri.size() * 4);
  if (out_rb && !rb.empty()) memcpy(out_rb, rb.data(), rb.size() * 4);
  for (int l = 0; l < L; l++) {
    if (out_cp) memcpy(out_cp + (size_t)l * D, cp[l].data(), 4 * D);
    if (out_cq) memcpy(out_cq + (size_t)l * D, cq[l].data(), 4 * D);
  }
  return OK;
}

}  // namespace exh
