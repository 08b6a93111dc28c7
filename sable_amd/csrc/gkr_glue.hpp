// gkr_glue.hpp -- the step between two layers' sumchecks of LogUp-GKR on the device (device code; see gkr.hip for
// the chain it belongs to), as a launch of its own and as the end of the launch that finishes a layer's rounds.
#pragma once
#include "sumcheck_kernels.hpp"

namespace exh {

// ------------------------------------------------------------------ the layers chained on the device
// The layers' sumchecks run back to back without the host: between two of them one workgroup
// does what PROVE-UPPER does on the host there (src/gkr.lisp:248-271) -- it sends the finished
// layer's finals and draws the fresh point (SEND-FINALS), forms the next layer's point, draws the layer's
// challenges (LAYER-CHALLENGES), absorbs the next sumcheck's header and writes that sumcheck's constants where its
// launches expect them: the eq point's factors, the message map, the head of the control block with the
// transcript's state.  Everything the host needs afterwards goes to a log it reads once at the end.
// With several blocks the layers of the tree over the block index come first, and then a layer is two sumchecks, its own
// with the block weights as HIGH table and the one over the block index: the step between those two only records the
// first one's rounds and opens the second, with the layer's challenges kept from the step before; the step behind the
// second one sends the finals, and forms the next layer's block weights (eq of the block point, src/gkr.lisp:73-77).
constexpr int GLUE_MAXBLOCKS = 64, GLUE_BLOCK_BITS = 6;  // a lane per block in the step that forms their weights
constexpr int GLUE_MAXCONST = 8;  // constants of a layer statement the launch can form: a_l and a_l lambda, l < 4
struct GkrChainState {
  DevB3S tr;                       // the transcript between launches
  uint32_t point[MAXROUNDS + 1][8];  // the next layer's eq point (canonical)
  uint32_t consts[GLUE_MAXCONST][8];  // the layer's a_l and a_l lambda, kept for its sumcheck over the block index
  // sticky: a chained layer's sumcheck did not complete (a workgroup of a grid launch gave up, or the control
  // block does not count the layer's rounds); the host reads it after its one wait and voids the proof
  uint32_t failed;
};

template <int D>
struct GlueArgs {
  GkrChainState *chain;
  // 0: nothing to close, 1: send the roots, 2: a layer's finals from its control block, 3: from tables, 4: the rounds of a
  // layer's own sumcheck (its finals are those of the one over the block index)
  int close_kind;
  const Ctrl *prev_ctrl;
  int prev_rounds, prev_points;
  int fin_skip;  // kind 2: the first tables in the control block's finals that are not sent (the block weights)
  // kind 2, a sumcheck over the block index (blocks_closed): its challenges are the block point, and the fresh point is
  // coordinate tt_at of the layer's point, whose others an earlier step left in the chain's state
  int blocks_closed, tt_at;
  const uint32_t *tabs[MAXT];  // kind 1: the root of p and of q per lookup; kind 3: the layer's tables (one entry each)
  int NT, L;
  uint32_t *log;  // kind 1: the roots (2 L D words); kinds 2, 3: the layer's messages, challenges, finals, fresh point
  int open;       // 1: open the next layer's sumcheck, 2: the one over the block index
  int n;          // its rounds
  // a layer of several blocks: the weights of blocks 0 .. K - 1, eq of the block point of lk coordinates, go to bw (the
  // sumcheck's HIGH table; null without rounds) and to bw_table (the first table of the one over the block index)
  int K, lk;
  uint32_t *bw, *bw_table;
  uint32_t header[16];  // its header's bytes (src/sumcheck.lisp:24-27), as little-endian words
  int header_len;
  uint32_t *factors, *mtilde, *c0;
  Ctrl *ctrl;
  int points, nacc, c0_words;
  DevB3S start;  // kind 1: the transcript's state
  // the last step of a chain: the whole log (log_words at log_all), the transcript's state and the sticky word go to pinned
  // host memory, then host_seq to the word behind them (null: the host copies them)
  const uint32_t *log_all;
  uint32_t log_words, host_seq;
  uint32_t *host_log;
  uint32_t lagfix[MAXPTS * MAXACC];
  uint8_t acc_const[MAXACC];  // the constant (a_l: 2 l, a_l lambda: 2 l + 1) that is the accumulator's group coefficient
};

// absorb(bytes) for LEN bytes held as little-endian words in LDS: the length as u64 LE, then the bytes
__device__ inline void dev_absorb_bytes(RunB3S &s, const uint32_t *words, uint32_t len) {
  const uint32_t lane = threadIdx.x & 63, total = 8 + len;
  for (uint32_t base = 0; base < total; base += 64) {
    const uint32_t g = base + lane;
    uint32_t word = g < 4 ? len : (g < 8 || g >= total) ? 0 : words[(g - 8) >> 2];
    if (g < total) rb3s_put_byte(s, lane, word >> (8 * (g & 3)));
    rb3s_advance(s, total - base < 64 ? total - base : 64);
  }
}

// a word of a control block that this workgroup, or a launch before it, wrote: through the L2 (the first-level
// cache may still hold the line as it was when the launch began)
__device__ __forceinline__ uint32_t fresh_word(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// absorb one message of `words` words (its length as u64 LE before it) after the other, sixteen words of the stream at a time;
// message m's word w is at(m, w).  Message by message, eight of four words were 2,500 cycles more.
template <class At>
__device__ __forceinline__ void dev_absorb_messages(RunB3S &s, uint32_t messages, uint32_t words, At at) {
  const uint32_t lane = threadIdx.x & 63, each = words + 2, total = messages * each;
  for (uint32_t base = 0; base < total; base += 16) {
    const uint32_t g = base + lane, m = g / each, w = g % each;
    if (lane < 16 && g < total) rb3s_put_word(s, 4 * lane, w == 0 ? 4 * words : w == 1 ? 0u : at(m, w - 2));
    rb3s_advance(s, 4 * (total - base < 16 ? total - base : 16));
  }
}

// A workgroup of four wavefronts.  The first one runs the transcript, a chain of compressions that nothing else here is as
// long as; the others fetch what it needs last, record the finished layer and form the block weights beside it, and once the
// challenges are drawn write the next sumcheck's constants while it absorbs that one's header.  On one wavefront, each of
// those between two of the transcript's operations and most with a trip to memory, the step behind a layer's rounds was 24,500
// cycles (one lookup) and 30,700 (the blocks' sumcheck of two) and is 17,800 and 20,500; one that only opens the blocks' sumcheck
// 12,500 and is 6,600; the last one's delivery of the log 23,000 and is 6,700.
// `end`: where the launch's own rounds left the transcript and the finals (null: they are in the control block), `capacity` the
// entries between two of its tables; `completed`: they all ran.
template <int D, bool FUSED>
__device__ __forceinline__ void gkr_glue_body(const GlueArgs<D> &a, TailEnd &end, uint32_t capacity, bool completed) {
  __shared__ uint32_t ring[RING_WORDS];
  __shared__ uint32_t buf[64];
  __shared__ uint32_t header[16];
  __shared__ uint32_t chal[16], fresh[8];
  __shared__ uint32_t fin[MAXT * 8];
  __shared__ uint32_t consts[GLUE_MAXCONST][8];
  __shared__ uint32_t point[MAXROUNDS + 1][8];
  __shared__ uint32_t block_point[GLUE_BLOCK_BITS][8];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const bool from_ctrl = a.close_kind == 2 || a.close_kind == 4, finals = a.close_kind == 2 || a.close_kind == 3;
  const int R = a.prev_rounds, mw = a.prev_points * D;
  uint32_t *log_msg = a.log, *log_chal = log_msg + R * mw, *log_fin = log_chal + R * D, *log_tt = log_fin + a.NT * D;
  RunB3S &tr = end.tr;
  // the lane's block's weight, eq of the block point of coordinates at(v, .)
  auto weight_of = [&](auto at) {
    Ext<D> e = ext_lift<D>(1);
    for (int v = 0; v < a.lk; v++) {
      const bool set = (lane >> v) & 1;
      Ext<D> f;
#pragma unroll
      for (int c = 0; c < D; c++) f.c[c] = to_mont(set ? at(v, c) : fsub(c == 0 ? 1u : 0u, at(v, c)));
      e = ext_mul_mont<D>(e, f);
    }
    return e;
  };
  Ext<D> block_weight = ext_zero<D>();
  auto final_word = [&](uint32_t t, uint32_t c) {
    return end.tables[(size_t)(t + (uint32_t)a.fin_skip) * capacity * D + c];
  };
  if (wave == 0) {
    if (!FUSED || !from_ctrl) {  // the transcript's state and the finals where the last launch left them
      const uint32_t *g = reinterpret_cast<const uint32_t *>(from_ctrl ? &a.prev_ctrl->tr : &a.chain->tr);
      if (lane < sizeof(DevB3S) / 4)
        buf[lane] = a.close_kind == 1 ? reinterpret_cast<const uint32_t *>(&a.start)[lane] : fresh_word(g + lane);
      if (finals)
        for (int u = lane; u < a.NT * D; u += 64)
          fin[u] = a.close_kind == 2 ? fresh_word(&a.prev_ctrl->finals[a.fin_skip * D + u]) : a.tabs[u / D][u % D];
      if (a.close_kind == 1)  // the roots
        for (int u = lane; u < 2 * a.L * D; u += 64) fin[u] = a.log[u] = a.tabs[u / D][u % D];
      __builtin_amdgcn_wave_barrier();
      rb3s_load(tr, ring, reinterpret_cast<const DevB3S *>(buf));
      __builtin_amdgcn_wave_barrier();
    } else {
      rb3s_flush(tr, end.pending);
    }
    if (a.close_kind == 1) {  // one message (2, D) per lookup
      dev_absorb_messages(tr, (uint32_t)a.L, 2 * D, [&](uint32_t m, uint32_t w) { return fin[m * 2 * D + w]; });
    } else if (finals) {
      // SEND-FINALS: one message (1, D) per table, then the fresh point
      dev_absorb_messages(tr, (uint32_t)a.NT, D, [&](uint32_t m, uint32_t w) {
        return FUSED && from_ctrl ? final_word(m, w) : fin[m * D + w];
      });
      dev_challenge(tr, D, fresh);
    }
    if (a.open == 1) {
      // LAYER-CHALLENGES: a_l from one stream of L D base challenges, then lambda
      __builtin_amdgcn_wave_barrier();
      dev_challenge(tr, a.L * D, chal);
      __builtin_amdgcn_wave_barrier();
      if (lane < (uint32_t)(a.L * D)) consts[2 * (lane / D)][lane % D] = chal[lane];
      __builtin_amdgcn_wave_barrier();
      dev_challenge(tr, D, chal);
    }
  } else if (wave == 1) {  // the point, and the block weights
    if (from_ctrl) {
      for (int u = lane; u < R * D; u += 64) {
        const uint32_t v = fresh_word(&a.prev_ctrl->chal[u / D][u % D]);
        log_chal[u] = v;
        if (a.blocks_closed)
          block_point[u / D][u % D] = v;
        else
          point[u / D][u % D] = v;  // the layer's challenges open the next layer's point
      }
    }
    const int kept = a.blocks_closed && finals ? a.tt_at : a.open == 1 && (a.close_kind == 0 || a.close_kind == 1) ? a.n : 0;
    for (int u = lane; u < kept * D; u += 64) point[u / D][u % D] = fresh_word(&a.chain->point[u / D][u % D]);
    __builtin_amdgcn_wave_barrier();
    if (a.open == 1 && a.K > 1 && a.blocks_closed) {
      block_weight = weight_of([&](int v, int c) { return block_point[v][c]; });  // (of the challenges just closed)
    }
  } else if (wave == 2) {  // the log
    if (from_ctrl) {
      for (int u = lane; u < R * mw; u += 64) log_msg[u] = fresh_word(&a.prev_ctrl->msg[u / mw][u % mw]);
      if (lane == 0 && (fresh_word(&a.prev_ctrl->gave_up) != 0 ||
                        (FUSED ? !completed : fresh_word(&a.prev_ctrl->round) != (uint32_t)R)))
        a.chain->failed = 1;
    }
    if (a.close_kind == 1 && lane == 0) a.chain->failed = 0;
  } else {
    if (a.open && lane < 16) header[lane] = a.header[lane];
    if (a.open == 2)
      for (int u = lane; u < 2 * a.L * D; u += 64) consts[u / D][u % D] = fresh_word(&a.chain->consts[u / D][u % D]);
    if (FUSED && from_ctrl && finals)
      for (int u = lane; u < a.NT * D; u += 64) log_fin[u] = final_word(u / D, u % D);
  }
  // (the next sumcheck's constants may lie where the finished one's control block does: its words have all been read here)
  lds_barrier();
  if (!FUSED && finals)
    for (int u = tid; u < a.NT * D; u += BLOCK) log_fin[u] = fin[u];
  const int tt_at = a.blocks_closed ? a.tt_at : R;
  if (finals && tid < (uint32_t)D) log_tt[tid] = fresh[tid];
  auto coordinate = [&](int v, int k) { return finals && v == tt_at ? fresh[k] : point[v][k]; };
  if (wave == 0 && a.open) {
    dev_absorb_bytes(tr, header, (uint32_t)a.header_len);
    if (a.n > 0) rb3s_store(tr, &a.ctrl->tr);
  } else if (wave == 1 || !a.open) {
    if (wave == 1 && a.close_kind >= 2) {
      const int coords = finals ? tt_at + 1 : R;
      for (int u = lane; u < coords * D; u += 64) a.chain->point[u / D][u % D] = coordinate(u / D, u % D);
    }
    if (wave == 1 && a.open == 1 && a.K > 1) {
      if (!a.blocks_closed) block_weight = weight_of(coordinate);  // (of the point that the tree over the block index left)
      if (lane < (uint32_t)a.K) {
        store_ext<D>(a.bw_table + lane * D, block_weight);
        if (a.bw) store_ext<D>(a.bw + lane * D, block_weight);
      }
    }
    if (wave == 1 && a.open == 1) {
      // the eq point's factors r_v R and (1 - r_v) R, variable by variable
      for (int u = lane; u < a.n * D; u += 64) {
        const uint32_t v = u / D, k = u % D, r = coordinate((int)v, (int)k);
        a.factors[(2 * v) * D + k] = to_mont(r);
        a.factors[(2 * v + 1) * D + k] = to_mont(fsub(k == 0 ? 1u : 0u, r));
      }
    }
  } else if (wave == 2) {
    if (a.open == 1) {  // a_l lambda, exact: one factor carries R
      if (lane < (uint32_t)a.L) {
        Ext<D> x, y;
#pragma unroll
        for (int c = 0; c < D; c++) x.c[c] = consts[2 * lane][c], y.c[c] = to_mont(chal[c]);
        const Ext<D> z = ext_mul_mont<D>(x, y);
#pragma unroll
        for (int c = 0; c < D; c++) consts[2 * lane + 1][c] = z.c[c];
      }
      __builtin_amdgcn_wave_barrier();
      if (a.K > 1)
        for (int u = lane; u < 2 * a.L * D; u += 64) a.chain->consts[u / D][u % D] = consts[u / D][u % D];
    }
    // the message map: the accumulator's group coefficient times its scalar, in Montgomery form
    for (int u = lane; a.n > 0 && u < a.points * a.nacc * D; u += 64) {
      const int e = u / D, c = u % D;
      a.mtilde[u] = to_mont(fmul(consts[a.acc_const[e % a.nacc]][c], a.lagfix[e]));
    }
  } else if (a.n > 0) {
    for (int u = lane; u < a.c0_words; u += 64) a.c0[u] = 0;
    uint32_t *head = reinterpret_cast<uint32_t *>(a.ctrl);
    for (uint32_t u = sizeof(DevB3S) / 4 + lane; u < offsetof(Ctrl, msg) / 4; u += 64) head[u] = 0;
  }
  if (wave == 0) rb3s_store(tr, &a.chain->tr);
  if (a.host_log) {
    // (what this workgroup stored a moment ago is read back through the L2)
    __syncthreads();
    const uint32_t state_words = sizeof(DevB3S) / 4, total = a.log_words + state_words + 1;
    const uint32_t *state = reinterpret_cast<const uint32_t *>(&a.chain->tr);
    for (uint32_t base = 0; base < total; base += 8 * BLOCK) {
      uint32_t w[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint32_t u = base + BLOCK * k + tid;
        w[k] = fresh_word(u < a.log_words                 ? a.log_all + u
                          : u < a.log_words + state_words ? state + (u - a.log_words)
                                                          : &a.chain->failed);
      }
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (base + BLOCK * k + tid < total) a.host_log[base + BLOCK * k + tid] = w[k];
    }
    __threadfence_system();
    __syncthreads();
    if (tid == 0)
      __hip_atomic_store(a.host_log + total, a.host_seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

template <int D>
__global__ __launch_bounds__(BLOCK) void gkr_glue_kernel(GlueArgs<D> a) {
  TailEnd end;
  gkr_glue_body<D, false>(a, end, 0, true);
}

// The launch that finishes a layer's rounds (one workgroup, the tables in LDS) going straight on to the step
// above: the first wavefront has the transcript and LDS the finals, and the workgroup closes the layer and opens the
// next one without a launch in between.
template <int D, class S>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(1, 1))) void tail_glue_kernel(TailArgs<D> t,
                                                                                                    GlueArgs<D> g) {
  TailEnd end;
  const bool completed = tail_body<D, Tail::WHOLE, true>(S::d, t, end);
  gkr_glue_body<D, true>(g, end, t.capacity, completed);
}

}  // namespace exh
