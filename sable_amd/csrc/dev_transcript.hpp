// dev_transcript.hpp -- the Fiat-Shamir transcript on the device, so the rounds of a sumcheck run back
// to back without a host round trip: the sequential BLAKE3 mode (src/blake3.lisp:125-155) and the
// transcript operations a prover round needs (src/transcript.lisp:95-100, 116-128, 152-176).  It absorbs
// and squeezes exactly the bytes the host transcript would.
//
// One wavefront runs it, every lane executing the same (uniform) steps.  A lone wavefront issues dependent instructions
// 8.0 cycles apart and independent ones 5.0 (256 of a kind in a row between two clock readings), so a step costs its
// longest chain first and its number of instructions second.
// The compression function is spread over the four lanes of each quad: lane i holds column i of the 4x4 state, so the
// four G functions of a half-round run side by side.  The chaining value stays in registers, where the compression
// takes and leaves it (lane i: words i and 4 + i); the pending block is a 128-byte ring in LDS (two 64-byte halves
// used alternately, zero wherever nothing has been appended), read at byte offsets every lane keeps in registers.
// Between launches the state is a DevB3S in device memory.
#pragma once
#include "blake3.hpp"

namespace exh {

struct DevB3S {
  uint32_t cv[8];
  uint32_t block[16];  // the pending block as little-endian words, zero beyond `used`
  uint32_t used;       // bytes taken in the pending block
  uint32_t counter_lo, counter_hi;
};

// S[r][k]: the message word used k-th in round r (G number g = k / 2 of columns 0-3 then diagonals 0-3, first
// and second operand): the BLAKE3 message permutation applied r times (src/blake3.lisp:37-40).  Lane i of a
// quad needs S[r][first + 2 i]: the four numbers, one nibble each, as a compile-time constant.
__host__ __device__ constexpr uint32_t b3_lane_words(int r, int first) {
  constexpr uint8_t S[7][16] = {
      {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15}, {2, 6, 3, 10, 7, 0, 4, 13, 1, 11, 12, 5, 9, 14, 15, 8},
      {3, 4, 10, 12, 13, 2, 7, 14, 6, 5, 9, 0, 11, 15, 8, 1}, {10, 7, 12, 9, 14, 3, 13, 15, 4, 0, 11, 2, 5, 8, 1, 6},
      {12, 13, 9, 11, 15, 10, 14, 8, 7, 2, 5, 3, 0, 1, 6, 4}, {9, 14, 11, 5, 8, 12, 15, 1, 13, 3, 0, 10, 2, 6, 4, 7},
      {11, 15, 5, 0, 1, 9, 8, 6, 14, 10, 2, 12, 3, 4, 7, 13}};
  return (uint32_t)S[r][first] | (uint32_t)S[r][first + 2] << 4 | (uint32_t)S[r][first + 4] << 8 |
         (uint32_t)S[r][first + 6] << 12;
}

#define EXH_QUAD(v, ctrl) ((uint32_t)__builtin_amdgcn_mov_dpp((int)(v), (ctrl), 0xf, 0xf, true))

// The running state.  In LDS (`ring`, RING_WORDS words): the pending block as a 128-byte ring (32 words), and 16 words
// that stage a squeeze's output when its candidates have to be sorted out.
constexpr int RING_WORDS = 48;
struct RunB3S {
  uint32_t *ring;
  uint32_t used, half;  // bytes taken in the pending half
  uint64_t counter;
  uint32_t cva, cvb;    // lane i of every quad: words i and 4 + i of the chaining value
  uint32_t at[28];      // where in a block (bytes) this lane's message words of each round lie: columns x, y, diagonals x, y
};

// where in a block (bytes) a lane's message words of each round lie
__device__ __forceinline__ void b3_quad_offsets(uint32_t at[28]) {
  const uint32_t i = threadIdx.x & 3, di = (i + 3) & 3;  // (the diagonal G that runs on this lane, see b3_quad_rounds)
#pragma unroll
  for (int r = 0; r < 7; r++) {
    // the four lanes' word numbers sit in the nibbles of a compile-time constant: no table in memory to read
    at[4 * r] = 4 * ((b3_lane_words(r, 0) >> (4 * i)) & 15u), at[4 * r + 1] = 4 * ((b3_lane_words(r, 1) >> (4 * i)) & 15u);
    at[4 * r + 2] = 4 * ((b3_lane_words(r, 8) >> (4 * di)) & 15u);
    at[4 * r + 3] = 4 * ((b3_lane_words(r, 9) >> (4 * di)) & 15u);
  }
}
__device__ __forceinline__ void rb3s_init(RunB3S &s, uint32_t *ring) {
  s.ring = ring;
  b3_quad_offsets(s.at);
}

// The compression with the state's columns spread over the lanes of a quad (of the pending half, below); d: the state's last
// row (counter low, counter high, block length, flags on lanes 0 to 3).  Lane i of each quad returns w0 = out[i],
// w1 = out[4+i], w2 = out[8+i], w3 = out[12+i].
// For the diagonals row b, the last one a half-round computes, stays where it is and rows a, c and d come to it: a
// inside the addition of its message word, c and d by moves that are done before b is (a permuted operand has to wait
// two instructions for its source, and the compiler counts every operand of such an instruction: permuting c and d
// inside the addition and the exclusive-or put two waits into every half-round).  With the chaining value and the
// word offsets in registers a compression takes 600 ns on a lone wavefront; rotating b, c and d, from LDS, 675 ns.
// m: the lane's message words; cva, cvb: words i and 4 + i of the chaining value.
__device__ __forceinline__ void b3_quad_rounds(const uint32_t m[28], uint32_t cva, uint32_t cvb, uint32_t d, uint32_t &w0,
                                               uint32_t &w1, uint32_t &w2, uint32_t &w3) {
  const uint32_t i = threadIdx.x & 3;
  uint32_t a = cva, b = cvb, c = i == 0 ? EXH_B3_IV0 : i == 1 ? EXH_B3_IV1 : i == 2 ? EXH_B3_IV2 : EXH_B3_IV3;
#define EXH_B3_HALF(A, C, D, x, y)                  \
  {                                                 \
    uint32_t t = (A) + (x), cq = (C), dq = (D);     \
    asm("" : "+v"(t), "+v"(cq), "+v"(dq));          \
    a = t + b;                                      \
    d = b3_rotr(dq ^ a, 16);                        \
    c = cq + d;                                     \
    b = b3_rotr(b ^ c, 12);                         \
    a = a + b + (y);                                \
    d = b3_rotr(d ^ a, 8);                          \
    c = c + d;                                      \
    b = b3_rotr(b ^ c, 7);                          \
  }
#pragma unroll
  for (int r = 0; r < 7; r++) {
    if (r == 0)
      EXH_B3_HALF(a, c, d, m[0], m[1])
    else  // back to the columns
      EXH_B3_HALF(EXH_QUAD(a, 0x39), EXH_QUAD(c, 0x93), EXH_QUAD(d, 0x4E), m[4 * r], m[4 * r + 1])
    // lane j: b_j with a_(j-1), c_(j+1), d_(j+2)
    EXH_B3_HALF(EXH_QUAD(a, 0x93), EXH_QUAD(c, 0x39), EXH_QUAD(d, 0x4E), m[4 * r + 2], m[4 * r + 3])
  }
#undef EXH_B3_HALF
  a = EXH_QUAD(a, 0x39), c = EXH_QUAD(c, 0x93), d = EXH_QUAD(d, 0x4E);
  w0 = a ^ c, w1 = b ^ d, w2 = c ^ cva, w3 = d ^ cvb;
}
__device__ __forceinline__ void b3_compress_quad(const RunB3S &s, uint32_t d, uint32_t &w0, uint32_t &w1, uint32_t &w2,
                                                 uint32_t &w3) {
  uint32_t m[28];
  const uint8_t *block = reinterpret_cast<const uint8_t *>(s.ring);
  // (the half as a constant in either branch: it then is part of the instructions' offsets)
  if (s.half == 0) {
#pragma unroll
    for (int k = 0; k < 28; k++) m[k] = *reinterpret_cast<const uint32_t *>(block + s.at[k]);
  } else {
#pragma unroll
    for (int k = 0; k < 28; k++) m[k] = *reinterpret_cast<const uint32_t *>(block + 64 + s.at[k]);
  }
  b3_quad_rounds(m, s.cva, s.cvb, d, w0, w1, w2, w3);
}

// lane i of a quad: the i-th of four uniform values
__device__ __forceinline__ uint32_t quad_pick(uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
  const uint32_t i = threadIdx.x & 3;
  return i == 0 ? v0 : i == 1 ? v1 : i == 2 ? v2 : v3;
}

__device__ inline void rb3s_load(RunB3S &s, uint32_t *ring, const DevB3S *g) {
  const uint32_t lane = threadIdx.x & 63;
  rb3s_init(s, ring);
  s.cva = g->cv[lane & 3], s.cvb = g->cv[4 + (lane & 3)];
  if (lane < 16) ring[lane] = g->block[lane], ring[16 + lane] = 0;
  __builtin_amdgcn_wave_barrier();
  s.used = g->used, s.half = 0;
  s.counter = ((uint64_t)g->counter_hi << 32) | g->counter_lo;
}
__device__ inline void rb3s_store(const RunB3S &s, DevB3S *g) {
  const uint32_t lane = threadIdx.x & 63;
  if (lane < 4) g->cv[lane] = s.cva, g->cv[4 + lane] = s.cvb;
  if (lane < 16) g->block[lane] = s.ring[16 * s.half + lane];
  g->used = s.used;
  g->counter_lo = (uint32_t)s.counter, g->counter_hi = (uint32_t)(s.counter >> 32);
}

// Input goes in as bytes at their place in the stream: byte k of what is appended next lies at rb3s_at(s, k), k <= 64
// (bytes that do not fit the pending half land in the other one); whichever lanes hold the bytes store them, and then
// the wavefront takes them in with rb3s_advance: a full half with more input behind it is compressed, cleared, and
// the halves change roles.  (A wavefront's LDS operations complete in order.)
__device__ __forceinline__ uint32_t rb3s_at(const RunB3S &s, uint32_t k) { return (64 * s.half + s.used + k) & 127u; }
__device__ __forceinline__ void rb3s_put_byte(const RunB3S &s, uint32_t k, uint32_t byte) {
  reinterpret_cast<uint8_t *>(s.ring)[rb3s_at(s, k)] = (uint8_t)byte;
}
__device__ __forceinline__ void rb3s_put_word(const RunB3S &s, uint32_t k, uint32_t word) {
#pragma unroll
  for (int b = 0; b < 4; b++) rb3s_put_byte(s, k + b, word >> (8 * b));
}
__device__ inline void rb3s_advance(RunB3S &s, uint32_t len) {
  __builtin_amdgcn_wave_barrier();
  if (s.used + len > 64) {
    uint32_t w0, w1, w2, w3;
    b3_compress_quad(s, quad_pick((uint32_t)s.counter, (uint32_t)(s.counter >> 32), 64, 0), w0, w1, w2, w3);
    s.cva = w0, s.cvb = w1;
    if ((threadIdx.x & 63) < 16) s.ring[16 * s.half + (threadIdx.x & 15)] = 0;
    __builtin_amdgcn_wave_barrier();
    s.counter++;
    s.half ^= 1;
    s.used = s.used + len - 64;
  } else {
    s.used += len;
  }
}

// absorb(data) for NWORDS little-endian words in LDS: the length as u64 LE, then the bytes
// (src/transcript.lisp:95-100)
__device__ inline void dev_absorb_words(RunB3S &s, const uint32_t *words, uint32_t nwords) {
  const uint32_t lane = threadIdx.x & 63, total = 2 + nwords;  // the stream in words, sixteen at a time
  for (uint32_t base = 0; base < total; base += 16) {
    const uint32_t g = base + lane;
    if (lane < 16 && g < total) rb3s_put_word(s, 4 * lane, g == 0 ? 4 * nwords : g == 1 ? 0u : words[g - 2]);
    rb3s_advance(s, 4 * (total - base < 16 ? total - base : 16));
  }
}

// The bytes a squeeze leaves to absorb -- "squeeze" and the first 32 bytes of its output -- kept for later: the caller
// absorbs them (rb3s_flush) before anything else goes through the transcript; in a round's serial part they would
// stand between the challenge and the fold that waits for it.
struct PendingAppend {
  uint32_t w0, w1;   // lane i of every quad: words i and 4 + i of the output
  uint32_t pending;  // 0: nothing
};
__device__ __forceinline__ void rb3s_put_echo(const RunB3S &s, uint32_t w0, uint32_t w1) {
  const uint32_t lane = threadIdx.x & 63;
  if (lane < 7) rb3s_put_byte(s, lane, (lane < 4 ? 0x65757173u >> (8 * lane) : 0x00657a65u >> (8 * (lane - 4))) & 0xff);
  // byte b of word i on lane i + 4 b, of word 4 + i as well
  if (lane < 16) {
    rb3s_put_byte(s, 7 + 4 * (lane & 3) + (lane >> 2), w0 >> (8 * (lane >> 2)));
    rb3s_put_byte(s, 23 + 4 * (lane & 3) + (lane >> 2), w1 >> (8 * (lane >> 2)));
  }
}
// `next_words`: the words of the message that is absorbed next (its length goes in with the echo), or 0
__device__ inline void rb3s_flush(RunB3S &s, PendingAppend &pending, uint32_t next_words = 0) {
  const uint32_t lane = threadIdx.x & 63, echo = pending.pending ? 39 : 0;
  if (echo) rb3s_put_echo(s, pending.w0, pending.w1);
  if (next_words && lane < 8) rb3s_put_byte(s, echo + lane, lane < 4 ? (4 * next_words) >> (8 * lane) : 0u);
  rb3s_advance(s, echo + (next_words ? 8 : 0));
  pending.pending = 0;
}

// K <= 12 base-field challenges (CHALLENGE-BASE, src/transcript.lisp:159-172): squeeze 4 (missing + 4)
// bytes (at most 64: one output block), keep the 31-bit words below p, repeat until K are kept; each squeeze then absorbs "squeeze" and
// the first min(32, n) bytes of its output (src/transcript.lisp:152-157): 32, since at least five words are squeezed
// where eight are fed -- a squeeze of fewer than eight words (K - kept < 4) feeds all of them.  put(i, v) takes the i-th
// challenge from whichever lane holds it; `ready` is called by the whole wavefront once all K are out: what follows (absorbing the last
// squeeze's bytes, a compression when they fill the block) is the transcript's own bookkeeping, which whoever waits
// for the challenge need not wait for.  With `pending` (not null) those bytes are handed back instead of absorbed, if
// they are 39 (see PendingAppend).
template <class Put, class Ready>
__device__ __forceinline__ void dev_challenge(RunB3S &s, int k, Put put, Ready ready, PendingAppend *pending) {
  const uint32_t lane = threadIdx.x & 63;
  int have = 0;
  while (have < k) {
    const uint32_t words = (uint32_t)(k - have + 4);  // at most 16: one output block
    uint32_t w0, w1, w2, w3;
    b3_compress_quad(s, quad_pick(0, 0, s.used, B3_CHUNK_END | B3_ROOT), w0, w1, w2, w3);
    bool done = false;
    if (have == 0 && (k == 4 || k == 8)) {
      // the usual case: the first K words are all below p, and lane i holds words i and 4 + i
      const bool fit = (w0 & 0x7fffffffu) < P && (k == 4 || (w1 & 0x7fffffffu) < P);
      if (__ballot(!fit) == 0) {
        if (lane < 4) {
          put(lane, w0 & 0x7fffffffu);
          if (k == 8) put(4 + lane, w1 & 0x7fffffffu);
        }
        have = k;
        done = true;
        __builtin_amdgcn_wave_barrier();
      }
    }
    if (!done) {
      uint32_t *stage = s.ring + 32;
      if (lane < 4) stage[lane] = w0, stage[4 + lane] = w1, stage[8 + lane] = w2, stage[12 + lane] = w3;
      __builtin_amdgcn_wave_barrier();
      const uint32_t cand = lane < words ? stage[lane & 15] & 0x7fffffffu : P;
      // the candidates below p, in order, as far as needed
      const uint64_t ok = __ballot(cand < P);
      const int rank = __popcll(ok & (((uint64_t)1 << lane) - 1));
      if (cand < P && have + rank < k) put((uint32_t)(have + rank), cand);
      have += __popcll(ok);
      __builtin_amdgcn_wave_barrier();
    }
    if (have >= k) ready();
    if (words >= 8) {
      if (have >= k && pending) {
        pending->w0 = w0, pending->w1 = w1, pending->pending = 1;
        return;
      }
      rb3s_put_echo(s, w0, w1);
      rb3s_advance(s, 39);
    } else {  // fewer than eight words were squeezed: all of them are fed (their other bytes are not part of it)
      if (lane < 7) rb3s_put_byte(s, lane, (lane < 4 ? 0x65757173u >> (8 * lane) : 0x00657a65u >> (8 * (lane - 4))) & 0xff);
      if (lane < 4) rb3s_put_word(s, 7 + 4 * lane, w0);
      if (lane < 4 && 4 + lane < words) rb3s_put_word(s, 23 + 4 * lane, w1);
      rb3s_advance(s, 7 + 4 * words);
    }
  }
}
__device__ inline void dev_challenge(RunB3S &s, int k, uint32_t *out) {
  dev_challenge(s, k, [&](uint32_t at, uint32_t v) { out[at] = v; }, [] {}, nullptr);
}

}  // namespace exh
