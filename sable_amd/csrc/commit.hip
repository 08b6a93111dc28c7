// commit.hip -- see commit.hpp.
#include "commit.hpp"

#include <array>

#include <string.h>

#include <algorithm>
#include <atomic>
#include <map>
#include <vector>

#include "blake3.hpp"
#include "context.hpp"
#include "hostfield.hpp"
#include "prover.hpp"
#include "sumcheck.hpp"
#include "sumcheck_kernels.hpp"

namespace exh {

// ------------------------------------------------------------------ twiddle tables of a domain
// Level l of the 2^n tables (src/rs.lisp:44-55) holds x_s = w_n^(2^l bitrev_{n-1-l}(s)) for the
// 2^(n-1-l) position pairs of the level-l codeword.  Both x (for the encoder's butterflies) and
// 1/(2x) (for folding) are kept on the device, levels concatenated: x as the plain residue, 1/(2x) in Montgomery form.
struct Domain {
  int n = 0;
  uint32_t *tw = nullptr, *tw_inv2 = nullptr;
  uint64_t off[32];
};
static std::map<int, Domain> g_domains;

struct LevelOffsets {
  uint64_t off[32];
  int levels, n;
};

__device__ __forceinline__ uint32_t bitrev_dev(uint32_t v, int bits) { return bits ? __brev(v) >> (32 - bits) : 0; }

// pw: w_n^e for e < 4096, then w_n^(4096 e) for e < 4096 (Montgomery form); pw_inv the same for
// the inverse root times 1/2 folded into the first table
__global__ __launch_bounds__(BLOCK) void twiddle_kernel(LevelOffsets lv, const uint32_t *pw, const uint32_t *pw_inv,
                                                        uint32_t *tw, uint32_t *tw_inv2, uint64_t total) {
  uint64_t gid = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (gid >= total) return;
  int l = 0;
  while (l + 1 < lv.levels && gid >= lv.off[l + 1]) l++;
  uint32_t s = (uint32_t)(gid - lv.off[l]);
  uint32_t e = bitrev_dev(s, lv.n - 1 - l) << l;  // exponent of w_n, below 2^(n-1)
  // mont_mul of two Montgomery-form values is the Montgomery form of the product
  // (the encoder multiplies in double precision and takes the plain residue, the fold the Montgomery form)
  tw[gid] = mont_mul(mont_mul(pw[e & 4095], pw[4096 + (e >> 12)]), 1);
  tw_inv2[gid] = mont_mul(pw_inv[e & 4095], pw_inv[4096 + (e >> 12)]);
}

static int get_domain(int n, Domain **out) {
  auto it = g_domains.find(n);
  if (it != g_domains.end()) {
    *out = &it->second;
    return OK;
  }
  Context &c = ctx();
  Domain d;
  d.n = n;
  int levels = n - 1 > 1 ? n - 1 : 1;
  uint64_t total = 0, len = (uint64_t)1 << (n - 1);
  LevelOffsets lv;
  memset(&lv, 0, sizeof(lv));
  for (int l = 0; l < levels; l++, len /= 2) {
    d.off[l] = lv.off[l] = total;
    total += len;
  }
  lv.levels = levels;
  lv.n = n;
  uint32_t w = fpow(3, (uint64_t)(P - 1) >> n), winv = finv(w);
  std::vector<uint32_t> pw(8192), pwi(8192);
  uint32_t x = 1, xi = INV2;  // the 1/2 of 1/(2x) rides on the low table
  for (int e = 0; e < 4096; e++) {
    pw[e] = to_mont(x), pwi[e] = to_mont(xi);
    x = fmul(x, w), xi = fmul(xi, winv);
  }
  uint32_t w4096 = fpow(w, 4096), wi4096 = fpow(winv, 4096);
  x = 1, xi = 1;
  for (int e = 0; e < 4096; e++) {
    pw[4096 + e] = to_mont(x), pwi[4096 + e] = to_mont(xi);
    x = fmul(x, w4096), xi = fmul(xi, wi4096);
  }
  uint32_t *d_pw = nullptr;
  EXH_HIP(hipMalloc((void **)&d_pw, 2 * 8192 * 4));
  EXH_HIP(hipMemcpy(d_pw, pw.data(), 8192 * 4, hipMemcpyHostToDevice));
  EXH_HIP(hipMemcpy(d_pw + 8192, pwi.data(), 8192 * 4, hipMemcpyHostToDevice));
  EXH_HIP(hipMalloc((void **)&d.tw, total * 4));
  EXH_HIP(hipMalloc((void **)&d.tw_inv2, total * 4));
  uint32_t grid = (uint32_t)((total + BLOCK - 1) / BLOCK);
  hipLaunchKernelGGL(twiddle_kernel, dim3(grid), dim3(BLOCK), 0, c.stream, lv, d_pw, d_pw + 8192, d.tw, d.tw_inv2,
                     total);
  EXH_HIP(hipGetLastError());
  EXH_HIP(hipStreamSynchronize(c.stream));
  EXH_HIP(hipFree(d_pw));
  g_domains[n] = d;
  *out = &g_domains[n];
  return OK;
}

// ------------------------------------------------------------------ the encoder
// One pass of the butterflies (src/rs.lisp:60-73) for the stages b = b_hi .. b_lo over tiles held
// in LDS.  An index is (top | mid | low) with mid the bits b_lo..b_hi; a workgroup takes one top,
// all 2^S mids and C consecutive lows (C = tile / 2^S), so its loads are segments of C words and
// every butterfly of these stages stays inside the tile.  With `first` the input is the message
// m, read as m || m (src/rs.lisp:81).
//
// Inside the tile the stages run four at a time in registers: a thread gathers the 16 elements that
// differ in the four stage bits, does the 32 butterflies, and scatters them back, so LDS and the
// workgroup barrier are touched once per four stages.  The tile is padded by one element per 16 so that
// the strided gathers fall on distinct banks.
// A tile is 2^12 elements, 16 per thread: a domain of 2^24 takes three passes (6 + 5 + 12 stages) with
// global segments of at least 64 words.
// The butterflies run in double precision (field.hpp), eight instructions each where Montgomery arithmetic takes
// about twenty (the multiplies issue at the same rate either way): a product by a twiddle is six operations and
// leaves a residue within about p/2 of zero, and the sum and the difference that follow are one operation each
// with no reduction, exact as long as the values stay integers below 2^53: a tile's elements start below p and
// grow by less than 0.57 p per stage, so after a pass's twelve stages at most they are below 8 p, and a product
// with a twiddle below 2^65.  The tile in LDS therefore holds doubles; a pass ends by writing canonical residues.
// The passes are bound by their instructions all the same (some 330 per thread and round of four stages, the
// vector units busy nine tenths of the time): both columns of 2^24 take 64 + 56 + 92 us, against 300 us with
// Montgomery products and the tile fetched word by word.
constexpr int NTT_TILE_BITS = 12;
constexpr int NTT_BLOCK = 256;
constexpr int NTT_MAX_UPPER_STAGES = 7;  // per pass above the last: segments of 2^(12-7) words at least
static_assert(NTT_TILE_BITS <= 12, "a pass's stages, the bound on the lazily reduced values");
static_assert((1 << NTT_TILE_BITS) == 16 * NTT_BLOCK, "a thread moves a whole tile's sixteen words as four vectors");
__device__ __forceinline__ uint32_t ntt_pad(uint32_t e) { return e + (e >> 4); }
constexpr uint32_t ntt_lds_bytes(int tile_bits) {
  return (((uint32_t)1 << tile_bits) + ((uint32_t)1 << tile_bits >> 4) + 1) * 8;
}

// R stages d_lo .. d_lo + R - 1 of the pass (stage d pairs tile indices differing in bit cbits + d).  A thread
// takes groups of 2^R elements, its number of groups known at compile time for a FULL tile (2^NTT_TILE_BITS): the
// twiddles of all its groups are then fetched before the first butterfly, one wait for memory per round where a
// loop over the groups has one per group.  (Deriving a group's 2^R - 1 twiddles from one table entry, by squarings
// and products with fixed roots of unity, was measured: the passes are bound by their instructions, and fourteen
// more products per thirty-two butterflies cost more than the fetches.)
template <int R, bool FULL>
__device__ __forceinline__ void ntt_round(double *lds, uint32_t tile, int cbits, int d_lo, int b_lo, int b_hi,
                                          uint64_t top, const uint32_t *__restrict__ tw, const LevelOffsets &lv) {
  constexpr int GROUPS = FULL ? ((1 << NTT_TILE_BITS) >> R) / NTT_BLOCK : 1;
  const int p = cbits + d_lo;
  // a FULL tile's rounds have p = 0 or p >= 4 (a pass above the last keeps 2^cbits >= 32 consecutive indices, the
  // last one runs its twelve stages four at a time): a group's padded positions are then evenly spaced
  const uint32_t spacing = (1u << p) + ((1u << p) >> 4);
  for (uint32_t g0 = threadIdx.x; g0 < (tile >> R); g0 += GROUPS * NTT_BLOCK) {
    uint32_t t[GROUPS][(1 << R) - 1];
    // the twiddles of stage d_lo + s: 2^(R-1-s) of them, index (top | mid above the stage bit)
#pragma unroll
    for (int it = 0; it < GROUPS; it++) {
      const uint32_t upper = (g0 + it * NTT_BLOCK) >> p;
#pragma unroll
      for (int s = R - 1; s >= 0; s--) {
        const int b = b_lo + d_lo + s;
        const uint32_t *level = tw + lv.off[b] + ((top << (b_hi - b)) | ((uint64_t)upper << (R - 1 - s)));
#pragma unroll
        for (int jh = 0; jh < (1 << (R - 1 - s)); jh++) t[it][(1 << (R - 1 - s)) - 1 + jh] = level[jh];
      }
    }
#pragma unroll
    for (int it = 0; it < GROUPS; it++) {
      const uint32_t g = g0 + it * NTT_BLOCK, upper = g >> p, e_base = (upper << (p + R)) | (g & ((1u << p) - 1));
      double *const group = lds + ntt_pad(e_base);
      auto at = [&](int j) -> double & { return FULL ? group[j * spacing] : lds[ntt_pad(e_base | ((uint32_t)j << p))]; };
      double v[1 << R];
#pragma unroll
      for (int j = 0; j < (1 << R); j++) v[j] = at(j);
#pragma unroll
      for (int s = R - 1; s >= 0; s--) {
#pragma unroll
        for (int jh = 0; jh < (1 << (R - 1 - s)); jh++) {
          const double x = (double)t[it][(1 << (R - 1 - s)) - 1 + jh];
#pragma unroll
          for (int jl = 0; jl < (1 << s); jl++) {
            const int j = (jh << (s + 1)) | jl;
            const double a = v[j], tc = f_mul(x, v[j + (1 << s)]);
            v[j] = a + tc;
            v[j + (1 << s)] = a - tc;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < (1 << R); j++) at(j) = v[j];
    }
  }
}

// FULL: the tile is 2^NTT_TILE_BITS words and `in`, `out` and the columns' strides are multiples of 16 bytes: a
// thread moves its sixteen words as four vectors of four consecutive ones (a segment of consecutive indices is a
// multiple of four long, or the tile is one segment), all four fetches in flight at once.
template <bool FULL>
__global__ __launch_bounds__(NTT_BLOCK) __attribute__((amdgpu_waves_per_eu(5, 8))) void ntt_pass_kernel(
    const uint32_t *in, uint32_t *out, int n, int b_hi, int b_lo, int tile_bits,
    const uint32_t *__restrict__ tw, LevelOffsets lv, int first, uint64_t in_stride, uint64_t out_stride) {
  extern __shared__ double lds[];  // 2^tile_bits elements plus one per 16
  const int S = b_hi - b_lo + 1, cbits = tile_bits - S;
  const uint32_t tile = 1u << tile_bits, C = 1u << cbits;
  in += (uint64_t)blockIdx.y * in_stride;
  out += (uint64_t)blockIdx.y * out_stride;
  const uint64_t chunks_per_top = ((uint64_t)1 << b_lo) >> cbits;
  const uint64_t top = blockIdx.x / chunks_per_top, chunk = blockIdx.x % chunks_per_top;
  const uint64_t base = (top << (b_hi + 1)) | (chunk << cbits);
  const uint64_t msg_mask = ((uint64_t)1 << (n - 1)) - 1;
  auto global_index = [&](uint32_t e) { return base | ((uint64_t)(e >> cbits) << b_lo) | (e & (C - 1)); };
  if (FULL) {
    uint4 w[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint64_t g = global_index(4 * (threadIdx.x + k * NTT_BLOCK));
      w[k] = *reinterpret_cast<const uint4 *>(in + (first ? g & msg_mask : g));
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      double *at = lds + ntt_pad(4 * (threadIdx.x + k * NTT_BLOCK));  // (four elements never straddle a pad)
      at[0] = (double)w[k].x, at[1] = (double)w[k].y, at[2] = (double)w[k].z, at[3] = (double)w[k].w;
    }
  } else {
    for (uint32_t e = threadIdx.x; e < tile; e += NTT_BLOCK) {
      const uint64_t g = global_index(e);
      lds[ntt_pad(e)] = (double)(first ? in[g & msg_mask] : in[g]);
    }
  }
  __syncthreads();
  for (int d_hi = S - 1; d_hi >= 0;) {
    const int R = d_hi + 1 < 4 ? d_hi + 1 : 4, d_lo = d_hi - R + 1;
    if (R == 4)
      ntt_round<4, FULL>(lds, tile, cbits, d_lo, b_lo, b_hi, top, tw, lv);
    else if (R == 3)
      ntt_round<3, FULL>(lds, tile, cbits, d_lo, b_lo, b_hi, top, tw, lv);
    else if (R == 2)
      ntt_round<2, FULL>(lds, tile, cbits, d_lo, b_lo, b_hi, top, tw, lv);
    else
      ntt_round<1, FULL>(lds, tile, cbits, d_lo, b_lo, b_hi, top, tw, lv);
    __syncthreads();
    d_hi = d_lo - 1;
  }
  if (FULL) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t e = 4 * (threadIdx.x + k * NTT_BLOCK);
      const double *at = lds + ntt_pad(e);
      *reinterpret_cast<uint4 *>(out + global_index(e)) =
          make_uint4(f_canonical(at[0]), f_canonical(at[1]), f_canonical(at[2]), f_canonical(at[3]));
    }
  } else {
    for (uint32_t e = threadIdx.x; e < tile; e += NTT_BLOCK) out[global_index(e)] = f_canonical(lds[ntt_pad(e)]);
  }
}

// m || m for the degenerate domains with no butterfly stage
__global__ void dup_kernel(const uint32_t *in, uint32_t *out, uint64_t half, uint64_t in_stride, uint64_t out_stride) {
  uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid < 2 * half) out[blockIdx.y * out_stride + gid] = in[blockIdx.y * in_stride + (gid % half)];
}

int rs_encode_columns(const uint32_t *d_messages, int ncols, int c, uint32_t *d_codewords) {
  Context &cx = ctx();
  int status = cx.require();
  if (status) return status;
  int n = c + 1;
  uint64_t len = (uint64_t)1 << n;
  if (n < 2) {
    hipLaunchKernelGGL(dup_kernel, dim3(1, ncols), dim3(64), 0, cx.stream, d_messages, d_codewords, len / 2, len / 2, len);
    EXH_HIP(hipGetLastError());
    return OK;
  }
  Domain *dom;
  if ((status = get_domain(n, &dom))) return status;
  LevelOffsets lv;
  memset(&lv, 0, sizeof(lv));
  lv.levels = n - 1, lv.n = n;
  for (int l = 0; l < n - 1; l++) lv.off[l] = dom->off[l];
  int tile_bits = n - 1 < NTT_TILE_BITS ? n - 1 : NTT_TILE_BITS;  // a tile never spans two tops
  const uint32_t lds_bytes = ntt_lds_bytes(tile_bits);
  // whole tiles whose words move four at a time: every address and stride a multiple of 16 bytes, segments of
  // consecutive indices at least four long (a pass above the last has 2^(tile_bits - stages) >= 32 of them)
  const bool full = tile_bits == NTT_TILE_BITS && (reinterpret_cast<uintptr_t>(d_messages) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(d_codewords) & 15) == 0;
  static_assert(NTT_TILE_BITS - NTT_MAX_UPPER_STAGES >= 2, "segments of four words at least");
  // stages n-2 .. 0: the last pass takes the low tile_bits stages, earlier passes share the rest
  int b = n - 2;
  bool first = true;
  while (b >= 0) {
    int b_lo;
    if (b < tile_bits)
      b_lo = 0;
    else {
      int remaining = b - tile_bits + 1;  // stages above the last pass
      int take = remaining > NTT_MAX_UPPER_STAGES
                     ? (remaining > 2 * NTT_MAX_UPPER_STAGES ? NTT_MAX_UPPER_STAGES : (remaining + 1) / 2)
                     : remaining;
      b_lo = b - take + 1;
    }
    uint32_t grid = (uint32_t)(len >> tile_bits);
    hipLaunchKernelGGL(full ? ntt_pass_kernel<true> : ntt_pass_kernel<false>, dim3(grid, ncols), dim3(NTT_BLOCK),
                       lds_bytes, cx.stream, first ? d_messages : d_codewords, d_codewords, n, b, b_lo, tile_bits,
                       dom->tw, lv, first ? 1 : 0, first ? len / 2 : len, len);
    first = false;
    b = b_lo - 1;
  }
  EXH_HIP(hipGetLastError());
  return OK;
}

// ------------------------------------------------------------------ codeword folding
// pair (a, b) at twiddle x: f0 = (a + b)/2, f1 = (a - b)/(2x), out = f0 + r (f1 - f0)
template <int D>
__global__ __launch_bounds__(BLOCK) void rs_fold_kernel(const uint32_t *cw, const uint32_t *tw_inv2, uint32_t *out,
                                                        uint64_t m, RoundArgs<D> args) {
  uint64_t s = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (s >= m) return;
  Ext<D> r;
#pragma unroll
  for (int c = 0; c < D; c++) r.c[c] = args.r_mont[c];
  Ext<D> a = load_ext<D>(cw + 2 * s * D), b = load_ext<D>(cw + (2 * s + 1) * D);
  Ext<D> f0 = ext_scale_mont<D>(ext_add<D>(a, b), mont_mul(INV2, R2));
  Ext<D> f1 = ext_scale_mont<D>(ext_sub<D>(a, b), tw_inv2[s]);
  store_ext<D>(out + s * D, ext_add<D>(f0, ext_mul_mont<D>(r, ext_sub<D>(f1, f0))));
}

static int rs_fold_launch(int D, uint64_t m, const uint32_t *tw_inv2_level, const uint32_t *d_cw, const uint32_t *r,
                          uint32_t *d_out) {
  Context &c = ctx();
  uint32_t grid = (uint32_t)((m + BLOCK - 1) / BLOCK);
  if (D == 4) {
    RoundArgs<4> a;
    memset(&a, 0, sizeof(a));
    for (int k = 0; k < 4; k++) a.r_mont[k] = to_mont(r[k] % P);
    hipLaunchKernelGGL(rs_fold_kernel<4>, dim3(grid), dim3(BLOCK), 0, c.stream, d_cw, tw_inv2_level, d_out, m, a);
  } else {
    RoundArgs<8> a;
    memset(&a, 0, sizeof(a));
    for (int k = 0; k < 8; k++) a.r_mont[k] = to_mont(r[k] % P);
    hipLaunchKernelGGL(rs_fold_kernel<8>, dim3(grid), dim3(BLOCK), 0, c.stream, d_cw, tw_inv2_level, d_out, m, a);
  }
  EXH_HIP(hipGetLastError());
  return OK;
}

int rs_fold_device(int D, uint64_t m, int n_domain, int level, const uint32_t *d_cw, const uint32_t *r, uint32_t *d_out) {
  int status = ctx().require();
  if (status) return status;
  Domain *dom;
  if ((status = get_domain(n_domain, &dom))) return status;
  return rs_fold_launch(D, m, dom->tw_inv2 + dom->off[level], d_cw, r, d_out);
}

// ------------------------------------------------------------------ COMBINE-COLUMNS (src/pcs.lisp:434-441)
// g[x] = sum_k coefficient_k * column_k[x]: base columns (column k at cols + k * len), extension coefficients,
// the table BaseFold opens.  One pass: 4 ncols bytes read and 4 D written per x, one x per thread (four per
// thread measured a third slower: the 128-byte strides between lanes' stores).  The coefficients arrive as
// kernel arguments in Montgomery form, so a reduction of four products gives their exact sum.
constexpr int COMBINE_COLS = 32;  // columns whose coefficients travel as kernel arguments; more take the other kernel
template <int D>
struct CombineArgs {
  uint32_t coef_mont[COMBINE_COLS][D];
};
template <int D>
__global__ __launch_bounds__(BLOCK) void combine_columns_kernel(const uint32_t *cols, uint64_t len, int ncols,
                                                                CombineArgs<D> a, uint32_t *out, const uint32_t *add) {
  const uint64_t x = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (x >= len) return;
  Ext<D> g = add ? load_ext<D>(add + x * D) : ext_zero<D>();
  for (int k0 = 0; k0 < ncols; k0 += 4) {  // four columns per reduction: 4 p^2 < 2^64
    uint32_t val[4];
#pragma unroll
    for (int q = 0; q < 4; q++) val[q] = k0 + q < ncols ? cols[(uint64_t)(k0 + q) * len + x] : 0u;
#pragma unroll
    for (int c = 0; c < D; c++) {
      uint64_t t = 0;
#pragma unroll
      for (int q = 0; q < 4; q++) t += (uint64_t)(k0 + q < ncols ? a.coef_mont[k0 + q][c] : 0u) * val[q];
      g.c[c] = fadd(g.c[c], mont_reduce4(t));
    }
  }
  store_ext<D>(out + x * D, g);  // (non-temporal stores measured a third slower)
}

// The same sum for many columns in one pass: the output stays in registers across all of them instead of being
// read and written again every 32 columns.  The coefficients (Montgomery form, padded with zeros to a multiple of
// eight columns) come from device memory at addresses every lane shares, eight columns' loads are in flight at
// once, and a lane walks the columns at its own x.
template <int D>
__global__ __launch_bounds__(BLOCK) void combine_columns_many_kernel(const uint32_t *__restrict__ cols, uint64_t len,
                                                                     int ncols, const uint32_t *__restrict__ coef_mont,
                                                                     uint32_t *__restrict__ out) {
  const uint64_t x = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (x >= len) return;
  Ext<D> g = ext_zero<D>();
  for (int k0 = 0; k0 < ncols; k0 += 8) {
    uint32_t val[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {  // a column past the last is read again with a zero coefficient
      const int k = k0 + q < ncols ? k0 + q : ncols - 1;
      val[q] = cols[(uint64_t)k * len + x];
    }
#pragma unroll
    for (int half = 0; half < 2; half++) {  // four columns per reduction: 4 p^2 < 2^64
      const uint32_t *cf = coef_mont + (size_t)(k0 + 4 * half) * D;
#pragma unroll
      for (int c = 0; c < D; c++) {
        uint64_t t = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) t += (uint64_t)cf[q * D + c] * val[4 * half + q];
        g.c[c] = fadd(g.c[c], mont_reduce4(t));
      }
    }
  }
  store_ext<D>(out + x * D, g);
}

template <int D>
static int combine_many_launch(const uint32_t *d_cols, int ncols, uint64_t len, const uint32_t *coef, uint32_t *d_out) {
  Context &c = ctx();
  const int padded = (ncols + 7) / 8 * 8;
  std::vector<uint32_t> cm((size_t)padded * D, 0u);
  for (size_t i = 0; i < (size_t)ncols * D; i++) cm[i] = to_mont(coef[i] % P);
  uint32_t *d_coef = (uint32_t *)c.pool.alloc(cm.size() * 4);
  if (!d_coef) {
    set_error("device-out-of-memory: combine-columns coefficients");
    return E_NOMEM;
  }
  struct Release {
    Pool &pool;
    void *ptr;
    ~Release() { pool.release(ptr); }
  } release{c.pool, d_coef};
  // (from pageable memory: the call returns once the words are staged, so `cm` may go)
  EXH_HIP(hipMemcpyAsync(d_coef, cm.data(), cm.size() * 4, hipMemcpyHostToDevice, c.stream));
  uint32_t grid = (uint32_t)((len + BLOCK - 1) / BLOCK);
  hipLaunchKernelGGL((combine_columns_many_kernel<D>), dim3(grid), dim3(BLOCK), 0, c.stream, d_cols, len, ncols, d_coef,
                     d_out);
  EXH_HIP(hipGetLastError());
  return OK;
}

// out = add + sum_k coefficient_k * column_k (add null: zero; it may be `out` itself) for at most COMBINE_COLS columns
template <int D>
static void combine_few_launch(const uint32_t *d_cols, int ncols, uint64_t len, const uint32_t *coef, const uint32_t *add,
                               uint32_t *d_out) {
  CombineArgs<D> a;
  memset(&a, 0, sizeof(a));
  for (int k = 0; k < ncols; k++)
    for (int cc = 0; cc < D; cc++) a.coef_mont[k][cc] = to_mont(coef[(size_t)k * D + cc] % P);
  const uint32_t grid = (uint32_t)((len + BLOCK - 1) / BLOCK);
  hipLaunchKernelGGL((combine_columns_kernel<D>), dim3(grid), dim3(BLOCK), 0, ctx().stream, d_cols, len, ncols, a, d_out,
                     add);
}
template <int D>
static int combine_launch(const uint32_t *d_cols, int ncols, uint64_t len, const uint32_t *coef, uint32_t *d_out) {
  if (ncols > COMBINE_COLS) return combine_many_launch<D>(d_cols, ncols, len, coef, d_out);
  combine_few_launch<D>(d_cols, ncols, len, coef, nullptr, d_out);
  EXH_HIP(hipGetLastError());
  return OK;
}

int combine_columns_device(int D, const uint32_t *d_cols, int ncols, uint64_t len, const uint32_t *coef,
                           uint32_t *d_out) {
  int status = ctx().require();
  if (status) return status;
  ctx().prof_begin("combine_columns", 0, len * (4 * (uint64_t)ncols + 4 * (uint64_t)D));
  status = D == 4 ? combine_launch<4>(d_cols, ncols, len, coef, d_out) : combine_launch<8>(d_cols, ncols, len, coef, d_out);
  ctx().prof_end();
  return status;
}

// ------------------------------------------------------------------ Merkle trees
// LEAF-DIGEST (src/pcs.lisp:44-52) of leaf l of ncols codewords: one row of 4 symbols per column,
// rows hashed 64 at a time and chained h = BLAKE3(h || d).
__device__ __forceinline__ void column_leaf_digest(const uint32_t *cw, int ncols, uint64_t cw_len, uint64_t l,
                                                   uint32_t h[8]) {
  uint32_t d[8], m[16];
  bool have = false;
  for (int start = 0; start < ncols; start += 64) {
    int rows = ncols - start < 64 ? ncols - start : 64;
    int nblocks = (rows + 3) / 4;
    b3_iv(d);
    for (int b = 0; b < nblocks; b++) {
      int have_rows = rows - 4 * b < 4 ? rows - 4 * b : 4;
#pragma unroll
      for (int k = 0; k < 4; k++) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (k < have_rows) v = *reinterpret_cast<const uint4 *>(cw + (uint64_t)(start + 4 * b + k) * cw_len + 4 * l);
        m[4 * k] = v.x, m[4 * k + 1] = v.y, m[4 * k + 2] = v.z, m[4 * k + 3] = v.w;
      }
      uint32_t flags = (b == 0 ? B3_CHUNK_START : 0u) | (b == nblocks - 1 ? (B3_CHUNK_END | B3_ROOT) : 0u);
      b3_compress(d, m, 0, (uint32_t)(16 * have_rows), flags, d, 0);
    }
    if (have)
      b3_node(h, d, h);
    else {
#pragma unroll
      for (int i = 0; i < 8; i++) h[i] = d[i];
      have = true;
    }
  }
}

// leaf l of an oracle codeword of EXT8s: one row per coordinate, symbols 4l..4l+3
// (ORACLE-ROWS, src/pcs.lisp:577-579): 128 bytes, two blocks
__device__ __forceinline__ void oracle_leaf_digest(const uint32_t *cw, uint64_t l, uint32_t h[8]) {
  uint32_t sym[4][8];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    Ext<8> e = load_ext<8>(cw + (4 * l + s) * 8);
#pragma unroll
    for (int d = 0; d < 8; d++) sym[s][d] = e.c[d];
  }
  uint32_t m[16];
  b3_iv(h);
#pragma unroll
  for (int b = 0; b < 2; b++) {
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int s = 0; s < 4; s++) m[4 * k + s] = sym[s][4 * b + k];
    uint32_t flags = b == 0 ? B3_CHUNK_START : (B3_CHUNK_END | B3_ROOT);
    b3_compress(h, m, 0, 64, flags, h, 0);
  }
}

__device__ __forceinline__ void store_digest(uint32_t *p, const uint32_t h[8]) {
  uint4 *o = reinterpret_cast<uint4 *>(p);
  o[0] = make_uint4(h[0], h[1], h[2], h[3]);
  o[1] = make_uint4(h[4], h[5], h[6], h[7]);
}
__device__ __forceinline__ void load_digest(const uint32_t *p, uint32_t h[8]) {
  const uint4 *i = reinterpret_cast<const uint4 *>(p);
  uint4 a = i[0], b = i[1];
  h[0] = a.x, h[1] = a.y, h[2] = a.z, h[3] = a.w, h[4] = b.x, h[5] = b.y, h[6] = b.z, h[7] = b.w;
}

// Up to `height` levels of nodes above 2 * BLOCK consecutive nodes of `level` (n of them), node =
// BLAKE3(left || right) (src/pcs.lisp:54-55, 64-77), every level written behind the one below
// (level k + 1 starts 8 * n_k words after level k) and carried to the next step through LDS.
// LEAVES 0: `level` holds digests; 1: the bottom nodes are the leaf digests of ncols codewords
// (written too); 2: of an oracle codeword.
// With cap_out the last level is the cap: its words go to pinned host memory as 64-bit words (seq << 32 | value)
// too, eight lanes to a digest.  Height 0 (one workgroup, at most BLOCK / 2 leaves): the leaves are the cap.
template <int LEAVES>
__global__ __launch_bounds__(BLOCK) void subtree_kernel(uint32_t *level, uint64_t n, int height, const uint32_t *cw,
                                                        int ncols, uint64_t cw_len, unsigned long long *cap_out,
                                                        uint32_t seq) {
  __shared__ uint32_t lds[BLOCK][9];  // a digest per row, padded against bank conflicts
  const uint32_t t = threadIdx.x;
  uint64_t first = (uint64_t)blockIdx.x * BLOCK;  // this workgroup's first node of the level being written
  uint64_t count = n / 2;                         // nodes of that level
  uint32_t *out = level + 8 * n;
  uint32_t left[8], right[8], h[8];
  if (first + t < count) {
    const uint64_t c0 = 2 * (first + t);
    if (LEAVES == 0) {
      load_digest(level + 8 * c0, left);
      load_digest(level + 8 * (c0 + 1), right);
    } else {
      if (LEAVES == 1) {
        column_leaf_digest(cw, ncols, cw_len, c0, left);
        column_leaf_digest(cw, ncols, cw_len, c0 + 1, right);
      } else {
        oracle_leaf_digest(cw, c0, left);
        oracle_leaf_digest(cw, c0 + 1, right);
      }
      store_digest(level + 8 * c0, left);
      store_digest(level + 8 * (c0 + 1), right);
    }
    if (height > 0) {
      b3_node(left, right, h);
      store_digest(out + 8 * (first + t), h);
#pragma unroll
      for (int i = 0; i < 8; i++) lds[t][i] = h[i];
    } else if (2 * t + 1 < BLOCK) {
#pragma unroll
      for (int i = 0; i < 8; i++) lds[2 * t][i] = left[i], lds[2 * t + 1][i] = right[i];
    }
  }
  uint32_t width = BLOCK;  // nodes of the current level held by this workgroup (when full)
  if (height == 0) count = n;
  for (int s = 1; s < height; s++) {
    __syncthreads();
    out += 8 * count;
    count /= 2, first /= 2, width /= 2;
    const bool active = t < width && first + t < count;
    if (active) {
#pragma unroll
      for (int i = 0; i < 8; i++) left[i] = lds[2 * t][i], right[i] = lds[2 * t + 1][i];
      b3_node(left, right, h);
      store_digest(out + 8 * (first + t), h);
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int i = 0; i < 8; i++) lds[t][i] = h[i];
    }
  }
  if (cap_out) {
    __syncthreads();
    for (uint32_t w = t; w < 8 * width; w += BLOCK)
      if (first + w / 8 < count)
        __hip_atomic_store(cap_out + 8 * first + w, ((unsigned long long)seq << 32) | lds[w / 8][w % 8], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// The same for trees of few leaves and for the upper levels of large ones, a compression on the four lanes of a quad
// (dev_transcript.hpp): a thread hashing alone is a chain of 678 instructions five cycles apart, 1.4 us, and a leaf of many
// columns or a level above another is one such chain after the other while most of the device idles; on four lanes it is
// 0.6 us, for a third more instructions in all.  A workgroup of THREADS takes THREADS / 4 leaves or twice as many digests;
// both levels of a step lie in LDS, two digests -- one message -- a row.  Arguments as above; height at most the levels of
// the workgroup's own tree.  256 threads over the leaves: with 1024 (256 leaves, eight levels, fewer workgroups) 2^13
// leaves of 70 columns took 97 us for 79, 2^14 of 30 columns 77 for 68, and 2^16 of two 62 for 66.
constexpr int QUAD_LEAF_THREADS = 256, QUAD_LEAF_HEIGHT = 6;     // 64 leaves
constexpr int QUAD_NODE_THREADS = 1024, QUAD_NODE_HEIGHT = 9;    // 512 digests
constexpr uint64_t QUAD_LEAVES = 1 << 16, QUAD_DIGESTS = 1 << 17;  // trees and levels up to here (merkle_tree_launch)
constexpr int QUAD_ROW = 20;  // words of a row: rows begin on 16 bytes and four lanes' words of different quads meet on few banks
template <int LEAVES, int THREADS>
__global__ __launch_bounds__(THREADS) void quad_tree_kernel(uint32_t *level, uint64_t n, int height, const uint32_t *cw,
                                                            int ncols, uint64_t cw_len, unsigned long long *cap_out,
                                                            uint32_t seq) {
  constexpr int QUADS = THREADS / 4, BOTTOM = LEAVES ? QUADS : 2 * QUADS;
  __shared__ __align__(16) uint32_t rows[2][QUADS * QUAD_ROW];
  const uint32_t tid = threadIdx.x, quad = tid / 4, i = tid % 4;
  const uint32_t iva = i == 0 ? EXH_B3_IV0 : i == 1 ? EXH_B3_IV1 : i == 2 ? EXH_B3_IV2 : EXH_B3_IV3;
  const uint32_t ivb = i == 0 ? EXH_B3_IV4 : i == 1 ? EXH_B3_IV5 : i == 2 ? EXH_B3_IV6 : EXH_B3_IV7;
  uint32_t at[28];
  b3_quad_offsets(at);
  auto compress = [&](const uint32_t *row, uint32_t &a, uint32_t &b, uint32_t len, uint32_t flags) {
    uint32_t m[28], w2, w3;
#pragma unroll
    for (int k = 0; k < 28; k++) m[k] = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const uint8_t *>(row) + at[k]);
    b3_quad_rounds(m, a, b, i == 2 ? len : i == 3 ? flags : 0u, a, b, w2, w3);
  };
  auto digest_at = [&](int buffer, uint32_t d) { return rows[buffer] + (d >> 1) * QUAD_ROW + (d & 1) * 8; };
  uint64_t first = (uint64_t)blockIdx.x * BOTTOM, count = n;  // this workgroup's first node of the level at hand
  uint32_t *out = level;
  if constexpr (LEAVES != 0) {
    const uint64_t l = first + quad < n ? first + quad : n - 1;
    uint32_t *row = rows[1] + quad * QUAD_ROW, ha = 0, hb = 0;  // (the other buffer is free until the first level is done)
    if constexpr (LEAVES == 1) {
      for (int start = 0; start < ncols; start += 64) {
        const int have = ncols - start < 64 ? ncols - start : 64, nblocks = (have + 3) / 4;
        auto fetch = [&](int b) {
          const int k = 4 * b + (int)i;
          return k < have ? *reinterpret_cast<const uint4 *>(cw + (uint64_t)(start + k) * cw_len + 4 * l) : make_uint4(0, 0, 0, 0);
        };
        uint32_t da = iva, db = ivb;
        uint4 v = fetch(0);
        for (int b = 0; b < nblocks; b++) {
          __builtin_amdgcn_wave_barrier();
          *reinterpret_cast<uint4 *>(row + 4 * i) = v;
          __builtin_amdgcn_wave_barrier();
          if (b + 1 < nblocks) v = fetch(b + 1);
          const int here = have - 4 * b < 4 ? have - 4 * b : 4;
          compress(row, da, db, 16u * (uint32_t)here,
                   (b == 0 ? B3_CHUNK_START : 0u) | (b == nblocks - 1 ? (B3_CHUNK_END | B3_ROOT) : 0u));
        }
        if (start == 0) {
          ha = da, hb = db;
        } else {  // h = BLAKE3(h || d)
          __builtin_amdgcn_wave_barrier();
          row[i] = ha, row[4 + i] = hb, row[8 + i] = da, row[12 + i] = db;
          __builtin_amdgcn_wave_barrier();
          ha = iva, hb = ivb;
          compress(row, ha, hb, 64, B3_CHUNK_START | B3_CHUNK_END | B3_ROOT);
        }
      }
    } else {  // lane s holds symbol 4 l + s: word 4 k + s of block b is its coordinate 4 b + k
      const uint4 *sym = reinterpret_cast<const uint4 *>(cw + (4 * l + i) * 8);
      const uint4 v[2] = {sym[0], sym[1]};
      ha = iva, hb = ivb;
#pragma unroll
      for (int b = 0; b < 2; b++) {
        __builtin_amdgcn_wave_barrier();
        row[i] = v[b].x, row[4 + i] = v[b].y, row[8 + i] = v[b].z, row[12 + i] = v[b].w;
        __builtin_amdgcn_wave_barrier();
        compress(row, ha, hb, 64, b == 0 ? B3_CHUNK_START : (B3_CHUNK_END | B3_ROOT));
      }
    }
    uint32_t *to = digest_at(0, quad);
    to[i] = ha, to[4 + i] = hb;
    if (first + quad < n) out[8 * (first + quad) + i] = ha, out[8 * (first + quad) + 4 + i] = hb;
  } else {
    const uint64_t q = 2 * first + tid;  // two quads of words a digest, a row of four to two digests
    if (q < 2 * n) *reinterpret_cast<uint4 *>(rows[0] + (tid >> 2) * QUAD_ROW + (tid & 3) * 4) = reinterpret_cast<const uint4 *>(level)[q];
  }
  uint32_t width = BOTTOM;
  for (int s = 1; s <= height; s++) {
    __syncthreads();
    out += 8 * count;
    count /= 2, first /= 2, width /= 2;
    if (quad < width && first + quad < count) {
      uint32_t a = iva, b = ivb;
      compress(rows[(s - 1) & 1] + quad * QUAD_ROW, a, b, 64, B3_CHUNK_START | B3_CHUNK_END | B3_ROOT);
      uint32_t *to = digest_at(s & 1, quad);
      to[i] = a, to[4 + i] = b;
      out[8 * (first + quad) + i] = a, out[8 * (first + quad) + 4 + i] = b;
    }
  }
  if (cap_out) {
    __syncthreads();
    for (uint32_t w = tid; w < 8 * width; w += THREADS)
      if (first + w / 8 < count)
        __hip_atomic_store(cap_out + 8 * first + w, ((unsigned long long)seq << 32) | digest_at(height & 1, w / 8)[w % 8],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
static_assert(1 << QUAD_LEAF_HEIGHT == QUAD_LEAF_THREADS / 4 && 1 << QUAD_NODE_HEIGHT == QUAD_NODE_THREADS / 2, "a workgroup's own tree");

// a tree of a single leaf: its digest is the whole tree
template <int LEAVES>
__global__ void single_leaf_kernel(uint32_t *level, const uint32_t *cw, int ncols, uint64_t cw_len) {
  if (threadIdx.x || blockIdx.x) return;
  uint32_t h[8];
  if (LEAVES == 1)
    column_leaf_digest(cw, ncols, cw_len, 0, h);
  else
    oracle_leaf_digest(cw, 0, h);
  store_digest(level, h);
}

static int cap_level_of(uint64_t leaves) {  // src/pcs.lisp:57-59
  int il = 0;
  for (uint64_t v = leaves; v; v >>= 1) il++;
  return il - 1 - 7 > 0 ? il - 1 - 7 : 0;
}

// Every level of the tree at d_levels (leaves first), a few launches of up to nine levels each; the
// leaf digests are computed by the first launch (leaves 1: ncols codewords, 2: an oracle codeword) or
// already there (0).  A single leaf (no node above it) is hashed by the same kernel's bottom step.
// With cap_out (an oracle's tree, of two leaves or more) the tree ends at its cap, and the launch that reaches it
// writes the cap to the host, see subtree_kernel: nobody reads the levels above.  Seven levels of one compression's
// latency and one or two launches less per oracle: an opening at nv = 23 (eight oracles) 1312 -> 1207 us.  Not for a
// tree that is handed out: the words arrive before the launch has ended, when a reader on another stream may not yet
// look at the levels.
static int merkle_tree_launch(uint32_t *d_levels, uint64_t nleaves, int leaves, const uint32_t *cw, int ncols,
                              uint64_t cw_len, uint64_t *cap_rows, uint64_t *cap_off_words,
                              unsigned long long *cap_out = nullptr, uint32_t seq = 0) {
  Context &c = ctx();
  uint32_t *level = d_levels;
  uint64_t n = nleaves;
  int lc = cap_level_of(nleaves);
  uint64_t cap_off = 0;
  for (int l = 0; l < lc; l++) cap_off += 8 * (nleaves >> l);
  if (nleaves == 1 && leaves == 1)
    hipLaunchKernelGGL(single_leaf_kernel<1>, dim3(1), dim3(64), 0, c.stream, level, cw, ncols, cw_len);
  if (nleaves == 1 && leaves == 2)
    hipLaunchKernelGGL(single_leaf_kernel<2>, dim3(1), dim3(64), 0, c.stream, level, cw, ncols, cw_len);
  const uint64_t stop = cap_out ? nleaves >> lc : 1;
  while (n > stop || (cap_out && leaves != 0)) {
    int height = 0;
    // The launch that hashes the leaves climbs few levels: above the leaves every level halves the threads at work
    // and costs a whole compression's latency, so a workgroup of a tall launch idles most of its life (measured at
    // 2^22 leaves: 246 us with nine levels in the first launch, 198 us with five, 175 us with three; five leaves the
    // fewest launches above -- over digests only, nine levels each -- and the shortest commit, 0.51 against 0.55 ms).
    static const int leaf_height = getenv("EXH_MERKLE_LEAF_HEIGHT") ? atoi(getenv("EXH_MERKLE_LEAF_HEIGHT")) : 5;
    // Four lanes a compression while that is what fills the device.  Whole commitments, a thread against four lanes:
    // 2^13 leaves of 70 columns 126 against 79 us, 2^16 leaves of 100 columns 240 against 195 and of 2 columns 73
    // against 66; 2^17 leaves 72 and 72, 2^18 91 against 97, 2^20 156 against 214 (the third more instructions).
    // Digests: under 2^22 leaves of two columns, 2^17 digests and fewer, 435 against 426; 2^18 to 2^20 digests level.
    const bool quads = n <= (leaves ? QUAD_LEAVES : QUAD_DIGESTS);
    const int max_height = quads ? (leaves ? QUAD_LEAF_HEIGHT : QUAD_NODE_HEIGHT) : leaves ? leaf_height : 9;
    for (uint64_t v = n; v > stop && height < max_height; v >>= 1) height++;
    unsigned long long *const out = n >> height == stop ? cap_out : nullptr;
    const uint64_t bottom = quads ? (leaves ? QUAD_LEAF_THREADS / 4 : QUAD_NODE_THREADS / 2) : 2 * BLOCK;
    uint32_t grid = (uint32_t)((n + bottom - 1) / bottom);
    c.prof_begin(leaves == 1 ? "merkle_leaves" : leaves == 2 ? "merkle_oracle_leaves" : "merkle_levels", 0,
                 (leaves == 1 ? (uint64_t)ncols * 16 * n : leaves == 2 ? 128 * n : 0) + 64 * n);
    if (quads && leaves == 1)
      hipLaunchKernelGGL((quad_tree_kernel<1, QUAD_LEAF_THREADS>), dim3(grid), dim3(QUAD_LEAF_THREADS), 0, c.stream, level, n,
                         height, cw, ncols, cw_len, out, seq);
    else if (quads && leaves == 2)
      hipLaunchKernelGGL((quad_tree_kernel<2, QUAD_LEAF_THREADS>), dim3(grid), dim3(QUAD_LEAF_THREADS), 0, c.stream, level, n,
                         height, cw, ncols, cw_len, out, seq);
    else if (quads)
      hipLaunchKernelGGL((quad_tree_kernel<0, QUAD_NODE_THREADS>), dim3(grid), dim3(QUAD_NODE_THREADS), 0, c.stream, level, n,
                         height, cw, ncols, cw_len, out, seq);
    else if (leaves == 1)
      hipLaunchKernelGGL(subtree_kernel<1>, dim3(grid), dim3(BLOCK), 0, c.stream, level, n, height, cw, ncols, cw_len, out,
                         seq);
    else if (leaves == 2)
      hipLaunchKernelGGL(subtree_kernel<2>, dim3(grid), dim3(BLOCK), 0, c.stream, level, n, height, cw, ncols, cw_len, out,
                         seq);
    else
      hipLaunchKernelGGL(subtree_kernel<0>, dim3(grid), dim3(BLOCK), 0, c.stream, level, n, height, cw, ncols, cw_len, out,
                         seq);
    c.prof_end();
    leaves = 0;
    for (int s = 0; s < height; s++) {
      level += 8 * n;
      n /= 2;
    }
  }
  EXH_HIP(hipGetLastError());
  *cap_rows = nleaves >> lc;
  *cap_off_words = cap_off;
  return OK;
}
__global__ void deliver_kernel(const uint32_t *src, uint32_t words, unsigned long long *host_dst, uint32_t seq);
static bool await_words(Context &c, const volatile unsigned long long *w, size_t n, uint32_t seq, uint32_t *out);
constexpr size_t CAP_PIN = 32768 + 40 * 40;  // (BaseFold's first cap slot: a commitment and an opening never overlap)

static int merkle_tree_device(uint32_t *d_levels, uint64_t nleaves, int leaves, const uint32_t *cw, int ncols,
                              uint64_t cw_len, uint8_t *cap, uint64_t *cap_rows) {
  Context &c = ctx();
  uint64_t cap_off = 0;
  int status = merkle_tree_launch(d_levels, nleaves, leaves, cw, ncols, cw_len, cap_rows, &cap_off);
  if (status) return status;
  // The cap comes to the host as the oracles' caps of BaseFold do: a small launch writes its words into pinned
  // memory, each with the delivery's number in its upper half, and the host polls them -- no copy to set up and no
  // wait on the stream to wake from (15 us of a commitment).
  if (*cap_rows <= 128 && c.host_pinned_dev && !c.profiling) {
    if (++c.log_seq == 0) ++c.log_seq;
    const uint32_t seq = c.log_seq, words = (uint32_t)(8 * *cap_rows);
    hipLaunchKernelGGL(deliver_kernel, dim3(1), dim3(BLOCK), 0, c.stream, d_levels + cap_off, words,
                       reinterpret_cast<unsigned long long *>(c.host_pinned_dev + CAP_PIN), seq);
    EXH_HIP(hipGetLastError());
    std::vector<uint32_t> cap_words(words);
    if (!await_words(c, reinterpret_cast<const volatile unsigned long long *>(c.host_pinned + CAP_PIN), words, seq,
                     cap_words.data())) {
      set_error("device-error: a commitment's cap did not arrive");
      return E_DEVICE;
    }
    memcpy(cap, cap_words.data(), 4 * (size_t)words);
    return OK;
  }
  EXH_HIP(hipMemcpyAsync(cap, d_levels + cap_off, 32 * *cap_rows, hipMemcpyDeviceToHost, c.stream));
  EXH_HIP(hipStreamSynchronize(c.stream));
  return OK;
}

int merkle_commit_columns(const uint32_t *d_codewords, int ncols, int c, uint32_t *d_levels, uint8_t *cap,
                          uint64_t *cap_rows) {
  Context &cx = ctx();
  int status = cx.require();
  if (status) return status;
  uint64_t nleaves = (uint64_t)1 << (c - 1), cw_len = (uint64_t)1 << (c + 1);
  return merkle_tree_device(d_levels, nleaves, 1, d_codewords, ncols, cw_len, cap, cap_rows);
}

// ---- trees of mixed height (src/pcs.lisp:64-77): a shorter class's leaf digests are hashed into the level of the
// taller class's tree that has as many nodes, node = H(H(left, right), injected).  One launch per level (these
// trees sit beside the large single-class ones, whose levels go nine to a launch).
__global__ __launch_bounds__(BLOCK) void node_level_kernel(const uint32_t *below, uint32_t *level, uint64_t count,
                                                           const uint32_t *inj0, const uint32_t *inj1) {
  const uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i >= count) return;
  uint32_t left[8], right[8], h[8], t[8];
  load_digest(below + 16 * i, left);
  load_digest(below + 16 * i + 8, right);
  b3_node(left, right, h);
  if (inj0) {
    load_digest(inj0 + 8 * i, right);
    b3_node(h, right, t);
#pragma unroll
    for (int k = 0; k < 8; k++) h[k] = t[k];
  }
  if (inj1) {
    load_digest(inj1 + 8 * i, right);
    b3_node(h, right, t);
#pragma unroll
    for (int k = 0; k < 8; k++) h[k] = t[k];
  }
  store_digest(level + 8 * i, h);
}

int merkle_levels_injected_device(const uint32_t *d_leaves, uint64_t nleaves, int ninj, const int *inj_level,
                                  const uint32_t *const *d_inj, uint32_t *d_levels) {
  Context &c = ctx();
  int status = c.require();
  if (status) return status;
  if (nleaves == 0 || (nleaves & (nleaves - 1))) {
    set_error("invalid-parameter: a tree has a power of two of leaves");
    return E_PARAM;
  }
  EXH_HIP(hipMemcpyAsync(d_levels, d_leaves, nleaves * 32, hipMemcpyDeviceToDevice, c.stream));
  uint32_t *below = d_levels;
  uint64_t n = nleaves;
  for (int l = 1; n > 1; l++) {
    uint32_t *level = below + 8 * n;
    n /= 2;
    const uint32_t *inj[2] = {nullptr, nullptr};
    int found = 0;
    for (int k = 0; k < ninj; k++)
      if (inj_level[k] == l) {
        if (found == 2) {
          set_error("invalid-parameter: at most two classes are injected into one level");
          return E_PARAM;
        }
        inj[found++] = d_inj[k];
      }
    hipLaunchKernelGGL(node_level_kernel, dim3((uint32_t)((n + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, c.stream, below,
                       level, n, inj[0], inj[1]);
    below = level;
  }
  EXH_HIP(hipGetLastError());
  return OK;
}

// ------------------------------------------------------------------ BaseFold
// DOT-PAIRS (src/pcs.lisp:473-483) for the three parities at once: sums over pairs of
// pick(tt) pick(et), pick = even entry, odd entry, 2 odd - even.  Partials per workgroup.
// Bound by memory: a wavefront's loads of a pair touch 8 KiB a quarter of a line at a time, and with more of them on a
// compute unit than its L1 holds lines for, the quarters come from L2 again.  Three wavefronts a SIMD, tables of 2^22 and
// 2^24: 51.7 and 213 us; five, as many as the registers allow, 58.7 and 266; four 75 and 278; two 54.3 and 214.
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(3, 3))) void dot_pairs_kernel(const uint32_t *tt, const uint32_t *et, uint64_t n_pairs,
                                                          uint32_t *partials) {
  AccLazy acc[3][8];
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int c = 0; c < 8; c++) acc_zero(acc[k][c]);
  for (uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; i < n_pairs; i += (uint64_t)gridDim.x * BLOCK) {
    Ext<8> t0 = load_ext<8>(tt + 2 * i * 8), t1 = load_ext<8>(tt + (2 * i + 1) * 8);
    Ext<8> e0 = load_ext<8>(et + 2 * i * 8), e1 = load_ext<8>(et + (2 * i + 1) * 8);
    ext_mul_acc<8>(acc[0], t0, e0);
    ext_mul_acc<8>(acc[1], t1, e1);
    Ext<8> t2 = ext_sub<8>(ext_add<8>(t1, t1), t0), e2 = ext_sub<8>(ext_add<8>(e1, e1), e0);
    ext_mul_acc<8>(acc[2], t2, e2);
  }
  __shared__ uint32_t lds[BLOCK / 64][24];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 3; k++)
#pragma unroll
    for (int c = 0; c < 8; c++) {
      uint32_t v = wave_sum(acc_reduce(acc[k][c]));
      if (lane == 0) lds[wave][k * 8 + c] = v;
    }
  __syncthreads();
  if (threadIdx.x < 24) {
    uint32_t v = lds[0][threadIdx.x];
    for (int w = 1; w < BLOCK / 64; w++) v = fadd(v, lds[w][threadIdx.x]);
    partials[(uint64_t)blockIdx.x * 24 + threadIdx.x] = v;
  }
}

__global__ __launch_bounds__(BLOCK) void sum_columns_kernel(const uint32_t *partials, uint32_t nblocks, uint32_t width,
                                                            uint32_t *sums) {
  __shared__ uint32_t lds[BLOCK / 64];
  uint32_t o = blockIdx.x, v = 0;
  for (uint32_t b = threadIdx.x; b < nblocks; b += BLOCK) v = fadd(v, partials[(uint64_t)b * width + o]);
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < BLOCK / 64; w++) v = fadd(v, lds[w]);
    sums[o] = v;
  }
}

// out[x] = h[x] + scale * column[x] over extension tables (h null: zero): the opening's table per class is the
// sum of its units' columns, each times the unit's scalar (src/pcs.lisp:709-716)
template <int D>
__global__ __launch_bounds__(BLOCK) void scale_add_kernel(const uint32_t *h, const uint32_t *column, uint32_t *out,
                                                          uint64_t len, RoundArgs<D> args) {
  uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i >= len) return;
  Ext<D> sc;
#pragma unroll
  for (int c = 0; c < D; c++) sc.c[c] = args.r_mont[c];
  Ext<D> v = ext_mul_mont<D>(sc, load_ext<D>(column + i * D));
  if (h) v = ext_add<D>(v, load_ext<D>(h + i * D));
  store_ext<D>(out + i * D, v);
}
template <int D>
static void scale_add_launch(const uint32_t *h, const uint32_t *column, uint32_t *out, uint64_t len,
                             const uint32_t *scale) {
  RoundArgs<D> a;
  memset(&a, 0, sizeof(a));
  for (int k = 0; k < D; k++) a.r_mont[k] = to_mont(scale[k] % P);
  uint32_t grid = (uint32_t)((len + BLOCK - 1) / BLOCK);
  hipLaunchKernelGGL(scale_add_kernel<D>, dim3(grid), dim3(BLOCK), 0, ctx().stream, h, column, out, len, a);
}
int scale_add_device(int D, const uint32_t *d_h, const uint32_t *d_column, uint64_t len, const uint32_t *scale,
                     uint32_t *d_out) {
  int status = ctx().require();
  if (status) return status;
  if (D == 4)
    scale_add_launch<4>(d_h, d_column, d_out, len, scale);
  else
    scale_add_launch<8>(d_h, d_column, d_out, len, scale);
  EXH_HIP(hipGetLastError());
  return OK;
}

// DOT-PAIRS of two device tables of len EXT8s for the three parities: out[parity][8] on the host (one wait)
int dot_pairs_device(const uint32_t *d_e, const uint32_t *d_v, uint64_t len, uint32_t *out) {
  Context &c = ctx();
  int status = c.require();
  if (status) return status;
  const uint64_t n_pairs = len / 2;
  const uint32_t grid = (uint32_t)std::min<uint64_t>((n_pairs + BLOCK - 1) / BLOCK, 1024);
  uint32_t *scratch = (uint32_t *)c.pool.alloc(((size_t)grid * 24 + 24) * 4);
  if (!scratch) {
    set_error("device-out-of-memory: dot-pairs partial sums");
    return E_NOMEM;
  }
  uint32_t *sums = scratch + (size_t)grid * 24;
  hipLaunchKernelGGL(dot_pairs_kernel, dim3(grid), dim3(BLOCK), 0, c.stream, d_e, d_v, n_pairs, scratch);
  hipLaunchKernelGGL(sum_columns_kernel, dim3(24), dim3(BLOCK), 0, c.stream, scratch, grid, 24u, sums);
  EXH_HIP(hipMemcpyAsync(out, sums, 96, hipMemcpyDeviceToHost, c.stream));
  EXH_HIP(hipStreamSynchronize(c.stream));
  c.pool.release(scratch);
  return OK;
}

// ---- DOT-PAIRS once more for callers that must not allocate: the workgroups' partial sums live in a static
// device array instead of a pooled buffer, and the 24 words of the result come back through the pinned host
// buffer the context has held since exh_init.  The array's name is a host-side stand-in: the address kernels
// can use comes from hipGetSymbolAddress, once per device, with that device current (each GPU holds its own
// copy of the array at its own address).  Every call on a GPU shares that GPU's array: calls that overlap on one
// GPU race.  A launch writes every word it later reads, so nothing has to be cleared between calls.
constexpr uint32_t STATIC_DOT_GRID = 512;                    // workgroups of the launch
constexpr uint64_t STATIC_DOT_MAX_LEN = (uint64_t)1 << 26;   // EXT8s per table: 2 GiB each
constexpr size_t STATIC_DOT_RESULT_AT = 4096;                // word of the pinned buffer the result lands at
static __device__ __align__(256) uint32_t scratch[STATIC_DOT_GRID * 24];  // 48 KiB per GPU until the process ends
constexpr int STATIC_MAX_DEVICES = 64;
static uint32_t *g_scratch_ptr[STATIC_MAX_DEVICES];

// the sums of the partial rows, written where `sums` points (mapped host memory here)
__global__ __launch_bounds__(BLOCK) void sum_columns_to_host_kernel(const uint32_t *partials, uint32_t nblocks,
                                                                    uint32_t width, uint32_t *sums) {
  __shared__ uint32_t lds[BLOCK / 64];
  uint32_t o = blockIdx.x, v = 0;
  for (uint32_t b = threadIdx.x; b < nblocks; b += BLOCK) v = fadd(v, partials[(uint64_t)b * width + o]);
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < BLOCK / 64; w++) v = fadd(v, lds[w]);
    __hip_atomic_store(sums + o, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

int dot_pairs_static_setup(int device) {
  if (device < 0 || device >= STATIC_MAX_DEVICES) {
    set_error("invalid-parameter: device index beyond the static scratch table");
    return E_PARAM;
  }
  if (g_scratch_ptr[device]) return OK;
  uint32_t *ptr = nullptr;
  EXH_HIP(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = ptr;
  return OK;
}

int dot_pairs_static_device(const uint32_t *d_e, const uint32_t *d_v, uint64_t len, uint32_t *out) {
  Context &c = ctx();
  int status = c.require();
  if (status) return status;
  if (len > STATIC_DOT_MAX_LEN) {
    set_error("invalid-parameter: dot-pairs without allocation takes tables of at most 2^26 EXT8s");
    return E_PARAM;
  }
  uint32_t *partials = c.device >= 0 && c.device < STATIC_MAX_DEVICES ? g_scratch_ptr[c.device] : nullptr;
  if (!partials) {
    set_error("device-error: the static scratch array was not set up on this device");
    return E_DEVICE;
  }
  const uint64_t n_pairs = len / 2;
  const uint32_t grid = (uint32_t)std::min<uint64_t>((n_pairs + BLOCK - 1) / BLOCK, STATIC_DOT_GRID);
  hipLaunchKernelGGL(dot_pairs_kernel, dim3(grid), dim3(BLOCK), 0, c.stream, d_e, d_v, n_pairs, partials);
  hipLaunchKernelGGL(sum_columns_to_host_kernel, dim3(24), dim3(BLOCK), 0, c.stream, partials, grid, 24u,
                     c.host_pinned_dev + STATIC_DOT_RESULT_AT);
  EXH_HIP(hipGetLastError());
  EXH_HIP(hipStreamSynchronize(c.stream));
  memcpy(out, c.host_pinned + STATIC_DOT_RESULT_AT, 96);
  return OK;
}

// FOLD-TABLE (src/field.lisp:365-370) of extension tables
template <int D>
__global__ __launch_bounds__(BLOCK) void fold_table_kernel(const uint32_t *in, uint32_t *out, uint64_t n_out,
                                                           RoundArgs<D> args) {
  uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i >= n_out) return;
  Ext<D> r;
#pragma unroll
  for (int c = 0; c < D; c++) r.c[c] = args.r_mont[c];
  store_ext<D>(out + i * D, fold_ext<D>(load_ext<D>(in + 2 * i * D), load_ext<D>(in + (2 * i + 1) * D), r));
}
template <int D>
static void fold_table_launch(const uint32_t *in, uint32_t *out, uint64_t n_out, const uint32_t *r) {
  RoundArgs<D> a;
  memset(&a, 0, sizeof(a));
  for (int k = 0; k < D; k++) a.r_mont[k] = to_mont(r[k] % P);
  uint32_t grid = (uint32_t)((n_out + BLOCK - 1) / BLOCK);
  hipLaunchKernelGGL(fold_table_kernel<D>, dim3(grid), dim3(BLOCK), 0, ctx().stream, in, out, n_out, a);
}
int fold_table_device(int D, const uint32_t *d_in, uint64_t len, const uint32_t *r, uint32_t *d_out) {
  int status = ctx().require();
  if (status) return status;
  if (D == 4)
    fold_table_launch<4>(d_in, d_out, len / 2, r);
  else
    fold_table_launch<8>(d_in, d_out, len / 2, r);
  EXH_HIP(hipGetLastError());
  return OK;
}

// EXT8 table (entries x 8) <-> 8 coordinate columns, for ENCODE-EXT (src/pcs.lisp:569-575)
__global__ __launch_bounds__(BLOCK) void split_coords_kernel(const uint32_t *table, uint32_t *cols, uint64_t len) {
  uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i >= len) return;
  Ext<8> e = load_ext<8>(table + i * 8);
#pragma unroll
  for (int d = 0; d < 8; d++) cols[(uint64_t)d * len + i] = e.c[d];
}
__global__ __launch_bounds__(BLOCK) void join_coords_kernel(const uint32_t *cols, uint32_t *table, uint64_t len) {
  uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (i >= len) return;
  Ext<8> e;
#pragma unroll
  for (int d = 0; d < 8; d++) e.c[d] = cols[(uint64_t)d * len + i];
  store_ext<8>(table + i * 8, e);
}

namespace {
struct Owned {
  std::vector<void *> ptrs;
  ~Owned() {
    for (void *p : ptrs) ctx().pool.release(p);
  }
  uint32_t *alloc(uint64_t words) {
    void *p = ctx().pool.alloc(words * 4);
    if (!p) {
      set_error("device-out-of-memory: BaseFold buffers");
      return nullptr;
    }
    ptrs.push_back(p);
    return (uint32_t *)p;
  }
};
struct OracleTree {
  int level;
  uint32_t *cw, *levels;
  uint64_t cw_len, nleaves;
  int lc;
};
}  // namespace

// OPEN-QUERIES' two gathers for one (unit, class) (src/pcs.lisp:721-734).  Leaves: out[(q * ncols + k) * 4 + s] =
// symbol 4 * leaf_q + s of column k (LEAF-ROWS, src/pcs.lisp:275-277, as the (Q, rows, 4) array of
// FIELD-ARRAY-OF-LEAVES, :659-665): one thread per (q, k), one 16-byte load.
__global__ __launch_bounds__(BLOCK) void open_leaves_kernel(const uint32_t *cw, uint64_t cw_len, uint32_t ncols,
                                                            const uint64_t *leaf, uint32_t count, uint32_t *out) {
  uint64_t gid = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (gid >= (uint64_t)count * ncols) return;
  uint32_t q = (uint32_t)(gid / ncols), k = (uint32_t)(gid % ncols);
  const uint4 v = *(const uint4 *)(cw + (uint64_t)k * cw_len + 4 * leaf[q]);
  *(uint4 *)(out + gid * 4) = v;
}

// Paths: out[(q * depth + d) * 8 ..] = the sibling of leaf_q's ancestor on level d (PATH, src/pcs.lisp:79-84); the
// levels lie leaves first, level d at digest 2 * nleaves - 2 * (nleaves >> d).  One thread per digest word.
__global__ __launch_bounds__(BLOCK) void open_paths_kernel(const uint32_t *levels, uint64_t nleaves, uint32_t depth,
                                                           const uint64_t *leaf, uint32_t count, uint32_t *out) {
  uint64_t gid = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
  if (gid >= (uint64_t)count * depth * 8) return;
  uint32_t w = (uint32_t)(gid % 8), d = (uint32_t)((gid / 8) % depth), q = (uint32_t)(gid / 8 / depth);
  uint64_t start = 2 * nleaves - 2 * (nleaves >> d);
  out[gid] = levels[(start + ((leaf[q] >> d) ^ 1)) * 8 + w];
}

int open_queries_device(const uint32_t *d_codewords, int ncols, int c, const uint32_t *d_levels, const uint64_t *leaves,
                        int count, uint32_t *out_leaves, uint8_t *out_paths, int *out_depth) {
  Context &cx = ctx();
  int status = cx.require();
  if (status) return status;
  const uint64_t nleaves = (uint64_t)1 << (c - 1), cw_len = (uint64_t)1 << (c + 1);
  const uint32_t depth = d_levels ? (uint32_t)cap_level_of(nleaves) : 0;
  if (out_depth) *out_depth = (int)depth;
  if (count == 0) return OK;
  const uint64_t leaf_words = (uint64_t)count * ncols * 4, path_words = (uint64_t)count * depth * 8;
  // one pooled buffer: the indices (padded to 16 bytes: the leaves are stored as uint4), the leaves, the paths
  const size_t idx_slots = ((size_t)count + 1) & ~(size_t)1;
  uint64_t *d_idx = (uint64_t *)cx.pool.alloc(idx_slots * 8 + (leaf_words + path_words) * 4);
  if (!d_idx) {
    set_error("device-out-of-memory: query openings");
    return E_NOMEM;
  }
  uint32_t *d_leaf_out = (uint32_t *)(d_idx + idx_slots), *d_path_out = d_leaf_out + leaf_words;
  hipError_t e = hipMemcpyAsync(d_idx, leaves, (size_t)count * 8, hipMemcpyHostToDevice, cx.stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(open_leaves_kernel, dim3((uint32_t)(((uint64_t)count * ncols + BLOCK - 1) / BLOCK)), dim3(BLOCK),
                       0, cx.stream, d_codewords, cw_len, (uint32_t)ncols, d_idx, (uint32_t)count, d_leaf_out);
    if (path_words)
      hipLaunchKernelGGL(open_paths_kernel, dim3((uint32_t)((path_words + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0,
                         cx.stream, d_levels, nleaves, depth, d_idx, (uint32_t)count, d_path_out);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(out_leaves, d_leaf_out, leaf_words * 4, hipMemcpyDeviceToHost, cx.stream);
  if (e == hipSuccess && path_words)
    e = hipMemcpyAsync(out_paths, d_path_out, path_words * 4, hipMemcpyDeviceToHost, cx.stream);
  hipError_t e2 = hipStreamSynchronize(cx.stream);  // the indices (pageable) and the pooled buffer are free after this
  cx.pool.release(d_idx);
  EXH_HIP(e);
  EXH_HIP(e2);
  return OK;
}

// ------------------------------------------------------------------ BASEFOLD's rounds
// The sumcheck of eq(rr, x) Phi(x) never needs the eq table or its folds.  After i rounds the folded eq table is
// prf_i eq(rr[i..], .) with prf_i = prod_{j<i} eq1(r_j, x_j), so with E = eq(rr[i+1..], .) over the pairs k,
//   DOT-PAIRS(tt, et, 0) = prf_i (1 - r_i) h0,  h0 = sum_k E[k] tt[2k]
//   DOT-PAIRS(tt, et, 1) = prf_i r_i h1,        h1 = sum_k E[k] tt[2k+1]
//   DOT-PAIRS(tt, et, 2) = prf_i (2 r_i - (1 - r_i)) (2 h1 - h0)
// (src/pcs.lisp:473-483, 607-612): the same field elements, from two weighted sums of the message table with split
// weights E[k] = LOW[k mod |LOW|] HIGH[k div |LOW|] as in the sumcheck prover (src/sumcheck.lisp:37-49).
//
// One launch per round does both of the round's passes over memory: its first workgroups fold the message table
// by the last challenge (FOLD-TABLE, src/field.lisp:365-370) and take h0, h1 of the folded table in the same
// pass; the others fold the codeword (RS:FOLD, src/rs.lisp:93-101).  The sums meet in counted totals (RoundTotals)
// and the last summing workgroup to arrive writes them into pinned host memory and raises a flag there, so the
// host neither copies nor waits on the stream: it polls the flag while the codeword's workgroups still run.
// A round whose message and challenge the device takes care of: what the elected workgroup's first wavefront needs for
// that, and where it leaves the results.
struct BfRound {
  DevB3S state;        // the transcript before the message
  uint32_t c[3][8];    // message k = c_k (h_k + ysum), h_2 = 2 h_1 - h_0; times R
  uint32_t ysum[8];
  uint32_t *r_out;     // the challenge times R, for the launches behind this one (device memory; null: the host's round)
  // pinned host memory: the message's 24 words, the challenge's 8, the transcript's state behind it, and a status word
  // (1: the totals did not complete), as 64-bit words (host_seq << 32 | value)
  unsigned long long *host_log;
  uint32_t host_seq;
};
constexpr uint32_t BF_LOG_WORDS = 24 + 8 + sizeof(DevB3S) / 4 + 1;
static_assert(BF_LOG_WORDS <= 64, "a word a lane");

struct BfStepArgs {
  // the message table's part: workgroups [0, tt_blocks)
  const uint32_t *tt_in;  // 4 entries per pair when folding, else 2
  uint32_t *tt_out;       // the folded table (fold)
  const uint32_t *low, *high;
  uint64_t n_pairs;  // pairs after the fold
  uint32_t low_bits, pairs_per_thread, fold, do_sums, tt_blocks;
  uint32_t r_mont[8];
  const uint32_t *r_dev;  // the fold's challenge, times R, where the device's round left it (null: r_mont)
  RoundTotals totals;
  BfRound round;
  // 17 64-bit words in pinned host memory, each (host_seq << 32 | value): h0, h1, then 1 when the totals never
  // completed.  Every word says itself that it has arrived, so no fence orders them: a release at system scope
  // writes back the whole L2 of the elected workgroup's XCD, which the fold's stores of the other workgroups keep
  // dirty (measured: 90 us per round)
  unsigned long long *host_out;
  uint32_t host_seq;
  // the codeword's part: workgroups [tt_blocks, gridDim.x)
  const uint32_t *cw_in, *tw_inv2;
  uint32_t *cw_out;
  uint64_t cw_m;  // elements after the fold
};

// the challenge that a step folds by
__device__ __forceinline__ Ext<8> bf_challenge(const BfStepArgs &a) {
  Ext<8> r;
  const uint32_t *from = a.r_dev ? a.r_dev : a.r_mont;
#pragma unroll
  for (int c = 0; c < 8; c++) r.c[c] = from[c];
  return r;
}

// What the first wavefront fetches for a device's round before the sums' exchange, which hides the trip.
struct BfRoundWords {
  uint32_t c, ysum, state;
};
__device__ __forceinline__ BfRoundWords bf_round_fetch(const BfRound &r) {
  const uint32_t lane = threadIdx.x & 63;
  return {(&r.c[0][0])[lane < 24 ? lane : 0], r.ysum[lane % 8],
          reinterpret_cast<const uint32_t *>(&r.state)[lane < sizeof(DevB3S) / 4 ? lane : 0]};
}
// A round's end on the device (the elected workgroup's first wavefront; sums: h0 and h1 in LDS, 16 words): its message from
// the sums, through the transcript, to the challenge, which goes to device memory for the launches that are already queued
// behind this one and with the message and the transcript's state to the host, which records them.
__device__ __forceinline__ void bf_round_end(const BfRound &r, const BfRoundWords &words, const uint32_t *sums) {
  struct Lds {
    uint32_t chal[8], r_mont[8];
  };
  __shared__ Lds lds;
  __shared__ uint32_t ring[RING_WORDS], map[24], value[3][16];  // map and values in powers of w; the values' triples behind them
  __shared__ DevB3S state;
  const uint32_t lane = threadIdx.x, power = __brev(lane % 8) >> 29;
  if (lane < 24) {
    map[lane / 8 * 8 + power] = words.c;
    const uint32_t h0 = sums[lane % 8], h1 = sums[8 + lane % 8], k = lane / 8;
    const uint32_t v = fadd(k == 0 ? h0 : k == 1 ? h1 : fsub(fdbl(h1), h0), words.ysum);
    value[k][power] = v, value[k][8 + power] = times3(v);
  }
  if (lane < sizeof(DevB3S) / 4) reinterpret_cast<uint32_t *>(&state)[lane] = words.state;
  __builtin_amdgcn_wave_barrier();
  RunB3S tr;
  PendingAppend pending{0, 0, 0};
  rb3s_load(tr, ring, &state);
  const MessageLane<8> ml = message_lane<8>(3);
  const uint32_t o = ml.o < 24 ? ml.o : 23, e = __brev(o % 8) >> 29;
  uint64_t t = 0;
#pragma unroll
  for (uint32_t i = 0; i < 8; i++) {
    if (i >= 4 && i % 2 == 0) t = mont_lazy(t);
    t += (uint64_t)map[o / 8 * 8 + i] * value[o / 8][((e - i) & 7) + (i > e ? 8 : 0)];
  }
  const uint32_t word = mont_reduce4(t);
  transcript_step<8>(tr, nullptr, 0, 3, &lds, ml, word, pending, false, false, [&] {
    __builtin_amdgcn_wave_barrier();
    if (lane < 8) r.r_out[lane] = lds.r_mont[lane];
  });
  rb3s_flush(tr, pending);
  rb3s_store(tr, &state);
  if (ml.part == 0 && ml.o < 24) map[ml.o] = word;
  __builtin_amdgcn_wave_barrier();
  const uint32_t out = lane < 24   ? map[lane]
                       : lane < 32 ? lds.chal[lane - 24]
                       : lane < BF_LOG_WORDS - 1 ? reinterpret_cast<const uint32_t *>(&state)[lane - 32] : 0u;
  if (lane < BF_LOG_WORDS)
    __hip_atomic_store(r.host_log + lane, ((unsigned long long)r.host_seq << 32) | out, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// The sums of a step's workgroup -> totals; the sums over all workgroups (LDS) in the one that arrives last, null in the
// others.  `mine`: the workgroup's `width` words; *ok is false when the totals did not complete.
__device__ __forceinline__ const uint32_t *bf_elect(const RoundTotals &totals, const uint32_t *mine, uint32_t width,
                                                    uint32_t workgroups, bool *ok) {
  __shared__ uint32_t sums[64];
  __shared__ uint32_t scratch[TOTALS_POLLS * BLOCK];
  *ok = true;
  if (workgroups == 1) return mine;  // nobody to wait for
  return add_and_elect(totals, mine, width, scratch, sums, ok, 0, width, workgroups - 1, workgroups) ? sums : nullptr;
}

// ... and to pinned host memory; host_out receives the words and a status word, see BfStepArgs.
__device__ __forceinline__ void bf_deliver_sums(const RoundTotals &totals, const uint32_t *mine, uint32_t width,
                                                uint32_t workgroups, unsigned long long *host_out, uint32_t host_seq) {
  const uint32_t tid = threadIdx.x;
  bool ok;
  const uint32_t *from = bf_elect(totals, mine, width, workgroups, &ok);
  if (from && tid <= width) {
    const uint32_t value = tid < width ? (ok ? from[tid] : 0u) : (ok ? 0u : 1u);
    __hip_atomic_store(host_out + tid, ((unsigned long long)host_seq << 32) | value, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// a step's two weighted sums, accumulated per lane, to their delivery
__device__ __forceinline__ void bf_finish_sums(const BfStepArgs &a, AccLazy (*acc)[8], uint64_t tile_start) {
  __shared__ uint32_t lds[BLOCK / 64][16];
  __shared__ uint32_t mine[16];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  BfRoundWords words{0, 0, 0};
  if (a.round.r_out) words = bf_round_fetch(a.round);
  const uint32_t total = wave_sums_transposed<16>([&](int k) -> uint32_t { return acc_reduce(acc[k / 8][k % 8]); });
  if (transposed_writer<16>(lane)) lds[tid >> 6][transposed_word<16>(lane)] = total;
  __syncthreads();
  if (tid < 2) {  // a workgroup's pairs share one HIGH weight (the tile is |LOW| pairs)
    Ext<8> t;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      uint32_t v = lds[0][tid * 8 + c];
#pragma unroll
      for (int w = 1; w < BLOCK / 64; w++) v = fadd(v, lds[w][tid * 8 + c]);
      t.c[c] = v;
    }
    // times HIGH / R, then times R: the plain product
    t = ext_mul_mont<8>(t, load_ext<8>(a.high + (tile_start >> a.low_bits) * 8));
#pragma unroll
    for (int c = 0; c < 8; c++) mine[tid * 8 + c] = mont_mul(t.c[c], R2);
  }
  __syncthreads();
  if (!a.round.r_out) {
    bf_deliver_sums(a.totals, mine, 16, a.tt_blocks, a.host_out, a.host_seq);
    return;
  }
  bool ok;
  const uint32_t *sums = bf_elect(a.totals, mine, 16, a.tt_blocks, &ok);
  if (!sums || tid >= 64) return;
  if (ok)
    bf_round_end(a.round, words, sums);
  else if (tid < BF_LOG_WORDS)
    __hip_atomic_store(a.round.host_log + tid, ((unsigned long long)a.round.host_seq << 32) | (tid == BF_LOG_WORDS - 1 ? 1u : 0u),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// RS:FOLD of one element: pair (a, b) at twiddle x: f0 = (a + b)/2, f1 = (a - b)/(2x), f0 + r (f1 - f0)
__device__ __forceinline__ void bf_fold_codeword(const BfStepArgs &a, const Ext<8> &r, uint64_t s) {
  if (s >= a.cw_m) return;
  const Ext<8> x = load_ext<8>(a.cw_in + 2 * s * 8), y = load_ext<8>(a.cw_in + (2 * s + 1) * 8);
  const Ext<8> f0 = ext_scale_mont<8>(ext_add<8>(x, y), mont_mul(INV2, R2));
  const Ext<8> f1 = ext_scale_mont<8>(ext_sub<8>(x, y), a.tw_inv2[s]);
  store_ext<8>(a.cw_out + s * 8, ext_add<8>(f0, ext_mul_mont<8>(r, ext_sub<8>(f1, f0))));
}

template <bool FOLD>
__global__ __launch_bounds__(BLOCK) void bf_step_kernel(BfStepArgs a) {
  const uint32_t tid = threadIdx.x;
  const Ext<8> r = bf_challenge(a);
  if (blockIdx.x >= a.tt_blocks) {
    bf_fold_codeword(a, r, (uint64_t)(blockIdx.x - a.tt_blocks) * BLOCK + tid);
    return;
  }
  const uint64_t tile = (uint64_t)BLOCK * a.pairs_per_thread, tile_start = (uint64_t)blockIdx.x * tile;
  const uint64_t low_mask = ((uint64_t)1 << a.low_bits) - 1;
  AccLazy acc[2][8];
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int c = 0; c < 8; c++) acc_zero(acc[q][c]);
  // a pair's words are requested one pair ahead of its arithmetic (Q quads per pair: 8 when folding, else 4)
  constexpr int Q = FOLD ? 8 : 4;
  uint4 raw[Q], ahead[Q];
  Ext<8> w = ext_zero<8>(), w_ahead = ext_zero<8>();
  auto fetch = [&](uint64_t i, uint4 *q, Ext<8> &wq) {
    const uint4 *p = reinterpret_cast<const uint4 *>(a.tt_in) + (uint64_t)Q * i;
#pragma unroll
    for (int j = 0; j < Q; j++) q[j] = p[j];
    if (a.do_sums) wq = load_ext<8>(a.low + (i & low_mask) * 8);
  };
  if (tile_start + tid < a.n_pairs) fetch(tile_start + tid, raw, w);
  for (uint32_t k = 0; k < a.pairs_per_thread; k++) {
    const uint64_t i = tile_start + (uint64_t)k * BLOCK + tid;
    if (i >= a.n_pairs) break;
    const bool more = k + 1 < a.pairs_per_thread && i + BLOCK < a.n_pairs;
    if (more) fetch(i + BLOCK, ahead, w_ahead);
    Ext<8> lo, hi;
    if constexpr (FOLD) {
      lo = fold_ext<8>(ext_from_quads<8>(raw), ext_from_quads<8>(raw + 2), r);
      hi = fold_ext<8>(ext_from_quads<8>(raw + 4), ext_from_quads<8>(raw + 6), r);
      store_ext<8>(a.tt_out + 2 * i * 8, lo);
      store_ext<8>(a.tt_out + (2 * i + 1) * 8, hi);
    } else {
      lo = ext_from_quads<8>(raw), hi = ext_from_quads<8>(raw + 2);
    }
    if (a.do_sums) {
      ext_mul_acc<8>(acc[0], lo, w);  // (the weight second: its tripled wrap coefficients serve both products)
      ext_mul_acc<8>(acc[1], hi, w);
    }
    if (more) {
#pragma unroll
      for (int j = 0; j < Q; j++) raw[j] = ahead[j];
      w = w_ahead;
    }
  }
  if (a.do_sums) bf_finish_sums(a, acc, tile_start);
}

// ---- the first rounds from the committed base columns
// The table that is opened is H = sum_j c_j col_j of few base columns, and its codeword the same combination of
// theirs.  Neither is formed.  With the first LB variables left open, T[b] = sum_k E[k] H[2^LB k + b] over the weights
// E of the variables above them, the rounds 0 .. LB - 1 are the host's: a round's h0, h1 are the sums over T folded by
// the challenges so far, weighted by eq of the open variables above -- one sweep over the base columns (4 bytes an
// entry) in place of LB passes over tables of 32-byte elements.  T[b] is itself sum_j c_j S_j[b] with base-field
// columns under the weights, so an entry costs eight multiply-adds.  Level LB's table comes straight from the base
// columns (2^LB products per column and coordinate: BIND-PREFIX, src/sumcheck.lisp:496-510), and so does the codeword
// of the first level that anybody looks at (level 2, or 1 when a class joins there): both are linear in H.
// At nv = 23 and two columns the combinations and the folds to the table of level 3 and the codeword of level 2 are
// 3.2 GB; this way they are 0.49 GB (by the counters), and an opening of 2^23 x 2 takes 918 us in place of 1517 (the same
// library with every class combined; 2^23 x 8: 1151 and 1589).
// The line at eight columns: their constants (384 bytes a column) fill the 4 KiB of a kernel's arguments.  The two ways
// meet there at 2^20 (base columns and combined, us: 588 / 656 at one column, 618 / 660 at four, 639 / 668 at six, 666 / 668
// at eight), at 2^16 (401 / 449 at one, 450 / 446 at eight) and below (2^13 x 8 305 / 318, 2^10 x 8 211 / 215); above 2^20
// the base columns would still be ahead.
constexpr int BF_BASE_MAX_COLS = 8;  // columns whose constants travel as kernel arguments
constexpr int BF_BASE_BITS = 3;      // variables left open at most: 2^3 sums of eight words in registers

struct BfBaseSumsArgs {
  const uint32_t *cols;  // ncols base columns of len values
  uint64_t len, n_cells;  // cells of 2^LB consecutive entries
  const uint32_t *low, *high;
  uint32_t low_bits, tiles;  // a workgroup takes one column's tile of 2^low_bits cells
  uint32_t coef[BF_BASE_MAX_COLS][8];  // times R^2
  RoundTotals totals;
  unsigned long long *host_out;
  uint32_t host_seq;
};

template <int LB>
__global__ __launch_bounds__(BLOCK) void bf_base_sums_kernel(BfBaseSumsArgs a) {
  constexpr int B = 1 << LB, WORDS = 8 * B, W = WORDS < 32 ? WORDS : 32;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t tile = blockIdx.x % a.tiles, column = blockIdx.x / a.tiles;
  const uint32_t *col = a.cols + (uint64_t)column * a.len;
  const uint64_t first = (uint64_t)tile << a.low_bits;
  const uint64_t left = a.n_cells - first;
  const uint32_t cells = left < ((uint64_t)1 << a.low_bits) ? (uint32_t)left : 1u << a.low_bits;
  uint64_t acc[B][8];
#pragma unroll
  for (int b = 0; b < B; b++)
#pragma unroll
    for (int c = 0; c < 8; c++) acc[b][c] = 0;
  for (uint32_t k = tid; k < cells; k += BLOCK) {
    uint32_t v[B];
    const uint32_t *p = col + (first + k) * B;
    if constexpr (B >= 4) {
#pragma unroll
      for (int q = 0; q < B / 4; q++) {
        const uint4 x = reinterpret_cast<const uint4 *>(p)[q];
        v[4 * q] = x.x, v[4 * q + 1] = x.y, v[4 * q + 2] = x.z, v[4 * q + 3] = x.w;
      }
    } else {
#pragma unroll
      for (int b = 0; b < B; b++) v[b] = p[b];
    }
    const Ext<8> w = load_ext<8>(a.low + (uint64_t)k * 8);
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
      for (int c = 0; c < 8; c++) lazy_mad(acc[b][c], w.c[c], v[b]);
  }
  __shared__ uint32_t lds[BLOCK / 64][WORDS];
  __shared__ uint32_t mine[WORDS];
#pragma unroll
  for (int at = 0; at < WORDS; at += W) {
    const uint32_t total =
        wave_sums_transposed<W>([&](int k) -> uint32_t { return lazy_reduce(acc[(at + k) / 8][(at + k) % 8]); });
    if (transposed_writer<W>(lane)) lds[wave][at + transposed_word<W>(lane)] = total;
  }
  __syncthreads();
  if (tid < B) {  // times the tile's HIGH weight and the column's coefficient
    Ext<8> t, c;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      uint32_t v = lds[0][tid * 8 + k];
#pragma unroll
      for (int w = 1; w < BLOCK / 64; w++) v = fadd(v, lds[w][tid * 8 + k]);
      t.c[k] = v;
      c.c[k] = a.coef[column][k];
    }
    t = ext_mul_mont<8>(ext_mul_mont<8>(t, load_ext<8>(a.high + (uint64_t)tile * 8)), c);
#pragma unroll
    for (int k = 0; k < 8; k++) mine[tid * 8 + k] = t.c[k];
  }
  __syncthreads();
  bf_deliver_sums(a.totals, mine, WORDS, gridDim.x, a.host_out, a.host_seq);
}

struct BfBaseArgs {
  BfStepArgs s;  // the table's part with tt_in unused; the codeword's part with cw_in, tw_inv2 when it is a plain fold
  const uint32_t *cols, *cws;  // ncols base columns of col_len values, their codewords of cw_len symbols
  uint64_t col_len, cw_len;
  uint32_t ncols;
  const uint32_t *tw0, *tw1;  // 1 / (2x) of the codeword's levels 0 and 1
  uint32_t tt_coef[BF_BASE_MAX_COLS][1 << BF_BASE_BITS][8];  // c_j eq((x_0, x_1, ..), b), times R
  uint32_t cw_coef[BF_BASE_MAX_COLS][4][8];                  // c_j {1, x_0, x_1, x_0 x_1}, times R
};
static_assert(sizeof(BfBaseArgs) <= 4096, "kernel arguments");

// TT: the table of level TT from the base columns, with the next round's sums (0: no table part).
// CW: the codeword of level CW = 1 or 2 from the base codewords; 3: a plain fold of a codeword of elements.
template <int TT, int CW>
__global__ __launch_bounds__(BLOCK) void bf_base_kernel(BfBaseArgs a) {
  const uint32_t tid = threadIdx.x;
  if (TT == 0 || blockIdx.x >= a.s.tt_blocks) {
    const uint64_t s = (uint64_t)(blockIdx.x - a.s.tt_blocks) * BLOCK + tid;
    if constexpr (CW == 3) {
      Ext<8> r;
#pragma unroll
      for (int c = 0; c < 8; c++) r.c[c] = a.s.r_mont[c];
      bf_fold_codeword(a.s, r, s);
    } else {
      if (s >= a.s.cw_m) return;
      const uint32_t half = mont_mul(INV2, R2);
      Ext<8> out = ext_zero<8>();
      uint32_t t0[2], t2 = 0;
      if constexpr (CW == 1)
        t0[0] = a.tw0[s];
      else
        t0[0] = a.tw0[2 * s], t0[1] = a.tw0[2 * s + 1], t2 = a.tw1[s];
      for (uint32_t j = 0; j < a.ncols; j++) {
        const uint32_t *cw = a.cws + (uint64_t)j * a.cw_len;
        uint32_t q[4];  // the base values that go with 1, x_0, x_1, x_0 x_1
        if constexpr (CW == 1) {
          const uint2 e = *reinterpret_cast<const uint2 *>(cw + 2 * s);
          q[0] = mont_mul(fadd(e.x, e.y), half);
          q[1] = fsub(mont_mul(fsub(e.x, e.y), t0[0]), q[0]);
        } else {
          const uint4 e = *reinterpret_cast<const uint4 *>(cw + 4 * s);
          // level 1's two elements u + x_0 v; their fold at level 1's twiddle
          const uint32_t u0 = mont_mul(fadd(e.x, e.y), half), v0 = fsub(mont_mul(fsub(e.x, e.y), t0[0]), u0);
          const uint32_t u1 = mont_mul(fadd(e.z, e.w), half), v1 = fsub(mont_mul(fsub(e.z, e.w), t0[1]), u1);
          q[0] = mont_mul(fadd(u0, u1), half), q[1] = mont_mul(fadd(v0, v1), half);
          q[2] = fsub(mont_mul(fsub(u0, u1), t2), q[0]), q[3] = fsub(mont_mul(fsub(v0, v1), t2), q[1]);
        }
#pragma unroll
        for (int c = 0; c < 8; c++) out.c[c] = fadd(out.c[c], mont_dot<CW == 1 ? 2 : 4>(a.cw_coef[j], c, q));
      }
      store_ext<8>(a.s.cw_out + s * 8, out);
    }
    return;
  }
  if constexpr (TT > 0) {
    constexpr int B = 1 << TT;
    const uint64_t tile = (uint64_t)BLOCK * a.s.pairs_per_thread, tile_start = (uint64_t)blockIdx.x * tile;
    const uint64_t low_mask = ((uint64_t)1 << a.s.low_bits) - 1;
    AccLazy acc[2][8];
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int c = 0; c < 8; c++) acc_zero(acc[q][c]);
    for (uint32_t k = 0; k < a.s.pairs_per_thread; k++) {
      const uint64_t i = tile_start + (uint64_t)k * BLOCK + tid;
      if (i >= a.s.n_pairs) break;
      Ext<8> lo = ext_zero<8>(), hi = ext_zero<8>(), w = ext_zero<8>();
      if (a.s.do_sums) w = load_ext<8>(a.s.low + (i & low_mask) * 8);
      for (uint32_t j = 0; j < a.ncols; j++) {
        const uint4 *p = reinterpret_cast<const uint4 *>(a.cols + (uint64_t)j * a.col_len + 2 * B * i);
        uint32_t v[2 * B];
#pragma unroll
        for (int q = 0; q < B / 2; q++) {
          const uint4 x = p[q];
          v[4 * q] = x.x, v[4 * q + 1] = x.y, v[4 * q + 2] = x.z, v[4 * q + 3] = x.w;
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
          lo.c[c] = fadd(lo.c[c], mont_dot<B>(a.tt_coef[j], c, v));
          hi.c[c] = fadd(hi.c[c], mont_dot<B>(a.tt_coef[j], c, v + B));
        }
      }
      store_ext<8>(a.s.tt_out + 2 * i * 8, lo);
      store_ext<8>(a.s.tt_out + (2 * i + 1) * 8, hi);
      if (a.s.do_sums) {
        ext_mul_acc<8>(acc[0], lo, w);
        ext_mul_acc<8>(acc[1], hi, w);
      }
    }
    if (a.s.do_sums) bf_finish_sums(a.s, acc, tile_start);
  }
}

// `count` quads (16 bytes each) from anywhere in device memory into pinned host memory, every word as a 64-bit word
// (seq << 32 | value); `src` lies in pinned memory as well.  The words cross LDS so that neighbouring lanes store
// neighbouring words: what bounds this kernel is the number of writes that reach the host, and a lane storing its own
// quad's four words made every one of them a write of 8 bytes (163 us for the 972 quads of an opening at nv = 23 and
// six queries, 5 us this way).
__global__ __launch_bounds__(BLOCK) void gather_quads_kernel(const uint32_t *const *src, uint32_t count,
                                                             unsigned long long *host_dst, uint32_t seq) {
  __shared__ uint4 quads[BLOCK];
  const uint32_t tid = threadIdx.x, first = blockIdx.x * BLOCK;
  if (first + tid < count) quads[tid] = *reinterpret_cast<const uint4 *>(src[first + tid]);
  __syncthreads();
  const uint32_t words = 4 * (count - first < BLOCK ? count - first : BLOCK);
  const uint32_t *w = reinterpret_cast<const uint32_t *>(quads);
#pragma unroll
  for (uint32_t k = tid; k < 4 * BLOCK; k += BLOCK)
    if (k < words)
      __hip_atomic_store(host_dst + 4 * (uint64_t)first + k, ((unsigned long long)seq << 32) | w[k], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
}

// `words` words from device memory into pinned host memory as 64-bit words (seq << 32 | value), each its own flag
__global__ __launch_bounds__(BLOCK) void deliver_kernel(const uint32_t *src, uint32_t words, unsigned long long *host_dst,
                                                        uint32_t seq) {
  for (uint32_t u = threadIdx.x; u < words; u += BLOCK)
    __hip_atomic_store(host_dst + u, ((unsigned long long)seq << 32) | src[u], __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

// the host's side of such words in pinned memory: true once all n carry seq (their low halves then go to out);
// false when the stream ran dry without them
static bool await_words(Context &c, const volatile unsigned long long *w, size_t n, uint32_t seq, uint32_t *out) {
  auto all_there = [&]() {
    for (size_t u = n; u-- > 0;)
      if ((uint32_t)(w[u] >> 32) != seq) return false;
    return true;
  };
  uint32_t spins = 0;
  bool there = false;
  while (!(there = all_there())) {
    if ((++spins & 1023) == 0 && hipStreamQuery(c.stream) != hipErrorNotReady) break;
  }
  if (!there) {
    (void)hipStreamSynchronize(c.stream);
    if (!all_there()) return false;
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  for (size_t u = 0; u < n; u++) out[u] = (uint32_t)w[u];
  return true;
}

// regions of the context's pinned host buffer BaseFold uses (in 32-bit words): a slot of 17 64-bit words per round,
// a slot of 128 * 8 64-bit words per oracle cap, and above the first 2^16 words a slot of 65 64-bit words per class's
// sums, the point's factors, and a gather's addresses and words
constexpr size_t BF_PIN = 32768, BF_ROUND_SLOT = 40, BF_MAX_ROUNDS = 40, BF_CAP_SLOT = 2048, BF_MAX_ORACLES = 14;
static_assert(CAP_PIN == BF_PIN + BF_MAX_ROUNDS * BF_ROUND_SLOT, "a commitment's cap lands in the first cap slot");
static_assert(BF_PIN + BF_MAX_ROUNDS * BF_ROUND_SLOT + BF_MAX_ORACLES * BF_CAP_SLOT <= 65536, "the rounds' part");
constexpr size_t BF_CLASS_PIN = 65536, BF_CLASS_SLOT = 136, BF_MAX_CLASSES = 32;
constexpr size_t BF_FACTOR_PIN = BF_CLASS_PIN + BF_MAX_CLASSES * BF_CLASS_SLOT, BF_FACTOR_WORDS = 512;
constexpr size_t GATHER_PIN = BF_FACTOR_PIN + BF_FACTOR_WORDS, GATHER_QUADS = 8192;
constexpr size_t BF_LOG_PIN = GATHER_PIN + 10 * GATHER_QUADS, BF_LOG_SLOT = 128;  // a slot per round that the device ends
static_assert(BF_LOG_PIN + BF_MAX_ROUNDS * BF_LOG_SLOT <= ((size_t)1 << 18) && 2 * BF_LOG_WORDS <= BF_LOG_SLOT, "the pinned buffer");
static_assert(BF_LOG_PIN % 2 == 0, "64-bit words");
static_assert(GATHER_PIN % 2 == 0 && BF_CLASS_SLOT % 2 == 0, "64-bit words");
constexpr uint32_t BF_GROUPS = 32;  // rows of totals of a round's sums (16 words each) and of a class's (64 words)

// `quads` (addresses of 16 bytes each in device memory) to the host, four words a quad: the addresses go out and the
// words come back through pinned memory, one launch and one poll per GATHER_QUADS of them, where a copy of the
// addresses, a copy of the words and a wait on the stream are 50 us
static int gather_quads(const std::vector<const uint32_t *> &quads, uint32_t *out) {
  Context &c = ctx();
  for (size_t at = 0; at < quads.size(); at += GATHER_QUADS) {
    const size_t n = std::min(quads.size() - at, GATHER_QUADS);
    memcpy(c.host_pinned + GATHER_PIN, quads.data() + at, n * sizeof(quads[0]));
    if (++c.log_seq == 0) ++c.log_seq;
    constexpr size_t words_at = GATHER_PIN + 2 * GATHER_QUADS;
    hipLaunchKernelGGL(gather_quads_kernel, dim3((uint32_t)((n + BLOCK - 1) / BLOCK)), dim3(BLOCK), 0, c.stream,
                       reinterpret_cast<const uint32_t *const *>(c.host_pinned_dev + GATHER_PIN), (uint32_t)n,
                       reinterpret_cast<unsigned long long *>(c.host_pinned_dev + words_at), c.log_seq);
    EXH_HIP(hipGetLastError());
    if (!await_words(c, reinterpret_cast<const volatile unsigned long long *>(c.host_pinned + words_at), 4 * n, c.log_seq,
                     out + 4 * at)) {
      set_error("device-error: an opening's words did not arrive");
      return E_DEVICE;
    }
  }
  return OK;
}

bool bf_base_source(const uint32_t *columns, const uint32_t *codewords, int ncols, int c) {
  // (whole quads are read: a column of 2^c values and its codeword begin on 16 bytes)
  return columns && codewords && ncols >= 1 && ncols <= BF_BASE_MAX_COLS && c >= 3 &&
         ((reinterpret_cast<uintptr_t>(columns) | reinterpret_cast<uintptr_t>(codewords)) & 15) == 0;
}

// BASEFOLD (src/pcs.lisp:581-657) over ncls size classes, ascending, the last one nv: class c's table (2^c EXT8s)
// joins the message table and the codeword at level nv - c (:590-600, :635-639).  A class given as a table without its
// codeword is encoded here, coordinate by coordinate (ENCODE-EXT); one given by base columns (BfSource) is read from
// them where it is needed: encoding is linear, so the codeword of a combination of committed columns is the same
// combination of their committed codewords.
int basefold_prove_classes(Transcript &tr, int nv, int ncls, const int *cls, const BfSource *src, const uint32_t *rr,
                           const uint32_t *v, int grind_bits, int queries, uint64_t *out_qs, uint32_t *out_chal,
                           uint32_t *out_final, BfMore *more_words) {
  Context &c = ctx();
  int status = c.require();
  if (status) return status;
  if (ncls < 1 || ncls > (int)BF_MAX_CLASSES || cls[ncls - 1] != nv || queries < 1 || nv > 30) {
    set_error("invalid-parameter: basefold takes its classes in ascending order, the largest being nv <= 30");
    return E_PARAM;
  }
  for (int k = 0; k < ncls; k++)
    if (cls[k] < 1 || (k && cls[k] <= cls[k - 1])) {
      set_error("invalid-parameter: basefold classes must ascend");
      return E_PARAM;
    }
  const BfSource &top = src[ncls - 1];
  const int fl = nv - 5 > 0 ? nv - 5 : 0;
  if (fl > (int)BF_MAX_ROUNDS) {
    set_error("invalid-parameter: basefold rounds beyond the buffers");
    return E_PARAM;
  }
  const uint64_t len = (uint64_t)1 << nv;
  Owned mem;
  auto grid_of = [](uint64_t n) { return dim3((uint32_t)((n + BLOCK - 1) / BLOCK)); };
  // ENCODE-EXT of a table of 2^cc EXT8s
  auto encode_ext = [&](const uint32_t *h, int cc) -> uint32_t * {
    const uint64_t n = (uint64_t)1 << cc;
    uint32_t *cols = mem.alloc(n * 8), *cwcols = mem.alloc(2 * n * 8), *cw = mem.alloc(2 * n * 8);
    if (!cols || !cwcols || !cw) {
      status = E_NOMEM;
      return nullptr;
    }
    hipLaunchKernelGGL(split_coords_kernel, grid_of(n), dim3(BLOCK), 0, c.stream, h, cols, n);
    if ((status = rs_encode_columns(cols, 8, cc, cwcols))) return nullptr;
    hipLaunchKernelGGL(join_coords_kernel, grid_of(2 * n), dim3(BLOCK), 0, c.stream, cwcols, cw, 2 * n);
    return cw;
  };
  // The largest class from its base columns: BB variables are left open (see bf_base_sums_kernel), up to the first
  // level a class joins at, since there the table has to exist; the codeword is formed at level CB.
  const bool base = !top.h && fl > 0;
  const int first_join = ncls > 1 ? nv - cls[ncls - 2] : BF_BASE_BITS;
  const int BB = base ? std::min({BF_BASE_BITS, first_join, fl}) : 0, CB = base ? std::min(BB, 2) : 0;
  const uint32_t *tt = top.h, *cw = top.cw;
  if (!base) {
    if (!tt) {  // (no rounds: the table itself goes out)
      uint32_t *h = mem.alloc(len * 8);
      if (!h) return E_NOMEM;
      combine_few_launch<8>(top.columns, top.ncols, len, top.coef, nullptr, h);
      tt = h;
    }
    if (fl > 0 && !cw && !(cw = encode_ext(tt, nv))) return status;
  }
  // the folded message tables ping-pong between two buffers (the class's own table is read in round 0 and never
  // written); so do the folded codewords, except that a level with an oracle tree keeps a buffer of its own
  const uint64_t tt_words = base ? (len >> BB) * 8 : len * 4 + 8, cw_words = base ? (2 * len >> CB) * 8 : len * 8;
  uint32_t *tt_a = mem.alloc(tt_words + 8), *tt_b = mem.alloc(tt_words / 2 + 8);
  uint32_t *cw_b = mem.alloc(cw_words), *cw_c = mem.alloc(cw_words / 2 + 8), *factors = mem.alloc((uint64_t)nv * 16 + 16);
  if (!tt_a || !tt_b || !cw_b || !cw_c || !factors) return E_NOMEM;
  // ---- the point's factors, staged in pinned memory for the launch that builds the weights
  uint32_t *pin_factors = c.host_pinned + BF_FACTOR_PIN;
  static_assert(30 * 16 <= BF_FACTOR_WORDS, "the factors' room");
  for (int b = 0; b < nv; b++)
    for (int k = 0; k < 8; k++) {
      uint32_t r = rr[(size_t)b * 8 + k] % P;
      pin_factors[((size_t)b * 2) * 8 + k] = to_mont(r);
      pin_factors[((size_t)b * 2 + 1) * 8 + k] = to_mont(fsub(k == 0 ? 1u : 0u, r));
    }
  // ---- split weights: round i sums over the pairs k of variables i+1 .. nv-1; LOW covers a workgroup's tile, HIGH the
  // rest.  A class's sums over base columns leave its first bits open and go over the variables above those.
  struct Split {
    int low_bits = 0, rest = 0;
    uint64_t low = 0, high = 0;
  };
  std::vector<int> first, bits;
  std::vector<uint64_t> off;
  uint64_t pos = 0;
  auto split = [&](int from, int low_bits) {
    Split w;
    w.rest = nv - from, w.low_bits = std::min(w.rest, low_bits);
    w.low = pos, first.push_back(from), bits.push_back(w.low_bits), off.push_back(pos);
    pos += (uint64_t)1 << w.low_bits;
    w.high = pos, first.push_back(from + w.low_bits), bits.push_back(w.rest - w.low_bits), off.push_back(pos);
    pos += (uint64_t)1 << (w.rest - w.low_bits);
    return w;
  };
  std::vector<Split> round_w(std::max(fl, 1)), class_w(ncls);
  // (tiles of 2^10 to 2^12 pairs, at least a thousand of them while the table is that large: long tiles in few
  // workgroups trail their loads one after another, short ones pay the reduction and the atomics per tile.  Tables of
  // under 2^18 pairs leave most of the device idle either way and take as many tiles as it has compute units, down to a
  // pair a thread: four pairs one after the other are 2 us of a round, an opening of 2^23 x 2 and 2^19 825 against
  // 787 us, of 2^18 x 2 359 against 328; twice or four times as many tiles made no difference.)
  auto tile_bits = [](int pair_bits) { return std::min(std::max(pair_bits - 10, std::min(std::max(pair_bits - 8, 8), 10)), 12); };
  for (int i = BB; i < fl; i++) round_w[i] = split(i + 1, tile_bits(nv - 1 - i));
  auto open_bits = [&](int k) { return k + 1 == ncls ? BB : BF_BASE_BITS; };
  for (int k = 0; k < ncls; k++)
    if (!src[k].h && (k + 1 < ncls || base)) {
      const int rest = cls[k] - open_bits(k);
      class_w[k] = split(nv - rest, std::min(std::max(rest - 8, 10), 13));
    }
  // ---- the sums' totals, cleared by the launch that builds the weights, and the pinned slots
  const uint64_t round_totals = (uint64_t)std::max(fl, 1) * BF_GROUPS * 16, class_totals = (uint64_t)ncls * BF_GROUPS * 64;
  const uint64_t total_words = 2 * (round_totals + class_totals) + std::max(fl, 1) + ncls;
  uint32_t *totals_mem = mem.alloc(total_words), *weights = mem.alloc(pos * 8 + 8);
  if (!totals_mem || !weights) return E_NOMEM;
  unsigned long long *totals64 = reinterpret_cast<unsigned long long *>(totals_mem);
  uint32_t *arrivals = totals_mem + 2 * (round_totals + class_totals);
  for (size_t t = 0; t < first.size(); t += 64) {
    const int count = (int)std::min<size_t>(64, first.size() - t);
    status = eq_tables_launch(8, count, first.data() + t, bits.data() + t, off.data() + t, factors, nv, weights,
                              t == 0 ? c.host_pinned_dev + BF_FACTOR_PIN : nullptr, totals_mem, t == 0 ? total_words : 0);
    if (status) return status;
  }
  volatile uint32_t *pin = c.host_pinned + BF_PIN;
  uint32_t *pin_dev = c.host_pinned_dev + BF_PIN;
  if (++c.log_seq == 0) ++c.log_seq;  // (a word of an earlier proof carries an earlier number)
  const uint32_t seq = c.log_seq;
  auto groups_of = [](uint32_t workgroups) {
    uint32_t groups = 1;
    while (groups * 2 <= BF_GROUPS && groups * 2 <= workgroups) groups *= 2;
    return groups;
  };
  auto class_slot = [&](int k) { return BF_CLASS_PIN + (size_t)k * BF_CLASS_SLOT; };
  // the sums of class k over its base columns, or h0 and h1 of its table under round nv - c's weights
  auto launch_class_sums = [&](int k) -> int {
    unsigned long long *host_out = reinterpret_cast<unsigned long long *>(c.host_pinned_dev + class_slot(k));
    RoundTotals t{totals64 + round_totals + (uint64_t)k * BF_GROUPS * 64, arrivals + std::max(fl, 1) + k, 1, 64, 200000};
    if (src[k].h) {
      const Split &w = round_w[nv - cls[k]];
      BfStepArgs a;
      memset(&a, 0, sizeof(a));
      a.tt_in = src[k].h, a.do_sums = 1, a.n_pairs = (uint64_t)1 << (cls[k] - 1);
      a.low = weights + w.low * 8, a.high = weights + w.high * 8, a.low_bits = (uint32_t)w.low_bits;
      const uint64_t tile = (uint64_t)1 << w.low_bits;
      a.pairs_per_thread = std::max<uint32_t>(1, (uint32_t)(tile / BLOCK));
      a.tt_blocks = (uint32_t)((a.n_pairs + tile - 1) / tile);
      t.groups = groups_of(a.tt_blocks), a.totals = t, a.host_out = host_out, a.host_seq = seq;
      hipLaunchKernelGGL(bf_step_kernel<false>, dim3(a.tt_blocks), dim3(BLOCK), 0, c.stream, a);
      EXH_HIP(hipGetLastError());
      return OK;
    }
    BfBaseSumsArgs a;
    memset(&a, 0, sizeof(a));
    const int lb = open_bits(k);
    const Split &w = class_w[k];
    a.cols = src[k].columns, a.len = (uint64_t)1 << cls[k], a.n_cells = a.len >> lb;
    a.low = weights + w.low * 8, a.high = weights + w.high * 8, a.low_bits = (uint32_t)w.low_bits;
    a.tiles = 1u << (w.rest - w.low_bits);
    for (int j = 0; j < src[k].ncols; j++)
      for (int q = 0; q < 8; q++) a.coef[j][q] = to_mont(to_mont(src[k].coef[(size_t)j * 8 + q] % P));
    const uint32_t grid = a.tiles * (uint32_t)src[k].ncols;
    t.groups = groups_of(grid), a.totals = t, a.host_out = host_out, a.host_seq = seq;
    c.prof_begin("basefold_base_sums", k, 4 * (uint64_t)src[k].ncols * a.len);
    hipLaunchKernelGGL(lb == 1 ? bf_base_sums_kernel<1> : lb == 2 ? bf_base_sums_kernel<2> : bf_base_sums_kernel<3>,
                       dim3(grid), dim3(BLOCK), 0, c.stream, a);
    c.prof_end();
    EXH_HIP(hipGetLastError());
    return OK;
  };
  auto await_class = [&](int k, int words, uint32_t *out) -> int {
    if (!await_words(c, reinterpret_cast<const volatile unsigned long long *>(c.host_pinned + class_slot(k)), words + 1,
                     seq, out) ||
        out[words]) {
      set_error("device-error: a basefold class's sums did not arrive");
      return E_DEVICE;
    }
    return OK;
  };
  // sum_b eq(r, b) T[b]
  auto eq_fold = [&](std::vector<hf::E> t, const uint32_t *r) {
    for (int b = 0; t.size() > 1; b++) {
      const hf::E rb = hf::from(r + 8 * (size_t)b, 8);
      for (size_t q = 0; q < t.size() / 2; q++) t[q] = hf::add(hf::mul(rb, hf::sub(t[2 * q + 1], t[2 * q])), t[2 * q]);
      t.resize(t.size() / 2);
    }
    return t[0];
  };
  std::vector<uint32_t> class_words(65);
  auto open_sums = [&](int k, std::vector<hf::E> *t) -> int {
    const int n = 1 << open_bits(k);
    if ((status = await_class(k, 8 * n, class_words.data()))) return status;
    t->clear();
    for (int b = 0; b < n; b++) t->push_back(hf::from(class_words.data() + 8 * b, 8));
    return OK;
  };

  // the launch of round i (level i): fold the table by the challenges it awaits, sum round i's h0, h1; with cw_out
  // fold the codeword to level i as well
  std::vector<hf::E> xs;  // the challenges
  const Domain *dom = nullptr;
  if (fl > 0) {
    Domain *d;
    if ((status = get_domain(nv + 1, &d))) return status;
    dom = d;
  }
  std::vector<OracleTree> oracles;
  // Odd rounds end on the device: their message waits for no oracle's cap, so the launch that sums round i can send it and
  // draw the challenge, and the launches of level i + 1, its oracle's tree among them, are queued behind it at once -- one
  // trip to the host for two rounds.  (A cap is 4 KiB for the transcript, 64 compressions one after the other: 38 us on a
  // wavefront, so the rounds behind a cap stay the host's.)  An opening with every round on the host (EXACTA_HIP_HOST_ROUNDS=1)
  // and this way, us: two columns of 2^23 and one of 2^19 969 and 922, two of 2^18 478 and 425, three classes up to 2^14
  // with the verification 629 and 583.
  const char *host_rounds = getenv("EXACTA_HIP_HOST_ROUNDS");
  const bool device_rounds = !(host_rounds && host_rounds[0] == '1');
  auto on_device = [&](int i) { return device_rounds && i % 2 == 1 && i >= std::max(BB, 1) && i < fl; };
  uint32_t *challenges = mem.alloc((uint64_t)std::max(fl, 1) * 8);
  if (!challenges) return E_NOMEM;
  hf::E prf = hf::lift(1, 8), claim = hf::from(v, 8), ysum = hf::zero(8);  // ysum: the classes still to join, :593-595
  // eq of round i's coordinate at X = 0, 1, 2
  auto eq_at = [&](int i, hf::E eqx[3]) {
    const hf::E ri = hf::from(rr + 8 * (size_t)i, 8);
    eqx[0] = hf::sub(hf::lift(1, 8), ri), eqx[1] = ri, eqx[2] = hf::sub(hf::scale(ri, 2), eqx[0]);
  };
  auto launch_step = [&](int i, bool fold, bool do_sums, uint32_t *cw_out) -> int {
    BfBaseArgs b;
    memset(&b, 0, sizeof(b));
    BfStepArgs &a = b.s;
    const uint64_t n_pairs = (len >> i) / 2;
    const bool tt_base = base && i <= BB, tt_part = !tt_base || i == BB;  // (below level BB the base columns stand)
    const bool from_base = fold && tt_base, cw_base = from_base && cw_out && i == CB;
    a.tt_in = tt, a.fold = fold ? 1 : 0, a.do_sums = do_sums && tt_part ? 1 : 0, a.n_pairs = n_pairs;
    if (fold && tt_part) a.tt_out = (tt == tt_a) ? tt_b : tt_a;
    uint64_t tile = n_pairs < (uint64_t)1 << 18 ? BLOCK : 4 * BLOCK;
    if (a.do_sums) {
      const Split &w = round_w[i];
      a.low = weights + w.low * 8, a.high = weights + w.high * 8, a.low_bits = (uint32_t)w.low_bits;
      tile = (uint64_t)1 << w.low_bits;  // |LOW| pairs: one HIGH weight per workgroup
    }
    a.pairs_per_thread = std::max<uint32_t>(1, (uint32_t)(tile / BLOCK));
    a.tt_blocks = tt_part ? (uint32_t)((n_pairs + tile - 1) / tile) : 0;
    if (fold && on_device(i - 1))
      a.r_dev = challenges + 8 * (size_t)(i - 1);
    else if (fold)
      for (int k = 0; k < 8; k++) a.r_mont[k] = to_mont(xs.back()[k]);
    if (a.do_sums && on_device(i)) {
      hf::E eqx[3];
      eq_at(i, eqx);
      BfRound &r = a.round;
      r.state = device_state(tr);
      for (int q = 0; q < 3; q++) {
        const hf::E m = hf::mul(prf, eqx[q]);
        for (int k = 0; k < 8; k++) r.c[q][k] = to_mont(m[k]);
      }
      for (int k = 0; k < 8; k++) r.ysum[k] = ysum[k];
      r.r_out = challenges + 8 * (size_t)i, r.host_seq = seq;
      r.host_log = reinterpret_cast<unsigned long long *>(c.host_pinned_dev + BF_LOG_PIN + (size_t)i * BF_LOG_SLOT);
    }
    if (a.do_sums) {
      a.totals = RoundTotals{totals64 + (uint64_t)i * BF_GROUPS * 16, arrivals + i, groups_of(a.tt_blocks), 16, 200000};
      a.host_out = reinterpret_cast<unsigned long long *>(pin_dev + (size_t)i * BF_ROUND_SLOT), a.host_seq = seq;
    }
    uint32_t cw_blocks = 0;
    if (cw_out) {
      a.cw_in = cw, a.cw_out = cw_out, a.cw_m = 2 * len >> i;  // elements of the folded codeword
      a.tw_inv2 = dom->tw_inv2 + dom->off[i - 1];
      cw_blocks = (uint32_t)((a.cw_m + BLOCK - 1) / BLOCK);
    }
    if (from_base) {
      b.cols = top.columns, b.cws = top.codewords, b.col_len = len, b.cw_len = 2 * len, b.ncols = (uint32_t)top.ncols;
      b.tw0 = dom->tw_inv2 + dom->off[0], b.tw1 = i >= 2 ? dom->tw_inv2 + dom->off[1] : nullptr;
      const hf::E one = hf::lift(1, 8);
      for (int j = 0; j < top.ncols; j++) {
        const hf::E cj = hf::from(top.coef + 8 * (size_t)j, 8);
        std::vector<hf::E> eqs{cj};
        for (int q = 0; q < i; q++) {  // entry b of 2^i: bit q of b goes with challenge q
          std::vector<hf::E> next(eqs.size() * 2);
          for (size_t e = 0; e < eqs.size(); e++) {
            next[e + eqs.size()] = hf::mul(eqs[e], xs[q]);
            next[e] = hf::sub(eqs[e], next[e + eqs.size()]);
          }
          eqs.swap(next);
        }
        for (size_t e = 0; e < eqs.size(); e++)
          for (int k = 0; k < 8; k++) b.tt_coef[j][e][k] = to_mont(eqs[e][k]);
        if (cw_base) {
          const hf::E x1 = i >= 2 ? xs[1] : one;
          const hf::E prods[4] = {cj, hf::mul(cj, xs[0]), hf::mul(cj, x1), hf::mul(hf::mul(cj, xs[0]), x1)};
          for (int e = 0; e < 4; e++)
            for (int k = 0; k < 8; k++) b.cw_coef[j][e][k] = to_mont(prods[e][k]);
        }
      }
    }
    const dim3 grid(a.tt_blocks + cw_blocks);
    if (grid.x == 0) return OK;
    c.prof_begin("basefold_step", i,
                 (tt_part ? (from_base ? 4 * (uint64_t)top.ncols * len + 64 * n_pairs : (fold ? 3 : 2) * n_pairs * 32) : 0) +
                     (cw_out ? (cw_base ? 8 * (uint64_t)top.ncols * len + 32 * a.cw_m : 3 * a.cw_m * 32) : 0));
    if (from_base) {
      if (i == 1)
        hipLaunchKernelGGL((bf_base_kernel<1, 1>), grid, dim3(BLOCK), 0, c.stream, b);
      else if (i == 2 && tt_part)
        hipLaunchKernelGGL((bf_base_kernel<2, 2>), grid, dim3(BLOCK), 0, c.stream, b);
      else if (i == 2)
        hipLaunchKernelGGL((bf_base_kernel<0, 2>), grid, dim3(BLOCK), 0, c.stream, b);
      else
        hipLaunchKernelGGL((bf_base_kernel<3, 3>), grid, dim3(BLOCK), 0, c.stream, b);
    } else if (fold) {
      hipLaunchKernelGGL(bf_step_kernel<true>, grid, dim3(BLOCK), 0, c.stream, a);
    } else {
      hipLaunchKernelGGL(bf_step_kernel<false>, grid, dim3(BLOCK), 0, c.stream, a);
    }
    c.prof_end();
    EXH_HIP(hipGetLastError());
    if (fold && tt_part) tt = a.tt_out;
    if (cw_out) cw = cw_out;
    return OK;
  };
  if (base) {
    if ((status = launch_class_sums(ncls - 1))) return status;
  } else if (fl > 0 && (status = launch_step(0, false, true, nullptr))) {
    return status;
  }
  // y_c = H_c at the point's last c coordinates, for the classes still to join
  std::vector<hf::E> yc(ncls, hf::zero(8));
  auto small_table = [&](int k) { return src[k].h && nv - cls[k] >= fl; };  // no round has its weights: 2^5 elements at most
  for (int k = 0; k + 1 < ncls; k++)
    if (!small_table(k) && (status = launch_class_sums(k))) return status;
  for (int k = 0; k + 1 < ncls; k++) {
    const uint32_t *point = rr + 8 * (size_t)(nv - cls[k]);
    if (small_table(k)) {
      const uint64_t n = (uint64_t)1 << cls[k];
      std::vector<uint32_t> h(n * 8);
      std::vector<const uint32_t *> quads;
      for (uint64_t q = 0; q < 2 * n; q++) quads.push_back(src[k].h + 4 * q);
      if ((status = gather_quads(quads, h.data()))) return status;
      yc[k] = hf::mle_eval(h.data(), cls[k], point, 8);
    } else if (src[k].h) {
      if ((status = await_class(k, 16, class_words.data()))) return status;
      yc[k] = eq_fold({hf::from(class_words.data(), 8), hf::from(class_words.data() + 8, 8)}, point);
    } else {
      std::vector<hf::E> t;
      if ((status = open_sums(k, &t))) return status;
      yc[k] = eq_fold(t, point);
    }
    ysum = hf::add(ysum, yc[k]);
  }

  std::vector<hf::E> open_t;  // the sums over the open variables, folded by the challenges so far
  if (base && (status = open_sums(ncls - 1, &open_t))) return status;
  size_t cap_slots = 0;
  // the round's claim, and what its message and challenge leave for the next
  auto end_round = [&](int i, const uint32_t *ev, const uint32_t *x) {
    xs.push_back(hf::from(x, 8));
    if (out_chal) memcpy(out_chal + 8 * i, x, 32);
    claim = hf::lagrange({hf::from(ev, 8), hf::from(ev + 8, 8), hf::from(ev + 16, 8)}, xs.back());
    prf = hf::mul(prf, hf::eq1(hf::from(rr + 8 * i, 8), xs.back()));
  };
  const uint64_t dims38[2] = {3, 8};
  auto refuse_round = [&](int i) {
    set_error("verification-failure: pcs: basefold sumcheck round " + std::to_string(i) + " failed");
    return E_REJECT;
  };
  auto claim_holds = [&](const uint32_t *ev) { return hf::add(hf::from(ev, 8), hf::from(ev + 8, 8)) == claim; };
  for (int i = 0; i < fl; i++) {
    if (!on_device(i)) {
      // ---- the round's message from h0, h1
      hf::E h0, h1;
      if (i < BB) {
        std::vector<hf::E> even, odd;
        for (size_t q = 0; q < open_t.size(); q += 2) even.push_back(open_t[q]), odd.push_back(open_t[q + 1]);
        h0 = eq_fold(even, rr + 8 * (size_t)(i + 1)), h1 = eq_fold(odd, rr + 8 * (size_t)(i + 1));
      } else {
        uint32_t hh[17];
        if (!await_words(c, reinterpret_cast<const volatile unsigned long long *>(pin + (size_t)i * BF_ROUND_SLOT), 17, seq,
                         hh) ||
            hh[16]) {
          set_error("device-error: a basefold round's sums did not arrive");
          return E_DEVICE;
        }
        h0 = hf::from(hh, 8), h1 = hf::from(hh + 8, 8);
      }
      hf::E eqx[3];
      eq_at(i, eqx);
      const hf::E hx[3] = {h0, h1, hf::sub(hf::scale(h1, 2), h0)};
      uint32_t ev[24], x[8];
      for (int parity = 0; parity < 3; parity++) {  // with the classes still to join, :607-612
        const hf::E t = hf::mul(hf::mul(prf, eqx[parity]), hf::add(hx[parity], ysum));
        memcpy(ev + 8 * parity, t.data(), 32);
      }
      if ((status = tr.send(ev, 2, dims38, nullptr))) return status;
      if (!claim_holds(ev)) return refuse_round(i);
      tr.challenge(8, x);
      end_round(i, ev, x);
      if (i < BB) {
        for (size_t q = 0; q < open_t.size() / 2; q++)
          open_t[q] = hf::add(open_t[2 * q], hf::mul(xs.back(), hf::sub(open_t[2 * q + 1], open_t[2 * q])));
        open_t.resize(open_t.size() / 2);
      }
    }
    // ---- level l: fold the table and the codeword by x; an oracle tree over the folded codeword; the joins
    const int l = i + 1;
    const uint64_t cur = len >> i;  // elements of the folded codeword
    const bool oracle = l >= 2 && l < fl && l % 2 == 0;
    bool joins = false;
    for (int k = 0; k + 1 < ncls; k++) joins = joins || nv - cls[k] == l;
    uint32_t *cw_out = nullptr;
    if (l < fl && l >= CB) {  // (the last level's codeword is never looked at)
      if (oracle) {
        if (oracles.size() >= BF_MAX_ORACLES) {
          set_error("invalid-parameter: basefold oracle levels beyond the buffers");
          return E_PARAM;
        }
        cw_out = mem.alloc(cur * 8);
        if (!cw_out) return E_NOMEM;
      } else {
        cw_out = (cw == cw_b) ? cw_c : cw_b;
        if (cur * 8 > (cw_out == cw_b ? cw_words : cw_words / 2)) cw_out = cw_b;  // (only the first needs the larger one)
      }
    }
    // the next round's sums ride on the fold unless a class joins in between
    const bool more = l < fl;
    if ((status = launch_step(l, true, more && !joins, cw_out))) return status;
    size_t cap_at = 0;
    uint64_t rows = 0;
    if (oracle) {  // an oracle tree over the folded codeword, its cap to the host behind a flag
      OracleTree o;
      o.level = l;
      o.cw_len = cur;
      o.nleaves = cur / 4;
      o.lc = cap_level_of(o.nleaves);
      o.cw = cw_out;
      o.levels = mem.alloc((2 * o.nleaves) * 8);
      if (!o.levels) return E_NOMEM;
      uint64_t cap_off = 0;
      cap_at = BF_MAX_ROUNDS * BF_ROUND_SLOT + cap_slots * BF_CAP_SLOT;
      if ((status = merkle_tree_launch(o.levels, o.nleaves, 2, o.cw, 1, o.cw_len, &rows, &cap_off,
                                       reinterpret_cast<unsigned long long *>(pin_dev + cap_at), seq)))
        return status;
      cap_slots++;
      oracles.push_back(o);
    }
    if (on_device(i)) {  // its message and challenge, recorded as they were sent
      uint32_t w[BF_LOG_WORDS];
      const size_t at = BF_LOG_PIN + (size_t)i * BF_LOG_SLOT;
      if (!await_words(c, reinterpret_cast<const volatile unsigned long long *>(c.host_pinned + at), BF_LOG_WORDS, seq, w) ||
          w[BF_LOG_WORDS - 1]) {
        set_error("device-error: a basefold round did not arrive");
        return E_DEVICE;
      }
      const bool holds = claim_holds(w);
      if ((status = tr.send(w, 2, dims38, nullptr, !holds))) return status;
      if (!holds) return refuse_round(i);  // (the transcript as it stands on the host: the message sent, nothing drawn)
      DevB3S state;
      memcpy(&state, w + 32, sizeof(state));
      if ((status = adopt_device_state(tr, state))) return status;
      end_round(i, w, w + 24);
    }
    if (oracle) {
      std::vector<uint32_t> cap_words(8 * rows);
      if (!await_words(c, reinterpret_cast<const volatile unsigned long long *>(pin + cap_at), 8 * rows, seq,
                       cap_words.data())) {
        set_error("device-error: a basefold oracle's cap did not arrive");
        return E_DEVICE;
      }
      if ((status = tr.send_bytes(reinterpret_cast<const uint8_t *>(cap_words.data()), (int64_t)(32 * rows), nullptr)))
        return status;
    }
    if (joins) {
      static const uint32_t one8[8] = {1, 0, 0, 0, 0, 0, 0, 0};
      for (int k = 0; k + 1 < ncls; k++)  // the classes that join at this level, :635-639
        if (nv - cls[k] == l) {
          const uint64_t clen = (uint64_t)1 << cls[k];
          uint32_t *tt_w = const_cast<uint32_t *>(tt);  // folded: ours to write
          if (src[k].h)
            scale_add_launch<8>(tt_w, src[k].h, tt_w, clen, one8);
          else
            combine_few_launch<8>(src[k].columns, src[k].ncols, clen, src[k].coef, tt_w, tt_w);
          if (l < fl) {
            // (an oracle keeps the codeword it hashed: the sum goes to a buffer of its own then)
            uint32_t *cw_w = oracle ? mem.alloc(2 * clen * 8) : const_cast<uint32_t *>(cw);
            if (!cw_w) return E_NOMEM;
            if (src[k].h) {
              const uint32_t *cwk = src[k].cw ? src[k].cw : encode_ext(src[k].h, cls[k]);
              if (!cwk) return status;
              scale_add_launch<8>(cw, cwk, cw_w, 2 * clen, one8);
            } else {
              combine_few_launch<8>(src[k].codewords, src[k].ncols, 2 * clen, src[k].coef, cw, cw_w);
            }
            cw = cw_w;
          }
          ysum = hf::sub(ysum, yc[k]);
        }
      EXH_HIP(hipGetLastError());
      if (more && (status = launch_step(l, false, true, nullptr))) return status;
    }
  }
  // the final table in the clear, the final claim, grinding, the query positions
  uint64_t mlen = len >> fl;
  std::vector<uint32_t> m(mlen * 8);
  std::vector<const uint32_t *> quads;
  for (uint64_t q = 0; q < 2 * mlen; q++) quads.push_back(tt + 4 * q);
  if ((status = gather_quads(quads, m.data()))) return status;
  uint64_t dims[2] = {mlen, 8};
  if ((status = tr.send(m.data(), 2, dims, nullptr))) return status;
  if (out_final) memcpy(out_final, m.data(), mlen * 32);
  hf::E mval = fl < nv ? hf::mle_eval(m.data(), nv - fl, rr + 8 * fl, 8) : hf::from(m.data(), 8);
  if (hf::mul(prf, mval) != claim) {
    set_error("verification-failure: pcs: basefold final claim");
    return E_REJECT;
  }
  tr.grind(grind_bits);
  std::vector<uint64_t> qs(queries);
  tr.challenge_bits(nv - 1, queries, qs.data());
  if (out_qs) memcpy(out_qs, qs.data(), 8 * (size_t)queries);
  // ---- the oracle openings, recorded (src/pcs.lisp:651-655): every queried leaf's four symbols and every path's
  // siblings of every oracle, and whatever else the caller opens at these positions, in one gather
  quads.clear();
  auto digest_quads = [&](const uint32_t *d) { quads.push_back(d), quads.push_back(d + 4); };
  for (const OracleTree &o : oracles)
    for (int q = 0; q < queries; q++) {
      const uint64_t li = qs[q] >> o.level;
      for (int sy = 0; sy < 4; sy++) digest_quads(o.cw + (4 * li + sy) * 8);
      uint64_t level_start = 0, n = o.nleaves, idx = li;
      for (int d = 0; d < o.lc; d++) {
        digest_quads(o.levels + (level_start + (idx ^ 1)) * 8);
        level_start += n;
        n /= 2;
        idx >>= 1;
      }
    }
  const size_t oracle_quads = quads.size();
  if (more_words) more_words->segments(qs.data(), &quads);
  std::vector<uint32_t> got(quads.size() * 4);
  if ((status = gather_quads(quads, got.data()))) return status;
  const uint32_t *at = got.data();
  for (const OracleTree &o : oracles) {
    std::vector<uint32_t> leaves((size_t)queries * 32);  // (Q, 8 rows, 4 symbols): row d holds coordinate d
    std::vector<uint32_t> path;
    for (int q = 0; q < queries; q++) {
      for (int sy = 0; sy < 4; sy++, at += 8)
        for (int d = 0; d < 8; d++) leaves[((size_t)q * 8 + d) * 4 + sy] = at[d];
      path.insert(path.end(), at, at + 8 * (size_t)o.lc);
      at += 8 * (size_t)o.lc;
    }
    uint64_t d3[3] = {(uint64_t)queries, 8, 4};
    if ((status = tr.send(leaves.data(), 3, d3, nullptr, false))) return status;
    if ((status = tr.send_bytes((const uint8_t *)path.data(), (int64_t)path.size() * 4, nullptr, false))) return status;
  }
  if (more_words) more_words->words.assign(got.begin() + 4 * oracle_quads, got.end());
  return OK;
}

int basefold_prove(Transcript &tr, int nv, const uint32_t *rr, const uint32_t *v, const uint32_t *d_h, int grind_bits,
                   int queries, uint64_t *out_qs, uint32_t *out_chal, uint32_t *out_final, const uint32_t *d_cw) {
  BfSource src;
  src.h = d_h, src.cw = d_cw;
  return basefold_prove_classes(tr, nv, 1, &nv, &src, rr, v, grind_bits, queries, out_qs, out_chal, out_final);
}

// The final opening over several size classes, one key per class, each a unit of its own with its own tree:
// the class's combined column H_c = COMBINE-COLUMNS of its columns with the caller's coefficients
// (src/pcs.lisp:434-441, 709-716), BASEFOLD over the classes, then OPEN-QUERIES (:721-734): per key the queried
// leaves (Q, ncols, 4), recorded, and its tree's paths up to the cap level, recorded.
int pcs_open(Transcript &tr, int nv, int nkeys, const OpenClass *keys, const uint32_t *rr, const uint32_t *v,
             int grind_bits, int queries, uint64_t *out_qs) {
  Context &c = ctx();
  int status = c.require();
  if (status) return status;
  if (nkeys < 1 || nkeys > 32) {
    set_error("invalid-parameter: opening keys");
    return E_PARAM;
  }
  Owned mem;
  std::vector<int> cls(nkeys), depth(nkeys, 0);
  std::vector<BfSource> src(nkeys);
  for (int k = 0; k < nkeys; k++) {
    const OpenClass &key = keys[k];
    cls[k] = key.c;
    if (key.c < 1 || key.c > 30 || key.ncols < 1) {
      set_error("invalid-parameter: opening key");
      return E_PARAM;
    }
    if (key.d_levels) depth[k] = cap_level_of((uint64_t)1 << (key.c - 1));
    if (bf_base_source(key.d_columns, key.d_codewords, key.ncols, key.c)) {
      src[k].columns = key.d_columns, src[k].codewords = key.d_codewords, src[k].coef = key.coef, src[k].ncols = key.ncols;
      continue;
    }
    uint32_t *h = mem.alloc(((uint64_t)8) << key.c);
    if (!h) return E_NOMEM;
    if ((status = combine_columns_device(8, key.d_columns, key.ncols, (uint64_t)1 << key.c, key.coef, h))) return status;
    src[k].h = h;
    // ENCODE-EXT of the combined column by the encoder's linearity: the same combination of the committed
    // codewords (2^(c+1) symbols per column), no transform
    if (key.d_codewords) {
      uint32_t *cwk = mem.alloc(((uint64_t)16) << key.c);
      if (!cwk) return E_NOMEM;
      if ((status = combine_columns_device(8, key.d_codewords, key.ncols, (uint64_t)2 << key.c, key.coef, cwk)))
        return status;
      src[k].cw = cwk;
    }
  }
  std::vector<uint64_t> qs(queries > 0 ? queries : 1);
  // OPEN-QUERIES rides on BaseFold's own gather: per key the queried leaves' rows, then their paths' siblings
  BfMore more;
  more.segments = [&](const uint64_t *at, std::vector<const uint32_t *> *quads) {
    for (int k = 0; k < nkeys; k++) {
      const OpenClass &key = keys[k];
      const uint64_t nleaves = (uint64_t)1 << (key.c - 1);
      for (int q = 0; q < queries; q++)
        for (int j = 0; j < key.ncols; j++)
          quads->push_back(key.d_codewords + (uint64_t)j * ((uint64_t)2 << key.c) + 4 * (at[q] >> (nv - key.c)));
      for (int q = 0; q < queries; q++)
        for (int d = 0; d < depth[k]; d++) {
          const uint64_t start = 2 * nleaves - 2 * (nleaves >> d);
          const uint32_t *digest = key.d_levels + (start + (((at[q] >> (nv - key.c)) >> d) ^ 1)) * 8;
          quads->push_back(digest), quads->push_back(digest + 4);
        }
    }
  };
  if ((status = basefold_prove_classes(tr, nv, nkeys, cls.data(), src.data(), rr, v, grind_bits, queries, qs.data(),
                                       nullptr, nullptr, &more)))
    return status;
  if (out_qs) memcpy(out_qs, qs.data(), 8 * (size_t)queries);
  const uint32_t *at = more.words.data();
  for (int k = 0; k < nkeys; k++) {
    uint64_t d3[3] = {(uint64_t)queries, (uint64_t)keys[k].ncols, 4};
    if ((status = tr.send(at, 3, d3, nullptr, false))) return status;
    at += (size_t)queries * keys[k].ncols * 4;
    const size_t path_words = (size_t)queries * depth[k] * 8;
    if ((status = tr.send_bytes(reinterpret_cast<const uint8_t *>(at), (int64_t)path_words * 4, nullptr, false)))
      return status;
    at += path_words;
  }
  return OK;
}

// ---- the verifier's side of that opening, on the host (src/pcs.lisp:39-95, 581-657, 752-843)
namespace {
using Digest = std::array<uint8_t, 32>;
// LEAF-DIGEST (:44-52): rows of 4 values hashed 64 at a time, chained h = BLAKE3(h || d_i)
Digest host_leaf_digest(const uint32_t *rows, uint64_t nrows) {
  Digest h{}, d{};
  bool have = false;
  std::vector<uint8_t> buf;
  for (uint64_t start = 0; start < nrows; start += 64) {
    const uint64_t cnt = std::min<uint64_t>(64, nrows - start);
    buf.resize(16 * cnt);
    for (uint64_t k = 0; k < 4 * cnt; k++)
      for (int b = 0; b < 4; b++) buf[4 * k + b] = (uint8_t)(rows[4 * start + k] >> (8 * b));
    blake3_hash(buf.data(), buf.size(), d.data(), 32);
    if (have) {
      uint8_t hd[64];
      memcpy(hd, h.data(), 32), memcpy(hd + 32, d.data(), 32);
      blake3_hash(hd, 64, h.data(), 32);
    } else {
      h = d, have = true;
    }
  }
  return h;
}
Digest host_node(const uint8_t *left, const uint8_t *right) {  // :54-55
  uint8_t lr[64];
  Digest out;
  memcpy(lr, left, 32), memcpy(lr + 32, right, 32);
  blake3_hash(lr, 64, out.data(), 32);
  return out;
}
// the twiddle of fold level l at index s in a domain of 2^n points: level 0 holds the powers of the root in
// bit-reversed order, level l + 1 [s] = level l [2 s]^2 (src/rs.lisp:39-55)
// -- w^(rev(s 2^l) 2^l) for w of order 2^n, a product of the roots of order 2^(n - b) for the exponent's bits b (by powers of
// the generator, and an inversion where its inverse is wanted, a verified opening of 2^14 entries spent 300 us on these)
uint32_t host_twiddle(int n, int l, uint64_t s, bool inverse = false) {
  static const std::array<std::array<uint32_t, 32>, 2> roots = [] {  // of order 2^k, and their inverses
    std::array<std::array<uint32_t, 32>, 2> r;
    for (int k = 0; k < 32; k++) r[0][k] = fpow(3, (uint64_t)(P - 1) >> k), r[1][k] = finv(r[0][k]);
    return r;
  }();
  const uint64_t i = s << l;
  uint32_t t = 1;
  for (int b = 0; b < n - 1; b++) {  // bit b of i is bit n - 2 - b of rev
    const int at = n - 2 - b + l;
    if (((i >> b) & 1) && at < n) t = fmul(t, roots[inverse ? 1 : 0][n - at]);
  }
  return t;
}
// ENCODE (src/rs.lisp:60-85) of 2^(n-1) elements to 2^n symbols, for the final table's few entries: coordinate by coordinate
std::vector<hf::E> host_encode(const uint32_t *message, int n) {
  const uint64_t len = (uint64_t)1 << n;
  std::vector<hf::E> x(len);
  for (uint64_t i = 0; i < len; i++) {
    x[i] = hf::from(message + i % (len / 2) * 8, 8);
    for (uint32_t &v : x[i]) v %= P;
  }
  for (int b = n - 2; b >= 0; b--) {
    const uint64_t half = (uint64_t)1 << b;
    for (uint64_t k = 0; k < len / (2 * half); k++) {
      const uint32_t t = host_twiddle(n, b, k);
      for (uint64_t j = 0; j < half; j++) {
        hf::E &lo = x[2 * half * k + j], &hi = x[2 * half * k + half + j];
        const hf::E th = hf::scale(hi, t), sum = hf::add(lo, th);
        hi = hf::sub(lo, th), lo = sum;
      }
    }
  }
  return x;
}
}  // namespace

// CHECK-PATH with INJECTED-AT (src/pcs.lisp:86-95)
bool check_path_host(const uint8_t *h_in, const uint8_t *path, int depth, uint64_t i, const uint8_t *cap, int ninj,
                     const int *inj_level, const uint8_t *inj_digests) {
  Digest h;
  memcpy(h.data(), h_in, 32);
  for (int l = 1; l <= depth; l++) {
    const uint8_t *sib = path + 32 * (size_t)(l - 1);
    h = (i & 1) ? host_node(sib, h.data()) : host_node(h.data(), sib);
    i >>= 1;
    for (int k = 0; k < ninj; k++)
      if (inj_level[k] == l) h = host_node(h.data(), inj_digests + 32 * (size_t)k);
  }
  return memcmp(h.data(), cap + 32 * i, 32) == 0;
}

static int reject(const std::string &what) {
  set_error("verification-failure: pcs: " + what);
  return E_REJECT;
}

int pcs_verify_opening(Transcript &tr, int nv, int nkeys, const OpenClass *keys, const uint32_t *rr, const uint32_t *v,
                       int grind_bits, int queries) {
  if (nkeys < 1 || nkeys > 32 || keys[nkeys - 1].c != nv || queries < 1) {
    set_error("invalid-parameter: opening keys");
    return E_PARAM;
  }
  const int fl = nv - 5 > 0 ? nv - 5 : 0, Q = queries;
  int status;
  hf::E prf = hf::lift(1, 8), claim = hf::from(v, 8);
  std::vector<hf::E> chal;
  std::vector<int> olv;
  std::vector<std::vector<uint8_t>> caps;
  for (int i = 0; i < fl; i++) {  // BASEFOLD, the verifier's side
    uint32_t ev[24], x[8];
    uint64_t dims[2] = {3, 8};
    if ((status = tr.send(nullptr, 2, dims, ev))) return status;
    if (hf::add(hf::from(ev, 8), hf::from(ev + 8, 8)) != claim) return reject("basefold sumcheck round " + std::to_string(i) + " failed");
    tr.challenge(8, x);
    chal.push_back(hf::from(x, 8));
    claim = hf::lagrange({hf::from(ev, 8), hf::from(ev + 8, 8), hf::from(ev + 16, 8)}, hf::from(x, 8));
    prf = hf::mul(prf, hf::eq1(hf::from(rr + 8 * (size_t)i, 8), hf::from(x, 8)));
    const int l = i + 1;
    if (l >= 2 && l < fl && l % 2 == 0) {
      std::vector<uint8_t> cap;
      if ((status = tr.send_bytes(nullptr, -1, &cap))) return status;
      olv.push_back(l);
      caps.push_back(cap);
    }
  }
  const uint64_t mlen = (uint64_t)1 << (nv - fl);
  std::vector<uint32_t> m(mlen * 8);
  {
    uint64_t dims[2] = {mlen, 8};
    if ((status = tr.send(nullptr, 2, dims, m.data()))) return status;
    hf::E mval = fl < nv ? hf::mle_eval(m.data(), nv - fl, rr + 8 * (size_t)fl, 8) : hf::from(m.data(), 8);
    if (hf::mul(prf, mval) != claim) return reject("basefold final claim");
  }
  uint64_t nonce;
  if ((status = tr.verify_grind(grind_bits, &nonce))) return status;
  std::vector<uint64_t> qs(Q);
  tr.challenge_bits(nv - 1, Q, qs.data());
  // ---- VERIFY-QUERIES: the oracles' leaves and paths (:763-774)
  std::vector<std::vector<uint32_t>> oleaves(olv.size());
  for (size_t o = 0; o < olv.size(); o++) {
    const int l = olv[o];
    const uint64_t nleaves = (uint64_t)1 << (nv - 1 - l);
    const int depth = cap_level_of(nleaves);
    uint64_t d3[3] = {(uint64_t)Q, 8, 4};
    oleaves[o].assign((size_t)Q * 32, 0);
    std::vector<uint8_t> paths;
    if ((status = tr.send(nullptr, 3, d3, oleaves[o].data(), false))) return status;
    if ((status = tr.send_bytes(nullptr, -1, &paths, false))) return status;
    if (paths.size() != (size_t)Q * depth * 32) return reject("merkle path length");
    if (caps[o].size() != 32 * (nleaves >> depth)) return reject("oracle opening shape");
    for (int q = 0; q < Q; q++) {
      const Digest h = host_leaf_digest(oleaves[o].data() + 32 * (size_t)q, 8);
      if (!check_path_host(h.data(), paths.data() + 32 * (size_t)q * depth, depth, qs[q] >> l, caps[o].data(), 0, nullptr,
                           nullptr))
        return reject("oracle merkle path");
    }
  }
  // every key's leaves and its tree's paths; inj_c += sum_k coef_k leaf_k (:776-808)
  std::vector<std::vector<hf::E>> inj(nkeys, std::vector<hf::E>((size_t)Q * 4, hf::zero(8)));
  for (int k = 0; k < nkeys; k++) {
    const OpenClass &key = keys[k];
    if (key.c < 1 || key.c > nv || (k && key.c <= keys[k - 1].c)) {
      set_error("invalid-parameter: opening keys must ascend in class");
      return E_PARAM;
    }
    const uint64_t nleaves = (uint64_t)1 << (key.c - 1);
    const int depth = cap_level_of(nleaves), nc = key.ncols;
    uint64_t d3[3] = {(uint64_t)Q, (uint64_t)nc, 4};
    std::vector<uint32_t> leaves((size_t)Q * nc * 4);
    std::vector<uint8_t> paths;
    if ((status = tr.send(nullptr, 3, d3, leaves.data(), false))) return status;
    if ((status = tr.send_bytes(nullptr, -1, &paths, false))) return status;
    if (paths.size() != (size_t)Q * depth * 32) return reject("merkle path length");
    for (int q = 0; q < Q; q++) {
      const Digest h = host_leaf_digest(leaves.data() + (size_t)q * nc * 4, nc);
      if (!check_path_host(h.data(), paths.data() + 32 * (size_t)q * depth, depth, qs[q] >> (nv - key.c), key.cap, 0,
                           nullptr, nullptr))
        return reject("merkle path of class " + std::to_string(key.c));
      for (int sy = 0; sy < 4; sy++) {
        hf::E &held = inj[k][(size_t)q * 4 + sy];
        for (int col = 0; col < nc; col++)
          held = hf::add(held, hf::scale(hf::from(key.coef + 8 * (size_t)col, 8), leaves[((size_t)q * nc + col) * 4 + sy]));
      }
    }
  }
  // fold each query's symbols down to the final table's codeword (:810-843)
  const std::vector<hf::E> menc = host_encode(m.data(), nv - fl + 1);  // ENCODE-EXT of the final table
  const uint32_t inv2 = finv(2);
  for (int q = 0; q < Q; q++) {
    uint64_t base = 4 * qs[q];
    std::vector<hf::E> held(4, hf::zero(8));
    for (int level = 0; level <= fl; level++) {
      if (level > 0) {
        const int l = level - 1;
        std::vector<hf::E> next;
        for (size_t t2 = 0; t2 + 1 < held.size(); t2 += 2) {  // RS:FOLD (src/rs.lisp:93-101)
          const uint64_t sidx = base / 2 + t2 / 2;
          const hf::E &a = held[t2], &b = held[t2 + 1];
          const hf::E f0 = hf::scale(hf::add(a, b), inv2);
          const hf::E f1 = hf::scale(hf::sub(a, b), fmul(inv2, host_twiddle(nv + 1, l, sidx, true)));
          next.push_back(hf::add(f0, hf::mul(chal[l], hf::sub(f1, f0))));
        }
        held = next;
        base /= 2;
        for (size_t o = 0; o < olv.size(); o++)
          if (olv[o] == level) {
            const uint32_t *leaf = oleaves[o].data() + 32 * (size_t)q;
            const uint64_t ob = 4 * (qs[q] >> level);
            std::vector<hf::E> sym(4, hf::zero(8));
            for (int sy = 0; sy < 4; sy++)
              for (int d = 0; d < 8; d++) sym[sy][d] = leaf[4 * d + sy];
            if (sym[base - ob] != held[0]) return reject("fold consistency");
            held = sym;
            base = ob;
          }
      }
      for (int k = 0; k < nkeys; k++)  // INJECT
        if (nv - keys[k].c == level) {
          const uint64_t cb = 4 * (qs[q] >> level);
          for (size_t sy = 0; sy < held.size(); sy++)
            held[sy] = hf::add(held[sy], inj[k][(size_t)q * 4 + (base - cb) + sy]);
        }
    }
    for (size_t sy = 0; sy < held.size(); sy++)
      if (held[sy] != menc[base + sy]) return reject("final codeword consistency");
  }
  return OK;
}

int basefold_verify(Transcript &tr, int nv, const uint32_t *rr, const uint32_t *v, int grind_bits, int queries,
                    uint64_t *out_qs) {
  const int fl = nv - 5 > 0 ? nv - 5 : 0;
  int status;
  hf::E prf = hf::lift(1, 8), claim = hf::from(v, 8);
  for (int i = 0; i < fl; i++) {
    uint32_t ev[24], x[8];
    uint64_t dims[2] = {3, 8};
    if ((status = tr.send(nullptr, 2, dims, ev))) return status;
    if (hf::add(hf::from(ev, 8), hf::from(ev + 8, 8)) != claim) {
      set_error("verification-failure: pcs: basefold sumcheck round " + std::to_string(i) + " failed");
      return E_REJECT;
    }
    tr.challenge(8, x);
    claim = hf::lagrange({hf::from(ev, 8), hf::from(ev + 8, 8), hf::from(ev + 16, 8)}, hf::from(x, 8));
    prf = hf::mul(prf, hf::eq1(hf::from(rr + 8 * i, 8), hf::from(x, 8)));
    int l = i + 1;
    if (l >= 2 && l < fl && l % 2 == 0) {
      uint64_t nleaves = ((uint64_t)1 << (nv + 1 - l)) / 4;
      uint64_t rows = nleaves >> cap_level_of(nleaves);
      if ((status = tr.send_bytes(nullptr, (int64_t)(32 * rows), nullptr))) return status;
    }
  }
  uint64_t mlen = (uint64_t)1 << (nv - fl);
  std::vector<uint32_t> m(mlen * 8);
  uint64_t dims[2] = {mlen, 8};
  if ((status = tr.send(nullptr, 2, dims, m.data()))) return status;
  hf::E mval = fl < nv ? hf::mle_eval(m.data(), nv - fl, rr + 8 * fl, 8) : hf::from(m.data(), 8);
  if (hf::mul(prf, mval) != claim) {
    set_error("verification-failure: pcs: basefold final claim");
    return E_REJECT;
  }
  uint64_t nonce;
  if ((status = tr.verify_grind(grind_bits, &nonce))) return status;
  std::vector<uint64_t> qs(queries);
  tr.challenge_bits(nv - 1, queries, qs.data());
  if (out_qs) memcpy(out_qs, qs.data(), 8 * (size_t)queries);
  return OK;
}

}  // namespace exh
