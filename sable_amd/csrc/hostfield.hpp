// hostfield.hpp -- exact tower arithmetic on the host with a run-time degree (4 or 8), for the
// O(rounds) protocol logic around the kernels: message assembly, claims, the verifier.
#pragma once
#include <string.h>

#include <algorithm>
#include <array>
#include <vector>

#include "field.hpp"

namespace exh {
namespace hf {

// D canonical words, tower order, D <= 8 (1 and 2 for the inverse's descent), held in place: a verifier's round is a few dozen
// of them, and as vectors on the heap they were most of its time.  (Nothing here checks D: the entry points do.)
class E {
  uint32_t w_[8];
  int n_ = 0;

 public:
  E() = default;
  explicit E(int n, uint32_t v = 0) : n_(n) { std::fill(w_, w_ + n, v); }
  E(const uint32_t *from, const uint32_t *to) : n_((int)(to - from)) { std::copy(from, to, w_); }
  E(std::vector<uint32_t>::const_iterator from, std::vector<uint32_t>::const_iterator to) : n_((int)(to - from)) {
    std::copy(from, to, w_);
  }
  size_t size() const { return (size_t)n_; }
  uint32_t *data() { return w_; }
  const uint32_t *data() const { return w_; }
  uint32_t *begin() { return w_; }
  uint32_t *end() { return w_ + n_; }
  const uint32_t *begin() const { return w_; }
  const uint32_t *end() const { return w_ + n_; }
  uint32_t &operator[](size_t i) { return w_[i]; }
  uint32_t operator[](size_t i) const { return w_[i]; }
  void assign(int n, uint32_t v) { n_ = n, std::fill(w_, w_ + n, v); }
  bool operator==(const E &o) const { return n_ == o.n_ && std::equal(begin(), end(), o.begin()); }
  bool operator!=(const E &o) const { return !(*this == o); }
};

inline E zero(int D) { return E(D, 0u); }
inline E lift(uint32_t v, int D) {
  E e(D, 0u);
  e[0] = v % P;
  return e;
}
inline E from(const uint32_t *p, int D) { return E(p, p + D); }
// the two halves of an element one after the other
inline E joined(const E &a, const E &b) {
  E o((int)(a.size() + b.size()));
  std::copy(a.begin(), a.end(), o.begin()), std::copy(b.begin(), b.end(), o.begin() + a.size());
  return o;
}
inline E add(const E &a, const E &b) {
  E o((int)a.size());
  for (size_t i = 0; i < a.size(); i++) o[i] = fadd(a[i], b[i]);
  return o;
}
inline E sub(const E &a, const E &b) {
  E o((int)a.size());
  for (size_t i = 0; i < a.size(); i++) o[i] = fsub(a[i], b[i]);
  return o;
}
inline E neg(const E &a) { return sub(zero((int)a.size()), a); }
inline E scale(const E &a, uint32_t s) {
  E o((int)a.size());
  for (size_t i = 0; i < a.size(); i++) o[i] = fmul(a[i], s % P);
  return o;
}
inline void mul_raw(int D, const uint32_t *a, const uint32_t *b, uint32_t *out) {
  if (D == 4) {
    Ext<4> x, y;
    memcpy(x.c, a, 16), memcpy(y.c, b, 16);
    Ext<4> z = ext_mul<4>(x, y);
    memcpy(out, z.c, 16);
  } else if (D == 8) {
    Ext<8> x, y;
    memcpy(x.c, a, 32), memcpy(y.c, b, 32);
    Ext<8> z = ext_mul<8>(x, y);
    memcpy(out, z.c, 32);
  } else if (D == 2) {  // F_p[x]/(x^2 - 3), for the inverse's descent
    uint32_t c0 = fadd(fmul(a[0], b[0]), times3(fmul(a[1], b[1])));
    uint32_t c1 = fadd(fmul(a[0], b[1]), fmul(a[1], b[0]));
    out[0] = c0, out[1] = c1;
  } else {
    out[0] = fmul(a[0], b[0]);
  }
}
inline E mul(const E &a, const E &b) {
  E o((int)a.size());
  mul_raw((int)a.size(), a.data(), b.data(), o.data());
  return o;
}
// a times the generator of a's level: (A0 + A1 w) w = A1 w^2 + A0 w (src/field.lisp:206-211)
inline E mul_by_generator(const E &a) {
  if (a.size() == 1) return E(1, times3(a[0]));
  size_t h = a.size() / 2;
  return joined(mul_by_generator(E(a.begin() + h, a.end())), E(a.begin(), a.begin() + h));
}
// 1/a by norms down the tower (src/field.lisp:236-243); zero -> zero (the RETURN-ZERO convention),
// callers that must signal check is_zero first
inline E inv(const E &a) {
  if (a.size() == 1) return E(1, finv(a[0]));
  size_t h = a.size() / 2;
  E a0(a.begin(), a.begin() + h), a1(a.begin() + h, a.end());
  E norm = sub(mul(a0, a0), mul_by_generator(mul(a1, a1)));
  E ninv = inv(norm);
  return joined(mul(a0, ninv), neg(mul(a1, ninv)));
}
inline bool is_zero(const E &a) {
  for (uint32_t v : a)
    if (v) return false;
  return true;
}
inline E eq1(const E &a, const E &b) {  // a b + (1 - a)(1 - b)
  E one = lift(1, (int)a.size());
  return add(mul(a, b), mul(sub(one, a), sub(one, b)));
}
// 1/k for small k (0 for 0): an inversion is some sixty products
inline uint32_t small_inverse(unsigned k) {
  static const std::array<uint32_t, 64> table = [] {
    std::array<uint32_t, 64> t;
    for (unsigned i = 0; i < 64; i++) t[i] = finv(i);
    return t;
  }();
  return k < 64 ? table[k] : finv(k);
}
// the polynomial through (xs[i], values[i]) at x, xs small distinct integers
inline E interpolate(const std::vector<int> &xs, const std::vector<E> &values, const E &x) {
  const int D = (int)x.size(), n = (int)xs.size();
  // before[i] and after: the products of x - xs[j] over j < i and j > i
  std::vector<E> diff((size_t)n), before((size_t)n);
  for (int i = 0; i < n; i++) {
    diff[i] = sub(x, lift((uint32_t)xs[i], D));
    before[i] = i == 0 ? lift(1, D) : i == 1 ? diff[0] : mul(before[i - 1], diff[i - 1]);
  }
  E acc = zero(D), after = lift(1, D);
  for (int i = n - 1; i >= 0; i--) {
    uint32_t w = 1;  // 1 / prod (xs[i] - xs[j])
    for (int j = 0; j < n; j++) {
      if (j == i) continue;
      const int d = xs[i] - xs[j];
      w = fmul(w, d > 0 ? small_inverse((unsigned)d) : fneg(small_inverse((unsigned)-d)));
    }
    E term = scale(values[i], w);
    if (i > 0) term = mul(term, before[i]);
    if (i + 1 < n) term = mul(term, after);
    acc = add(acc, term);
    if (i > 0) after = i + 1 < n ? mul(after, diff[i]) : diff[i];
  }
  return acc;
}
// LAGRANGE on the nodes 0..d (src/field.lisp:340-352)
inline E lagrange(const std::vector<E> &values, const E &x) {
  std::vector<int> xs(values.size());
  for (size_t i = 0; i < xs.size(); i++) xs[i] = (int)i;
  return interpolate(xs, values, x);
}
// EQ-TABLE (src/field.lisp:354-363), flat: 2^k entries of D words
inline std::vector<uint32_t> eq_table(const uint32_t *r, int k, int D) {
  std::vector<uint32_t> t((size_t)D << k, 0u);
  t[0] = 1;
  size_t len = 1;
  for (int b = 0; b < k; b++) {
    for (size_t i = 0; i < len; i++) {
      uint32_t up[8];
      mul_raw(D, &t[i * D], r + (size_t)b * D, up);
      for (int c = 0; c < D; c++) {
        t[(len + i) * D + c] = up[c];
        t[i * D + c] = fsub(t[i * D + c], up[c]);
      }
    }
    len *= 2;
  }
  return t;
}
// the multilinear extension of 2^k EXTs at r (LSB first), src/field.lisp:372-377
inline E mle_eval(const uint32_t *values, int k, const uint32_t *r, int D) {
  std::vector<uint32_t> t(values, values + ((size_t)D << k));
  size_t len = (size_t)1 << k;
  for (int b = 0; b < k; b++) {
    for (size_t i = 0; i < len / 2; i++) {
      uint32_t d[8], m[8];
      for (int c = 0; c < D; c++) d[c] = fsub(t[(2 * i + 1) * D + c], t[2 * i * D + c]);
      mul_raw(D, r + (size_t)b * D, d, m);
      for (int c = 0; c < D; c++) t[i * D + c] = fadd(t[2 * i * D + c], m[c]);
    }
    len /= 2;
  }
  return E(t.begin(), t.begin() + D);
}

}  // namespace hf
}  // namespace exh
