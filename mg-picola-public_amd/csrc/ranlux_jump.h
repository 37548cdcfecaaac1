// Jumping ahead in the RANLUX stream of ranlux.h.
//
// The subtract-with-borrow recurrence x_n = x_{n-5} - x_{n-12} - c in base b = 2^48 is
// a linear congruential generator in disguise (Luescher, Comput. Phys. Commun. 79
// (1994) 100; Marsaglia & Zaman 1991): with A = sum_j x_{n-12+j} b^j the state number
//   X = A - floor(A / b^7) + c,   m = b^12 - b^5 + 1 = 2^576 - 2^240 + 1,
// and every step multiplies X by a = 1/b mod m.  So k steps are one product by a^k,
// and the digits come back as A = floor(b^12 X / m), c = X - (A - floor(A / b^7)).
// The numbers are 576-bit, in nine 64-bit limbs, lowest first.
#pragma once

#include <stdint.h>
#include <string.h>

#include "ranlux.h"

namespace rlx {

constexpr int kW = 9;  // limbs of 576 bits
typedef unsigned __int128 u128;
struct Num {
  uint64_t w[kW];
};

inline Num modulus() {
  // 2^576 - 2^240 + 1: bits 240..575 set, and bit 0
  Num m;
  for (int i = 0; i < kW; i++) m.w[i] = i < 3 ? 0ull : ~0ull;
  m.w[0] = 1ull;
  m.w[3] = ~0ull << 48;  // 240 = 3 * 64 + 48
  return m;
}
inline int cmp(const uint64_t *a, const uint64_t *b) {
  for (int i = kW - 1; i >= 0; i--)
    if (a[i] != b[i]) return a[i] < b[i] ? -1 : 1;
  return 0;
}
// a -= b, the borrow returned
inline uint64_t sub(uint64_t *a, const uint64_t *b) {
  uint64_t br = 0;
  for (int i = 0; i < kW; i++) {
    const u128 t = (u128)a[i] - b[i] - br;
    a[i] = (uint64_t)t;
    br = (uint64_t)(t >> 64) & 1;
  }
  return br;
}
// r[0..n) += a[0..na) 2^shift, shift < 64 n; n limbs hold the result
inline void add_shifted(uint64_t *r, int n, const uint64_t *a, int na, int shift) {
  const int q = shift / 64, s = shift % 64;
  uint64_t carry = 0;
  for (int i = 0; i + q < n; i++) {
    uint64_t v = i < na ? a[i] << s : 0;
    if (s && i > 0 && i - 1 < na) v |= a[i - 1] >> (64 - s);
    const u128 t = (u128)r[i + q] + v + carry;
    r[i + q] = (uint64_t)t;
    carry = (uint64_t)(t >> 64);
    if (i >= na && !carry) break;
  }
}
// t[0..2 kW) mod m into x: 2^576 = 2^240 - 1 mod m, so high 2^576 + low = low + high 2^240 - high
inline Num reduce(const uint64_t *t) {
  uint64_t lo[2 * kW], hi[2 * kW];
  memcpy(lo, t, sizeof lo);
  for (;;) {
    bool any = false;
    for (int i = kW; i < 2 * kW; i++) any |= lo[i] != 0;
    if (!any) break;
    memset(hi, 0, sizeof hi);
    memcpy(hi, lo + kW, kW * sizeof(uint64_t));
    for (int i = kW; i < 2 * kW; i++) lo[i] = 0;
    // low + high 2^240 - high: never negative, as high 2^240 >= high
    add_shifted(lo, 2 * kW, hi, kW, 240);
    uint64_t br = 0;
    for (int i = 0; i < 2 * kW; i++) {
      const u128 d = (u128)lo[i] - hi[i] - br;
      lo[i] = (uint64_t)d;
      br = (uint64_t)(d >> 64) & 1;
    }
  }
  Num x;
  memcpy(x.w, lo, sizeof x.w);
  const Num m = modulus();
  while (cmp(x.w, m.w) >= 0) sub(x.w, m.w);
  return x;
}
inline Num mul(const Num &a, const Num &b) {
  uint64_t t[2 * kW] = {};
  for (int i = 0; i < kW; i++) {
    uint64_t carry = 0;
    for (int j = 0; j < kW; j++) {
      const u128 p = (u128)a.w[i] * b.w[j] + t[i + j] + carry;
      t[i + j] = (uint64_t)p;
      carry = (uint64_t)(p >> 64);
    }
    t[i + kW] = carry;
  }
  return reduce(t);
}
// a^k, a = 1/b mod m = m - (m - 1)/b = m - (2^528 - 2^192)
inline Num step_power(unsigned long long k) {
  Num a = modulus(), d;
  memset(&d, 0, sizeof d);
  // 2^528 - 2^192: bits 192..527
  for (int i = 3; i < 8; i++) d.w[i] = ~0ull;
  d.w[8] = (1ull << 16) - 1;
  sub(a.w, d.w);
  Num r;
  memset(&r, 0, sizeof r);
  r.w[0] = 1;
  for (; k; k >>= 1) {
    if (k & 1) r = mul(r, a);
    a = mul(a, a);
  }
  return r;
}
// floor(A / b^7) = A >> 336 (336 = 5 * 64 + 16)
inline void shr336(const uint64_t *a, uint64_t *o) {
  for (int i = 0; i < kW; i++) {
    const int q = i + 5;
    o[i] = q < kW ? (a[q] >> 16) | (q + 1 < kW ? a[q + 1] << 48 : 0) : 0;
  }
}
// X of a generator's state (canonical order, before its next advance)
inline Num from_state(const Ranlxd1 &g) {
  uint64_t A[kW] = {}, B[kW];
  for (int j = 0; j < 12; j++) {
    const uint64_t x = (uint64_t)(g.y[j] * 281474976710656.0);
    add_shifted(A, kW, &x, 1, 48 * j);
  }
  shr336(A, B);
  Num X;
  memcpy(X.w, A, sizeof A);
  sub(X.w, B);
  if (g.carry != 0) {
    const uint64_t one = 1;
    add_shifted(X.w, kW, &one, 1, 0);
  }
  const Num m = modulus();
  while (cmp(X.w, m.w) >= 0) sub(X.w, m.w);
  return X;
}
// The state with number X, after at least one advance of the generator.
// A = floor(2^576 X / m): 2^576 / m = 1 + (2^240 - 1)/m, so A = X + floor(X (2^240 - 1)/m),
// and X (2^240 - 1)/m = X 2^-336 (1 + about 2^-336) is within one of X >> 336: of the two
// candidates the one with c = X - (A - (A >> 336)) in {0, 1} and 2^576 X - A m in [0, m).
inline void to_state(const Num &X, Ranlxd1 &g) {
  const Num m = modulus();
  uint64_t A[kW], B[kW];
  shr336(X.w, B);
  memcpy(A, X.w, sizeof A);
  add_shifted(A, kW, B, kW, 0);
  for (int tries = 0; tries < 4; tries++) {
    // R = 2^576 X - A m, in 2 kW limbs: 2^576 (X - A) + A 2^240 - A
    uint64_t R[2 * kW] = {}, N[2 * kW] = {};
    add_shifted(R, 2 * kW, X.w, kW, 576);
    add_shifted(R, 2 * kW, A, kW, 240);
    add_shifted(N, 2 * kW, A, kW, 576);
    add_shifted(N, 2 * kW, A, kW, 0);
    uint64_t br = 0;
    for (int i = 0; i < 2 * kW; i++) {
      const u128 d = (u128)R[i] - N[i] - br;
      R[i] = (uint64_t)d;
      br = (uint64_t)(d >> 64) & 1;
    }
    const uint64_t one = 1;
    Num o;
    memset(&o, 0, sizeof o);
    o.w[0] = one;
    if (br) {  // A too large
      sub(A, o.w);
      continue;
    }
    bool big = cmp(R, m.w) >= 0;
    for (int i = kW; i < 2 * kW; i++) big |= R[i] != 0;
    if (!big) break;
    add_shifted(A, kW, &one, 1, 0);
  }
  shr336(A, B);
  uint64_t D[kW], C[kW];
  memcpy(D, A, sizeof D);
  sub(D, B);
  memcpy(C, X.w, sizeof C);
  sub(C, D);
  g.carry = C[0] & 1 ? Ranlxd1::one_bit() : 0.0;
  for (int j = 0; j < 12; j++) {
    const int q = 48 * j / 64, s = 48 * j % 64;
    uint64_t x = A[q] >> s;
    if (s > 16 && q + 1 < kW) x |= A[q + 1] << (64 - s);
    g.y[j] = (double)(x & 0xffffffffffffull) * Ranlxd1::one_bit();
  }
  g.pos = 12;
}

}  // namespace rlx
