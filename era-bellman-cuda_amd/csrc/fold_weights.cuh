// The weights 2^i of an MSM's per-bit results as short combinations of powers
// of two and a cube root of one.
//
// E: y^2 = x^3 + 3 has the endomorphism (x, y) -> (beta x, y), beta^3 = 1 in Fq.
// It multiplies the points by a cube root lambda of one in Fr, so Z[w] (w^2 + w + 1
// = 0, w acting as lambda) acts on them through Z[w] / pi = Fr, where pi =
// (6 x^2 + 4 x + 1) + (2 x + 1) w has norm r; x = 4965661367192848881 is the curve's
// parameter.  Reduced mod pi, 2^i is about sqrt(r / 3) long, and as 2 has norm
// 4 it is a sum of 127 terms 2^j u with u zero or one of the six units
// +-1, +-w, +-w^2: the residues mod 2 are 0, 1, w and w^2, each unit's sign is
// free and taken towards the smaller rest.
#pragma once

#include "field29.cuh"

namespace bc {
namespace fw {

constexpr unsigned BITS = 254;      // per-bit results of an MSM
constexpr unsigned POSITIONS = 127; // powers of two that remain

struct table {
  // digit[j][i - POSITIONS] of 2^i at 2^j: 0, or 1 + k for (1, w, w^2, -1, -w, -w^2)[k]
  uint8_t digit[POSITIONS][POSITIONS + 1];
};

struct eisenstein { // a + b w, mod 2^128 each
  __int128 a, b;
};

constexpr eisenstein sub(const eisenstein &x, const eisenstein &y) {
  return {(__int128)((unsigned __int128)x.a - (unsigned __int128)y.a), (__int128)((unsigned __int128)x.b - (unsigned __int128)y.b)};
}

constexpr eisenstein times_unit(const eisenstein &z, unsigned k) {
  eisenstein r = z;
  for (unsigned t = 0; t < k % 3; t++)
    r = {-r.b, r.a - r.b}; // w (a + b w) = -b + (a - b) w
  return k < 3 ? r : eisenstein{-r.a, -r.b};
}

constexpr table make_table() {
  constexpr __int128 x = 4965661367192848881;
  constexpr eisenstein pi{6 * x * x + 4 * x + 1, 2 * x + 1};
  constexpr eisenstein unit[6] = {{1, 0}, {0, 1}, {-1, -1}, {-1, 0}, {0, -1}, {1, 1}};
  table t{};
  eisenstein z{1, 0};
  for (unsigned i = 1; i < BITS; i++) {
    // 2 z less the multiple u pi, u zero or a unit, that brings it nearest to zero:
    // the lengths compared need only be about right
    const double a = 2 * (double)z.a, b = 2 * (double)z.b;
    double best = a * a - a * b + b * b;
    eisenstein off{0, 0};
    for (unsigned k = 0; k < 6; k++) {
      const eisenstein m = times_unit(pi, k);
      const double c = a - (double)m.a, d = b - (double)m.b;
      if (c * c - c * d + d * d < best) {
        best = c * c - c * d + d * d;
        off = m;
      }
    }
    z = sub(sub(z, {-z.a, -z.b}), off); // the sum may pass 2^127, the difference does not
    if (i < POSITIONS)
      continue;
    eisenstein v = z;
    unsigned j = 0;
    for (; v.a != 0 || v.b != 0; j++) {
      unsigned digit = 0;
      if ((v.a | v.b) & 1) {
        // the unit of v's class mod 2 on v's side: the sign of 2 Re(v / unit)
        unsigned k = (v.b & 1) == 0 ? 0 : (v.a & 1) == 0 ? 1 : 5; // 1, w, 1 + w = -w^2
        const __int128 side = k == 0 ? v.a - (v.b >> 1) : k == 1 ? v.b - (v.a >> 1) : (v.a >> 1) + (v.b >> 1) + 1;
        if (side < 0)
          k = (k + 3) % 6;
        v = {v.a - unit[k].a, v.b - unit[k].b};
        digit = 1 + k;
      }
      t.digit[j][i - POSITIONS] = digit; // out of range, no constant: a 128th digit would not compile
      v = {v.a / 2, v.b / 2};
    }
  }
  return t;
}

// beta in the 2^261 radix
constexpr c29::limbs make_beta() {
  c29::limbs b = c29::from_words({0x77fffffe, 0x57634731, 0xacdb5c4f, 0xd4f263f1, 0xa0d48bac, 0x59e26bce, 0, 0});
  for (unsigned i = 0; i < 261; i++) {
    b = c29::times(b, 2);
    if (c29::geq(b, P29<Fq>::n))
      b = c29::minus(b, P29<Fq>::n);
  }
  return b;
}

constexpr c29::limbs beta = make_beta();
// beta^2 = -1 - beta
constexpr c29::limbs beta2 = c29::minus(c29::minus(c29::times(P29<Fq>::n, 2), P29<Fq>::one), beta);

} // namespace fw
} // namespace bc
