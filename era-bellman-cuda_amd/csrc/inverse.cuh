// Field inversion by divsteps (Bernstein and Yang, "Fast constant-time gcd
// computation and modular inversion", 2019), on nine signed 29-bit limbs.
//
// One step maps (theta, f, g) to (-theta, g, (g - f) / 2) if g is odd and
// theta >= 0, else to (theta + 1, f, (g + (g mod 2) f) / 2), starting from
// (0, m, a); f ends as +-gcd = +-1 and g as 0.  The next 29 steps depend only on
// the low 29 bits of f and g, so they run on single words and collect a 2x2
// matrix t with 2^29 (f', g') = t (f, g); the full-width f, g and the
// multipliers d, e (f = d a / C, g = e a / C mod m) are updated once per batch.
//
// Every lane does the same work, no step depends on memory, and a batch is
// about 650 instructions: an inversion issues what 40 field products do, where
// the power a^(m - 2) takes 380 products.
#pragma once

#include "field29.cuh"

namespace bc {

namespace divsteps {

// A cap, not a count: the loop ends with g = 0.  The steps above start half a
// step lower (delta = 1/2) than those for which the paper proves at most
// (49 d + 57) / 17, 735 for d = 254 bits, and need fewer: 590 suffice for 256 bits
// by the convex-hull computation of Wuille, "Bounds on divsteps iterations in
// safegcd", 2021.
constexpr int BATCH = 29, MAX_BATCHES = (735 + BATCH - 1) / BATCH;

struct s29 {
  int32_t v[9]; // limbs 0..7 in [0, 2^29), the top one signed
};

BC_HD s29 from_limbs(const c29::limbs &c) {
  s29 r;
#pragma unroll
  for (int i = 0; i < 9; i++)
    r.v[i] = (int32_t)c.v[i];
  return r;
}

BC_HD s29 from_words(const fe &a) {
  s29 r;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int start = 29 * i, w = start >> 5, s = start & 31;
    r.v[i] = (int32_t)(funnel(w < 7 ? a.v[w + 1] : 0u, a.v[w], s) & MASK29);
  }
  r.v[8] = (int32_t)(a.v[7] >> 8);
  return r;
}

BC_HD bool any_nonzero(const s29 &g) {
  int32_t o = 0;
#pragma unroll
  for (int i = 0; i < 9; i++)
    o |= g.v[i];
#if defined(__HIP_DEVICE_COMPILE__)
  return __any(o != 0); // a wave goes on until its last lane is done
#else
  return o != 0;
#endif
}

// (u x + v y) / 2^29, exact
BC_HD s29 combine(int32_t u, const s29 &x, int32_t v, const s29 &y) {
  s29 r;
  int64_t c = ((int64_t)u * x.v[0] + (int64_t)v * y.v[0]) >> 29;
#pragma unroll
  for (int i = 1; i < 9; i++) {
    c += (int64_t)u * x.v[i] + (int64_t)v * y.v[i];
    r.v[i - 1] = (int32_t)((uint32_t)c & MASK29);
    c >>= 29;
  }
  r.v[8] = (int32_t)c;
  return r;
}

// (u x + v y + k m) / 2^29 with the k in [0, 2^29) that makes it exact; since
// |u| + |v| <= 2^29 the result is within m of the larger of |x|, |y|
template <class F> BC_HD s29 combine_mod(int32_t u, const s29 &x, int32_t v, const s29 &y) {
  constexpr c29::limbs N = P29<F>::n;
  s29 r;
  int64_t c = (int64_t)u * x.v[0] + (int64_t)v * y.v[0];
  const int32_t k = (int32_t)(((uint32_t)c * P29<F>::inv) & MASK29);
  c = (c + (int64_t)k * (int32_t)N.v[0]) >> 29;
#pragma unroll
  for (int i = 1; i < 9; i++) {
    c += (int64_t)u * x.v[i] + (int64_t)v * y.v[i] + (int64_t)k * (int32_t)N.v[i];
    r.v[i - 1] = (int32_t)((uint32_t)c & MASK29);
    c >>= 29;
  }
  r.v[8] = (int32_t)c;
  return r;
}

} // namespace divsteps

// a^-1 (0 for a = 0), canonical; Montgomery in (a < 2m) and out.
template <class F> BC_HD fe inverse(const fe &a) {
  using namespace divsteps;
  constexpr c29::limbs C = c29::from_words(F::r2); // R^2: a = x R gives d = C / a = x^-1 R
  s29 f = from_limbs(P29<F>::n), g = from_words(reduce<F>(a)), d{}, e = from_limbs(C);
  int32_t theta = 0;
  for (int batch = 0; batch < MAX_BATCHES && any_nonzero(g); batch++) {
    int32_t f0 = f.v[0], g0 = g.v[0], u = 1, v = 0, q = 0, r = 1;
#pragma unroll
    for (int i = 0; i < BATCH; i++) {
      const bool odd = g0 & 1, swap = odd && theta >= 0;
      const int32_t s = swap ? -1 : 0, keep = odd ? -1 : 0; // g + (+-f or 0)
      const int32_t gf = g0 + (((f0 ^ s) - s) & keep), qu = q + (((u ^ s) - s) & keep), rv = r + (((v ^ s) - s) & keep);
      f0 = swap ? g0 : f0;
      u = (swap ? q : u) << 1;
      v = (swap ? r : v) << 1;
      g0 = gf >> 1;
      q = qu;
      r = rv;
      theta = swap ? -theta : theta + 1;
    }
    const s29 nf = combine(u, f, v, g), nd = combine_mod<F>(u, d, v, e);
    g = combine(q, f, r, g);
    e = combine_mod<F>(q, d, r, e);
    f = nf;
    d = nd;
  }
  // f = +-1 (m for a = 0, when d = 0), |d| <= 27 m; 32 m +- d is positive
  const int32_t s = f.v[8] >> 31; // the sign of f
  constexpr c29::limbs N32 = c29::times(P29<F>::n, 32);
  f29 x;
  int32_t c = 0;
#pragma unroll
  for (int i = 0; i < 9; i++) {
    c += (int32_t)N32.v[i] + ((d.v[i] ^ s) - s);
    x.v[i] = i < 8 ? (uint32_t)c & MASK29 : (uint32_t)c;
    c >>= 29;
  }
  x = reduce_value29<F>(x);
  fe out;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const int i = 32 * j / 29, sh = 32 * j % 29;
    uint64_t w = (uint64_t)x.v[i] >> sh | (uint64_t)x.v[i + 1] << (29 - sh);
    if (58 - sh < 32 && i + 2 < 9)
      w |= (uint64_t)x.v[i + 2] << (58 - sh);
    out.v[j] = (uint32_t)w;
  }
  return reduce<F>(out);
}

} // namespace bc
