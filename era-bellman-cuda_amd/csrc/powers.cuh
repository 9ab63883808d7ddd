// Powers of one field element for many exponents at once: base^e as the product
// of one table entry per base-4 digit of e.  With the table made on the host and
// passed in the kernel arguments, a thread's power is a chain of one product per
// digit beyond the first, where square-and-multiply in the thread takes two per
// bit.
#pragma once

#include "device.cuh"

namespace bc {

constexpr unsigned POWER_DIGITS = 16; // exponents below 2^32

struct power_digits {
  fe p[POWER_DIGITS][3]; // p[d][j - 1] = base^(j 4^d), canonical
};

// the entries of the digits [0, digits)
BC_HD void power_digits_fill(power_digits &t, const fe &base, unsigned digits) {
  fe b = reduce<FrParams>(base);
  for (unsigned d = 0; d < digits; d++) {
    t.p[d][0] = b;
    const fe b2 = mul<FrParams>(b, b);
    t.p[d][1] = b2;
    t.p[d][2] = mul<FrParams>(b2, b);
    b = mul<FrParams>(b2, b2);
  }
}

// digits of the exponents [0, count), at least one
inline unsigned power_digits_for(size_t count) {
  unsigned d = 1;
  while (d < POWER_DIGITS && count > (size_t)1 << (2 * d))
    d++;
  return d;
}

// base^(e 4^first) for e below 4^digits, canonical
__device__ __forceinline__ fe power_of(const power_digits &t, unsigned e, unsigned digits, unsigned first = 0) {
  fe acc = fe_one<FrParams>();
  for (unsigned d = 0; d < digits; d++) {
    const unsigned j = (e >> (2 * d)) & 3;
    fe s;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const uint32_t low = j == 2 ? t.p[first + d][1].v[i] : t.p[first + d][0].v[i];
      s.v[i] = j == 3 ? t.p[first + d][2].v[i] : low;
    }
    const fe next = d == 0 ? s : mul<FrParams>(acc, s);
    if (j)
      acc = next;
  }
  return acc;
}

} // namespace bc
