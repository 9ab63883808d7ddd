// XYZZ point arithmetic by four neighbouring lanes (a quad) on 29-bit limbs.
//
// A lone wave runs a field product in about 0.5 us whatever its lanes hold, so
// a chain of point operations that cannot fill the GPU (the fold of an MSM's
// per-bit results, sums of a few hundred points) is bound by the number of
// products in sequence.  The products of one formula are mostly independent:
// a quad forms them in 3 (doubling) or 4 (addition) rounds instead of 9 or 14,
// one product per lane and round.  Operands move between the lanes with DPP
// quad permutations, one VALU move per limb.
//
// Lane l of a quad holds one coordinate: 0 Y, 1 X, 2 ZZZ, 3 ZZ.  All four
// lanes of a quad must be active in every function here, and flags returned
// are the same in the four lanes.
//
// Bounds, in multiples of m (a product of a m and b m is below (a b / 164 + 1) m,
// since m / 2^261 < 1 / 164): X < 18, Y < 6, ZZ < 2, ZZZ < 2; the values in
// between are given in the functions.  X, ZZ and ZZZ are normalized, Y is not
// (lower limbs below 2^31: the wide operand of a product).  Leaving X above 2 m
// and Y and the second factor of Y3 unnormalized takes 100 of the 930
// instructions of a doubling; a lone wave takes 5 cycles for one.
#pragma once

#include "curve29.cuh"

namespace bc {

enum : unsigned { QUAD_Y = 0, QUAD_X = 1, QUAD_ZZZ = 2, QUAD_ZZ = 3 };

__device__ __forceinline__ unsigned quad_lane() { return threadIdx.x & 3; }

template <int L0, int L1, int L2, int L3> __device__ __forceinline__ f29 quad_permute(const f29 &a) {
  f29 r;
#pragma unroll
  for (int i = 0; i < 9; i++)
    r.v[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a.v[i], L0 | L1 << 2 | L2 << 4 | L3 << 6, 0xf, 0xf, true);
  return r;
}

template <int L> __device__ __forceinline__ f29 quad_broadcast(const f29 &a) { return quad_permute<L, L, L, L>(a); }

__device__ __forceinline__ f29 select29(bool c, const f29 &a, const f29 &b) {
  f29 r;
#pragma unroll
  for (int i = 0; i < 9; i++)
    r.v[i] = c ? a.v[i] : b.v[i];
  return r;
}

// lane L's flag, in every lane of the quad
template <int L> __device__ __forceinline__ bool quad_flag(bool f) {
  return __builtin_amdgcn_update_dpp(0, f ? 1 : 0, L * 0x55, 0xf, 0xf, true) != 0;
}

__device__ __forceinline__ bool quad_is_infinity(const f29 &p) { return quad_flag<QUAD_ZZ>(is_zero29<Fq>(p)); }

// 2 p (dbl-2008-s-1 with a = 0).  Infinity stays infinity: ZZ = 0 exactly
// multiplies to 0.
__device__ __forceinline__ f29 quad_dbl(const f29 &p) {
  using P = P29<Fq>;
  const unsigned l = quad_lane();
  const f29 a = select29(l == QUAD_Y, norm29(add29(p, p)), p); // U = 2 Y < 12, X, ZZZ, ZZ
  const f29 r1 = sqr29<Fq>(a);                                 // V = U^2 < 1.9, X^2 < 3
  const f29 V = quad_broadcast<QUAD_Y>(r1), XX = quad_broadcast<QUAD_X>(r1);
  const f29 M = norm29(add29(XX, add29(XX, XX))); // < 9
  const f29 r2 = mul29<Fq>(select29(l == QUAD_ZZZ, M, a), select29(l == QUAD_ZZZ, M, V)); // W = U V, S = X V < 1.3, M^2 < 1.5, V ZZ
  const f29 W = quad_broadcast<QUAD_Y>(r2), MM = quad_broadcast<QUAD_ZZZ>(r2);
  // lane X
  const f29 X3 = norm29(sub29(MM, add29(r2, r2), P::c16e2)); // M^2 - 2 S < 17.5
  const f29 SX = sub29(r2, X3, P::c32);                      // S - X3 < 34, limbs below 2^31
  const f29 r3 = mul29<Fq>(select29(l == QUAD_X, M, W), select29(l == QUAD_X, SX, p)); // W Y < 1.1, M (S - X3) < 2.9, W ZZZ
  const f29 Y3 = sub29(quad_broadcast<QUAD_X>(r3), r3, P::c2);                         // < 4.9
  return select29(l == QUAD_Y, Y3, select29(l == QUAD_X, X3, select29(l == QUAD_ZZZ, r3, r2)));
}

// p + q (add-2008-s)
__device__ __forceinline__ f29 quad_add(const f29 &p, const f29 &q) {
  using P = P29<Fq>;
  const unsigned l = quad_lane();
  const bool p_inf = quad_is_infinity(p), q_inf = quad_is_infinity(q);
  const f29 r1 = mul29<Fq>(p, quad_permute<2, 3, 0, 1>(q)); // S1 = Y1 ZZZ2, U1 = X1 ZZ2, S2 = Y2 ZZZ1, U2 = X2 ZZ1
  const f29 d = norm29(sub29(quad_permute<2, 3, 0, 1>(r1), r1, P::c2)); // R = S2 - S1 (lane 0), Pd = U2 - U1 (lane 1)
  const bool zero = is_zero29<Fq>(d);
  const bool same_x = quad_flag<QUAD_X>(zero), same_y = quad_flag<QUAD_Y>(zero);
  const bool low = l < 2;
  const f29 r2 = mul29<Fq>(select29(low, d, p), select29(low, d, q)); // R^2, PP = Pd^2, ZZZ1 ZZZ2, ZZ1 ZZ2
  const f29 RR = quad_broadcast<0>(r2), PP = quad_broadcast<1>(r2), U1 = quad_broadcast<1>(r1);
  const f29 r3 = mul29<Fq>(select29(l == 0, U1, select29(l == 1, d, r2)), PP); // Q = U1 PP, PPP = Pd PP, -, ZZ3
  const f29 Q = quad_broadcast<0>(r3), PPP = quad_broadcast<1>(r3), R = quad_broadcast<0>(d); // < 1.1, 1.1, 3.3
  const f29 X3 = norm29(sub29(RR, add29(PPP, add29(Q, Q)), P::c16e2));                        // R^2 - PPP - 2 Q < 17.1
  const f29 QX = sub29(Q, X3, P::c32);                                                        // Q - X3 < 34, limbs below 2^31
  const f29 r4 = mul29<Fq>(select29(l == 0, r1, select29(l == 1, R, r2)), select29(l == 1, QX, PPP)); // S1 PPP, R (Q - X3), ZZZ3
  const f29 Y3 = sub29(quad_broadcast<QUAD_X>(r4), r4, P::c2); // < 4
  f29 s = select29(l == QUAD_Y, Y3, select29(l == QUAD_X, X3, select29(l == QUAD_ZZZ, r4, r3)));
  // infinities by selects, equal and opposite points behind a branch of the
  // whole wave: as lanes' branches the doubling was executed by every addition
  const bool special = same_x && !p_inf && !q_inf;
  if (__any(special)) {
    const f29 twice = quad_dbl(p);
    if (special)
      s = same_y ? twice : f29{}; // q = -p: infinity
  }
  return select29(p_inf, q, select29(q_inf, p, s));
}

// A Jacobian point of the library's format (coordinates below 2p); infinity has Z = 0.
__device__ __forceinline__ f29 quad_from_jacobian(const g1_jacobian *p) {
  const unsigned l = quad_lane();
  const f29 c = reduce_value29<Fq>(ext_to29(load_fe(l == QUAD_Y ? &p->y : l == QUAD_X ? &p->x : &p->z)));
  const f29 zz = sqr29<Fq>(c), zzz = mul29<Fq>(zz, c);
  return select29(l < 2, c, select29(l == QUAD_ZZZ, zzz, zz));
}

// XYZZ points in memory hold x, y, zz, zzz: lane l's coordinate is number l ^ 1.
// In the library's format (coordinates below 2p; infinity has ZZ = 0 mod p):
__device__ __forceinline__ f29 quad_load_xyzz(const g1_xyzz *p) { return reduce_value29<Fq>(ext_to29(load_fe(&p->x + (quad_lane() ^ 1)))); }
__device__ __forceinline__ void quad_store_xyzz(g1_xyzz *p, const f29 &c) { store_fe(&p->x + (quad_lane() ^ 1), to_ext<Fq>(norm29(c))); }

// and as a partial sum on 29-bit limbs (the accumulators' bounds: X < 2m, the
// other coordinates products, below 2^257.3, taken below 2m here)
__device__ __forceinline__ f29 quad_load_xyzz29(const xyzz29 *p) {
  const uint32_t *w = reinterpret_cast<const uint32_t *>(p) + 9 * (quad_lane() ^ 1);
  f29 r;
#pragma unroll
  for (int i = 0; i < 9; i++)
    r.v[i] = w[i];
  return reduce_value29<Fq>(r);
}
__device__ __forceinline__ void quad_store_xyzz29(xyzz29 *p, const f29 &c) {
  uint32_t *w = reinterpret_cast<uint32_t *>(p) + 9 * (quad_lane() ^ 1);
  const f29 r = reduce_value29<Fq>(norm29(c)); // X < 2 m again
#pragma unroll
  for (int i = 0; i < 9; i++)
    w[i] = r.v[i];
}

// the point of the quad `quads` quads away (a power of two): lane l ^ 4 quads
__device__ __forceinline__ f29 quad_from_neighbour(const f29 &a, unsigned quads) {
  f29 r;
#pragma unroll
  for (int i = 0; i < 9; i++)
    r.v[i] = __shfl_xor(a.v[i], 4 * quads, 64);
  return r;
}

} // namespace bc
