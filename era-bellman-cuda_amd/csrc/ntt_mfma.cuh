// Six stages of the Fr NTT on the matrix cores.
//
// A twiddle product is a contraction when lanes share the twiddle: with x in
// signed bytes d_j, w x = sum_j d_j (w 256^j mod r), so a 32x32 byte matrix T_w
// whose row j holds the signed bytes of w 256^j mod r (centred) takes 32 elements
// to the 32 signed digit columns of a value congruent to w x and below 2^11 r in
// one v_mfma_i32_32x32x32_i8.  No digit of a reduction is needed before the
// product is there: a wave only joins the digit columns to limbs and takes off
// one multiple q r, q from the top columns.  That is about 60 VALU instructions
// for a product (75 with the digits of its input), against 265 for the
// Montgomery product; and sums of products join their columns for nothing.
//
// A radix-4 step (stages s, s + 1 of the Cooley-Tukey network) is
//   y0, y1 = (x0 + a x2) +- (b0 x1 + a b0 x3),  y2, y3 = (x0 - a x2) +- (b1 x1 - a b1 x3)
// with the stage-s twiddle a and the stage-(s+1) twiddles b0, b1: five matrix
// products, three joins and six additions.
//
// Values are signed 256-bit integers, Montgomery form.  A join leaves |r| <=
// 0.501 r and x0 is brought to |x0| <= 0.51 r, so |y| <= 1.52 r; product inputs
// (and y) must stay below 2^255 = 2.64 r.  Elements are kept with B = 128 (1 +
// 256 + ... + 256^30) added: the signed bytes of x are then those of x + B with
// the top bit of every byte but the last flipped, and B passes through the step
// with x0.
//
// Lane layout (measured): of v_mfma_i32_32x32x32_i8, lane l holds row (A) or
// column (B) l % 32, bytes 16 (l / 32) .. + 15, and of the result column l % 32,
// rows 8 (i / 4) + 4 (l / 32) + i % 4 in register i.  A is the twiddle's matrix
// (rows: digits of the result), B the elements, so a lane holds whole limbs of
// its element's digits, the even ones in the low 32 lanes.
#pragma once

#include "device.cuh"

namespace bc {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));

namespace mf {

constexpr unsigned STAGES = 6, ROWS = 1u << STAGES, LOG_COLS = 5, COLS = 1u << LOG_COLS;
constexpr unsigned TILE = ROWS * COLS, BLOCK = TILE / 4; // a quad of elements a thread
constexpr unsigned LDS_BYTES = TILE * sizeof(fe) + 8 * sizeof(fe);
// the last pass's tile has rows of 33 16-byte slots: lanes on consecutive rows
// then meet no bank conflict either
constexpr unsigned LAST_ROW = COLS + 1, LAST_HALF = ROWS * LAST_ROW;
constexpr unsigned LAST_LDS_BYTES = LAST_HALF * sizeof(fe) + 8 * sizeof(fe);

// Matrices of a group of blocks (one pass position): per radix-4 block a, b0,
// a b0, b1, -a b1; one block at stage 0, four at stage 2, sixteen at stage 4.
constexpr unsigned PER_BLOCK = 5, GROUP_BLOCKS = 21, MATRIX_BYTES = 1024;
constexpr unsigned GROUPS = 1 + ROWS; // position 0: one group; position 6: 64
constexpr size_t TABLE_BYTES = (size_t)GROUPS * GROUP_BLOCKS * PER_BLOCK * MATRIX_BYTES; // 6.8 MB a direction

// Row factors of the pass over stages ROWS_STAGE..: 64 rows of 2^12 blocks (8 MB)
constexpr unsigned ROWS_STAGE = 12, ROW_FACTORS = ROWS << ROWS_STAGE;

constexpr uint32_t BIAS[8] = {0x80808080, 0x80808080, 0x80808080, 0x80808080, 0x80808080, 0x80808080, 0x80808080, 0x00808080};

// r as signed 32-bit limbs
struct signed_limbs {
  int32_t v[8];
};
constexpr signed_limbs modulus() {
  signed_limbs r{};
  int64_t carry = 0;
  for (int i = 0; i < 8; i++) {
    int64_t t = (int64_t)FrParams::m[i] + carry;
    carry = 0;
    if (i < 7 && t >= (1ll << 31)) {
      t -= 1ll << 32;
      carry = 1;
    }
    r.v[i] = (int32_t)t;
  }
  return r;
}
// k r + s B as 8 limbs mod 2^256
struct limbs8 {
  uint32_t v[8];
};
constexpr limbs8 offset(int k, int s) {
  limbs8 r{};
  int64_t carry = 0;
  for (int i = 0; i < 8; i++) {
    const int64_t t = carry + k * (int64_t)FrParams::m[i] + s * (int64_t)BIAS[i];
    r.v[i] = (uint32_t)t;
    carry = t >> 32;
  }
  return r;
}

__device__ __forceinline__ fe add_offset(const fe &a, const limbs8 &c) {
  fe r;
  unsigned carry = 0;
#pragma unroll
  for (int i = 0; i < 8; i++)
    r.v[i] = __builtin_addc(a.v[i], c.v[i], carry, &carry);
  return r;
}

// Matrix operands of the wave's 64 elements x (biased): elements of the low and
// of the high 32 lanes.
__device__ __forceinline__ void operands(const fe &x, v4i &low, v4i &high) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const unsigned pattern_high = i < 3 ? 0x80808080u : 0x00808080u;
    const v2u s = __builtin_amdgcn_permlane32_swap(x.v[i] ^ 0x80808080u, x.v[4 + i] ^ pattern_high, false, false);
    low[i] = (int)s.x;
    high[i] = (int)s.y;
  }
}

// The limbs of each lane's element from the digit columns of the two halves,
// less the nearest multiple of r.  |column| <= 2^20, so pairs of columns stay
// below 2^29 and limb sums below 2^46; `two16` is 65536, not known to the
// compiler, which else turns the multiply-adds into shifts and adds.
__device__ __forceinline__ fe join(const v16i &low, const v16i &high, int two16) {
  constexpr signed_limbs M = modulus();
  int t[8], u[8]; // limb g = t[g] + 2^16 u[g]
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const v2u a = __builtin_amdgcn_permlane32_swap((unsigned)(low[4 * g] + (low[4 * g + 1] << 8)), (unsigned)(high[4 * g] + (high[4 * g + 1] << 8)), false, false);
    const v2u b =
        __builtin_amdgcn_permlane32_swap((unsigned)(low[4 * g + 2] + (low[4 * g + 3] << 8)), (unsigned)(high[4 * g + 2] + (high[4 * g + 3] << 8)), false, false);
    t[2 * g] = (int)a.x;
    t[2 * g + 1] = (int)a.y;
    u[2 * g] = (int)b.x;
    u[2 * g + 1] = (int)b.y;
  }
  // q = round(V / r) from V / 2^240 (below 2^26, within 1.1 of h): 2^284 / r
  const int h = u[7] + (t[7] >> 16);
  const int nq = -(int)(((int64_t)h * 0x54a47462 + (1ll << 43)) >> 44);
  fe r;
  int64_t acc = 0;
#pragma unroll
  for (int g = 0; g < 8; g++) {
    const int c = t[g] + (int)(acc >> 32);
    acc = (int64_t)u[g] * two16 + c;
    acc += (int64_t)nq * M.v[g];
    r.v[g] = (uint32_t)acc;
  }
  return r;
}

// x - round(x / r) r for |x| < 2^255 (biased: B is 0.01 r), from the table of
// (4 - e) r, e < 8
__device__ __forceinline__ fe centre(const fe &x, const fe *multiples) {
  // 2^60 / (r >> 224)
  const int q = (int)(((int64_t)(int)x.v[7] * 0x54a47464 + (1ll << 59)) >> 60);
  fe r;
  add_limbs(r, x, multiples[q + 4]);
  return r;
}

// (4 - e) r for e < 8, by the block's first eight threads
__device__ __forceinline__ void make_multiples(fe *multiples) {
  if (threadIdx.x < 8) {
    const int64_t k = 4 - (int)threadIdx.x;
    int64_t acc = 0;
    fe v;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      acc += k * (int64_t)FrParams::m[i];
      v.v[i] = (uint32_t)acc;
      acc >>= 32;
    }
    multiples[threadIdx.x] = v;
  }
}

// One radix-4 step of a thread's quad, in place.  `matrix` points at the lane's
// 16 bytes of the five matrices for the low 32 lanes' elements, `matrix_high` for
// the high ones'.
__device__ __forceinline__ void radix4(fe (&x)[4], const v4i *matrix, const v4i *matrix_high, const fe *multiples, int two16) {
  constexpr unsigned STRIDE = MATRIX_BYTES / sizeof(v4i);
  v4i l1, h1, l2, h2, l3, h3;
  operands(x[2], l2, h2);
  const v16i zero = {};
  const v16i pl = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix[0], l2, zero, 0, 0, 0);
  const v16i ph = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix_high[0], h2, zero, 0, 0, 0);
  operands(x[1], l1, h1);
  operands(x[3], l3, h3);
  x[0] = centre(x[0], multiples);
  const fe p = join(pl, ph, two16);
  fe s0, s1;
  add_limbs(s0, x[0], p);
  sub_limbs(s1, x[0], p);
  {
    v16i ql = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix[STRIDE], l1, zero, 0, 0, 0);
    v16i qh = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix_high[STRIDE], h1, zero, 0, 0, 0);
    ql = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix[2 * STRIDE], l3, ql, 0, 0, 0);
    qh = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix_high[2 * STRIDE], h3, qh, 0, 0, 0);
    const fe q = join(ql, qh, two16);
    add_limbs(x[0], s0, q);
    sub_limbs(x[1], s0, q);
  }
  {
    v16i ql = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix[3 * STRIDE], l1, zero, 0, 0, 0);
    v16i qh = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix_high[3 * STRIDE], h1, zero, 0, 0, 0);
    ql = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix[4 * STRIDE], l3, ql, 0, 0, 0);
    qh = __builtin_amdgcn_mfma_i32_32x32x32_i8(matrix_high[4 * STRIDE], h3, qh, 0, 0, 0);
    const fe q = join(ql, qh, two16);
    add_limbs(x[2], s1, q);
    sub_limbs(x[3], s1, q);
  }
}

// Matrices of every group from the twiddle table TW[2^s + b]; one thread per row
// (input byte) of a matrix.
__global__ void matrix_kernel(const fe *tw, int8_t *table) {
  using F = FrParams;
  const unsigned id = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned j = id & 31, matrix = id >> 5;
  if (matrix >= GROUPS * GROUP_BLOCKS * PER_BLOCK)
    return;
  const unsigned kind = matrix % PER_BLOCK, block = matrix / PER_BLOCK % GROUP_BLOCKS, group = matrix / (PER_BLOCK * GROUP_BLOCKS);
  const unsigned k = block == 0 ? 0 : block < 5 ? 2 : 4; // first stage of the block's step
  const unsigned b = block - (k == 0 ? 0 : k == 2 ? 1 : 5);
  const unsigned s = (group == 0 ? 0 : STAGES) + k, index = ((group == 0 ? 0 : group - 1) << k) | b;
  const fe a = load_fe(tw + (1u << s) + index), w = load_fe(tw + (2u << s) + 2 * index + (kind >= 3));
  fe v = kind == 0 ? a : kind == 1 || kind == 3 ? w : mul<F>(a, w);
  if (kind == 4)
    v = sub<F>(fe_zero(), v);
  fe byte = fe_zero();
  byte.v[0] = 256;
  v = from_mont<F>(mul<F>(v, pow_u64<F>(to_mont<F>(byte), j))); // w 256^j
  // centred: v - r above r / 2, then the signed bytes
  fe half = fe_const<F>(F::m), centred;
#pragma unroll
  for (int i = 0; i < 8; i++)
    half.v[i] = (half.v[i] >> 1) | (i < 7 ? half.v[i + 1] << 31 : 0u);
  const bool above = lt(half, v);
  sub_const(centred, v, F::m);
#pragma unroll
  for (int i = 0; i < 8; i++)
    centred.v[i] = above ? centred.v[i] : v.v[i];
  centred = add_offset(centred, offset(0, 1));
  // row j of the matrix is byte j % 16 of the lanes 32 (j / 16) + digit
  int8_t *out = table + (size_t)matrix * MATRIX_BYTES + (j >> 4) * 512 + (j & 15);
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int d = 0; d < 4; d++)
      out[(4 * i + d) * 16] = (int8_t)(((centred.v[i] >> (8 * d)) & 0xff) ^ (i == 7 && d == 3 ? 0 : 0x80));
}

} // namespace mf

} // namespace bc
