// Fr vector API (ff_*): power tables, element-wise ops, scans, batch
// inverse, powers, shifts, permutations.  Semantics follow src/ff.cu and
// src/ff_kernels.cu; every result is a canonical Montgomery Fr element.
#include <cstring>
#include <mutex>

#include "common.h"
#include "inverse.cuh"
#include "powers.cuh"
#include "scan.h"
#include "sort.h"
#include "tables.h"

namespace bc {

namespace {

ff_state g_ff[MAX_DEVICES];
std::mutex g_ff_mutex;

// table entries: fine[j] = v^j, coarse[j] = v^(j << 14); one thread per entry
__global__ void build_power_table_kernel(fe *fine, fe *coarse, fe v) {
  const unsigned j = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned n = 1u << POW_FINE_BITS;
  if (j >= 2 * n)
    return;
  const bool is_coarse = j >= n;
  const unsigned e = j & (n - 1);
  // v^(e << 14) = (v^(2^14))^e
  fe base = v;
  if (is_coarse)
    for (unsigned i = 0; i < POW_FINE_BITS; i++)
      base = mul<FrParams>(base, base);
  const fe r = pow_u64<FrParams>(base, e);
  store_fe(is_coarse ? coarse + e : fine + e, r);
}

hipError_t build_table(power_table &t, fe *storage, fe v) {
  fe *fine = storage, *coarse = storage + (1u << POW_FINE_BITS);
  build_power_table_kernel<<<grid_for(2u << POW_FINE_BITS, 256), 256>>>(fine, coarse, v);
  BC_LAUNCH_CHECK();
  t.fine = fine;
  t.coarse = coarse;
  return hipSuccess;
}

} // namespace

const ff_state *ff_current() {
  const int d = device_slot();
  return d >= 0 && g_ff[d].ready ? &g_ff[d] : nullptr;
}

hipError_t ff_set_up_impl() {
  std::lock_guard<std::mutex> lock(g_ff_mutex);
  const int d = device_slot();
  if (d < 0)
    return hipErrorInvalidDevice;
  ff_state &s = g_ff[d];
  if (s.ready)
    return hipSuccess;
  const size_t per_table = 2u << POW_FINE_BITS;
  BC_TRY(hipMalloc(&s.storage, sizeof(fe) * per_table * 3));
  const fe w = fe_const<FrParams>(FrParams::omega);
  fe seven = fe_zero();
  seven.v[0] = FrParams::generator;
  const fe g = to_mont<FrParams>(seven);
  const fe gi = inverse<FrParams>(g);
  BC_TRY(build_table(s.w, s.storage, w));
  BC_TRY(build_table(s.g, s.storage + per_table, g));
  BC_TRY(build_table(s.gi, s.storage + 2 * per_table, gi));
  BC_TRY(hipDeviceSynchronize());
  s.ready = true;
  return hipSuccess;
}

hipError_t ff_tear_down_impl() {
  std::lock_guard<std::mutex> lock(g_ff_mutex);
  const int d = device_slot();
  if (d < 0)
    return hipErrorInvalidDevice;
  ff_state &s = g_ff[d];
  if (!s.ready)
    return hipSuccess;
  BC_TRY(hipDeviceSynchronize());
  BC_TRY(hipFree(s.storage));
  s = ff_state{};
  return hipSuccess;
}

// ---------------------------------------------------------------- element-wise
enum class ew_op { ax, a_plus_x, x_plus_y, ax_plus_y, x_minus_y, ax_minus_y, x_minus_ay, x_mul_y, set };

template <ew_op OP> __device__ __forceinline__ fe ew_apply(const fe &a, const fe *x, const fe *y, size_t i) {
  using F = FrParams;
  switch (OP) {
  case ew_op::ax:
    return mul<F>(a, load_fe(x + i));
  case ew_op::a_plus_x:
    return add<F>(a, load_fe(x + i));
  case ew_op::x_plus_y:
    return add<F>(load_fe(x + i), load_fe(y + i));
  case ew_op::ax_plus_y:
    return add<F>(mul<F>(a, load_fe(x + i)), load_fe(y + i));
  case ew_op::x_minus_y:
    return sub<F>(load_fe(x + i), load_fe(y + i));
  case ew_op::ax_minus_y:
    return sub<F>(mul<F>(a, load_fe(x + i)), load_fe(y + i));
  case ew_op::x_minus_ay:
    return sub<F>(load_fe(x + i), mul<F>(a, load_fe(y + i)));
  case ew_op::x_mul_y:
    return mul<F>(load_fe(x + i), load_fe(y + i));
  case ew_op::set:
  default:
    return a;
  }
}

// `a` is either a kernel argument (host scalar) or read once per thread from device memory.
template <ew_op OP>
__global__ __launch_bounds__(256) void ew_kernel(fe a_val, const fe *a_ref, const fe *__restrict__ x, const fe *__restrict__ y, fe *__restrict__ r,
                                                 unsigned count) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const fe a = a_ref ? load_fe(a_ref) : a_val;
  store_fe(r + i, ew_apply<OP>(a, x, y, i));
}

template <ew_op OP> hipError_t ew_launch(const void *a, const void *x, const void *y, void *r, unsigned count, hipStream_t stream) {
  if (count == 0)
    return hipSuccess;
  fe a_val = fe_zero();
  const fe *a_ref = nullptr;
  if (a) {
    if (classify_pointer(a) == mem_kind::device)
      a_ref = static_cast<const fe *>(a);
    else
      memcpy(&a_val, a, sizeof(fe));
  }
  ew_kernel<OP><<<grid_for(count, 256), 256, 0, stream>>>(a_val, a_ref, static_cast<const fe *>(x), static_cast<const fe *>(y), static_cast<fe *>(r), count);
  return hipGetLastError();
}

// ---------------------------------------------------------------- powers and shifts
// target[i] = omega_{2^log_degree}^(+-j), j = offset+i (bit-reversed over log_degree bits if asked)
__global__ void powers_of_w_kernel(power_table w, fe *target, unsigned log_degree, unsigned offset, unsigned count, bool inverse, bool bit_reversed) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const unsigned raw = offset + i;
  const unsigned idx = bit_reversed ? brev_bits(raw, log_degree) : raw;
  unsigned e = (idx << (POW_LOG_RANGE - log_degree)) & ((1u << POW_LOG_RANGE) - 1);
  if (inverse)
    e = inverse_exponent(e);
  store_fe(target + i, table_pow(w, e));
}

// target[i] = g^(+-j), j = (offset+i or its bit reverse) mod 2^28 — the reference's table range (src/ff_kernels.cu:573-585)
__global__ void powers_of_g_kernel(power_table g, fe *target, unsigned log_degree, unsigned offset, unsigned count, bool bit_reversed) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const unsigned raw = offset + i;
  const unsigned idx = bit_reversed ? brev_bits(raw, log_degree) : raw;
  store_fe(target + i, table_pow(g, idx & ((1u << POW_LOG_RANGE) - 1)));
}

// result[i] = values[i] * omega_{2^log_degree}^(+-shift*(offset+i))  (src/ff_kernels.cu:601-621)
__global__ void omega_shift_kernel(power_table w, const fe *values, fe *result, unsigned log_degree, unsigned shift, unsigned offset, unsigned count,
                                   bool inverse) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  unsigned e = ((shift * (offset + i)) << (POW_LOG_RANGE - log_degree)) & ((1u << POW_LOG_RANGE) - 1);
  if (inverse)
    e = inverse_exponent(e);
  store_fe(result + i, mul<FrParams>(load_fe(values + i), table_pow(w, e)));
}

// ---------------------------------------------------------------- permutations
// fewer than 2^BR_TILE_MIN elements: one thread an element
__global__ void bit_reverse_kernel(const fe *__restrict__ in, fe *__restrict__ out, unsigned log_n) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (1u << log_n))
    return;
  store_fe(out + brev_bits(i, log_n), load_fe(in + i));
}

__global__ void bit_reverse_in_place_kernel(fe *data, unsigned log_n) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (1u << log_n))
    return;
  const unsigned j = brev_bits(i, log_n);
  if (i >= j)
    return;
  const fe a = load_fe(data + i), b = load_fe(data + j);
  store_fe(data + i, b);
  store_fe(data + j, a);
}

// An index is (high, middle, low) with 4 bits in high and low: a block takes the 256
// elements of one middle, which go to the reversed middle with high and low
// exchanged and reversed, so it reads and writes runs of 512 bytes where a thread
// an element writes 32 bytes at a time.  In place, a block exchanges the
// elements of a middle and its reverse.  2^20 elements 21 -> 14 us, 2^24 921 -> 254 us
// (in place 685 -> 324; a copy takes 207), up to 2^18 a launch's 7 us either way.
constexpr unsigned BR_BITS = 4, BR_SIDE = 1u << BR_BITS, BR_TILE_MIN = 2 * BR_BITS;
template <bool IN_PLACE> __global__ __launch_bounds__(BR_SIDE *BR_SIDE) void bit_reverse_tile_kernel(const fe *in, fe *out, unsigned log_n) {
  __shared__ fe tile[IN_PLACE ? 2 : 1][BR_SIDE][BR_SIDE + 1]; // a column's elements lie in different banks
  const unsigned bits = log_n - 2 * BR_BITS, m = blockIdx.x, rm = bits ? brev_bits(m, bits) : 0;
  if (IN_PLACE && rm < m)
    return;
  const unsigned hi = threadIdx.x / BR_SIDE, lo = threadIdx.x % BR_SIDE;
  const size_t at = (size_t)hi << (log_n - BR_BITS) | lo, here = at | (size_t)m << BR_BITS, there = at | (size_t)rm << BR_BITS;
  const unsigned col = brev_bits(hi, BR_BITS), row = brev_bits(lo, BR_BITS);
  const bool both = IN_PLACE && rm != m;
  tile[0][hi][lo] = load_fe(in + here);
  if (both)
    tile[IN_PLACE][hi][lo] = load_fe(in + there);
  __syncthreads();
  store_fe(out + there, tile[0][row][col]);
  if (both)
    store_fe(out + here, tile[IN_PLACE][row][col]);
}

__global__ void select_kernel(const fe *__restrict__ src, fe *__restrict__ dst, const unsigned *__restrict__ idx, unsigned count) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  store_fe(dst + i, load_fe(src + idx[i]));
}

// ---------------------------------------------------------------- batch inverse
// Montgomery's trick in two levels, in one kernel and without scratch memory.
// A thread multiplies up G groups of K elements (a block's threads take
// neighbouring elements, so every access is coalesced) and keeps the product at
// each group's start; the block's totals meet in LDS, where the lanes of one
// wave multiply up the INV_WAVES totals of their column and invert the product;
// then each thread walks back over its groups, reading them once more.
// Bound by the products and by the latency of the inversion, which a lone wave
// takes 35 us for (inverse.cuh): 3 products an element (4 with G > 1, which
// form the products inside a group twice) and 50 / (G K INV_WAVES) for the
// inversion.  The inverting wave moves with the block index, or every inversion
// would land on the CU's first SIMD.
// 4194299 elements 0.58 -> 0.20 ms, 65539 0.33 -> 0.048 ms (one power
// a^(r-2) per 32 consecutive elements of a thread before).
constexpr unsigned INV_BLOCK = 256, INV_WAVES = INV_BLOCK / 64;
template <unsigned G, unsigned K> __global__ __launch_bounds__(INV_BLOCK, G == 2 ? 3 : 2) void batch_inverse_kernel(const fe *in, fe *out, unsigned count) {
  using F = FrParams;
  __shared__ fe totals[INV_WAVES][64], earlier[INV_WAVES][64]; // `earlier` in LDS: the inversion needs the registers
  __shared__ fe start[G][INV_BLOCK];                               // product of the thread's groups before g
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t first = (size_t)blockIdx.x * (G * K * INV_BLOCK) + threadIdx.x;
  fe before[K]; // product of the thread's elements before element k of the group
  fe acc = fe_one<F>();
  bool wide = false;
  // zero inverts to zero and leaves the products alone
  auto multiply_up = [&](unsigned g) {
    fe v[K];
#pragma unroll
    for (unsigned k = 0; k < K; k++) {
      const size_t i = first + (g * K + k) * INV_BLOCK;
      v[k] = i < count ? load_fe(in + i) : fe_zero();
    }
#pragma unroll
    for (unsigned k = 0; k < K; k++) {
      wide |= may_be_wide(v[k]);
      before[k] = acc;
      if (!fe_is_zero(v[k]))
        acc = mul_lazy<F>(acc, v[k]);
    }
  };
  // `acc` times the first `n` elements of group g, reduced
  auto multiply_up_wide = [&](unsigned g, unsigned n) {
#pragma unroll 1
    for (unsigned k = 0; k < n; k++) {
      const size_t i = first + (g * K + k) * INV_BLOCK;
      const fe v = i < count ? lazy_of_wide(load_fe(in + i)) : fe_zero();
      if (!fe_is_zero(v))
        acc = mul_lazy<F>(acc, v);
    }
  };
#pragma unroll 1
  for (unsigned g = 0; g < G; g++) {
    if (G > 1)
      start[g][threadIdx.x] = acc;
    multiply_up(g);
  }
  wide = __any(wide);
  if (wide) {
    acc = fe_one<F>();
#pragma unroll 1
    for (unsigned g = 0; g < G; g++) {
      start[g][threadIdx.x] = acc;
      multiply_up_wide(g, K);
    }
  }
  totals[wave][lane] = acc;
  __syncthreads();
  if (wave == blockIdx.x % INV_WAVES) {
    acc = totals[0][lane];
    for (unsigned w = 1; w < INV_WAVES; w++) {
      earlier[w][lane] = acc;
      acc = mul_lazy<F>(acc, totals[w][lane]);
    }
    fe inv = inverse<F>(acc);
    for (unsigned w = INV_WAVES - 1; w > 0; w--) {
      const fe t = totals[w][lane];
      totals[w][lane] = mul_lazy<F>(earlier[w][lane], inv);
      inv = mul_lazy<F>(inv, t);
    }
    totals[0][lane] = inv;
  }
  __syncthreads();
  fe inv = totals[wave][lane];
  auto put = [&](size_t i, const fe &v, const fe &product_before) {
    if (fe_is_zero(v)) {
      store_fe(out + i, v);
    } else {
      store_fe(out + i, mul<F>(product_before, inv));
      inv = mul_lazy<F>(inv, v);
    }
  };
  if (wide) { // rare: the products before an element once more for each, without registers for them
#pragma unroll 1
    for (unsigned g = G; g-- > 0;)
#pragma unroll 1
      for (unsigned k = K; k-- > 0;) {
        acc = start[g][threadIdx.x];
        multiply_up_wide(g, k);
        const size_t i = first + (g * K + k) * INV_BLOCK;
        if (i < count)
          put(i, lazy_of_wide(load_fe(in + i)), acc);
      }
    return;
  }
#pragma unroll 1
  for (unsigned g = G; g-- > 0;) {
    if (G > 1) {
      acc = start[g][threadIdx.x];
      multiply_up(g);
    }
#pragma unroll
    for (unsigned k = K; k-- > 0;) {
      const size_t i = first + (g * K + k) * INV_BLOCK;
      if (i < count)
        put(i, load_fe(in + i), before[k]);
    }
  }
}

template <unsigned G, unsigned K> void batch_inverse_launch(const fe *in, fe *out, unsigned count, hipStream_t s) {
  batch_inverse_kernel<G, K><<<grid_for(count, G * K * INV_BLOCK), INV_BLOCK, 0, s>>>(in, out, count);
}

// The smallest share a thread for which the blocks the GPU holds at once take
// the whole vector (four, two, then two or three blocks a CU): a second round
// of blocks waits for an inversion again (700000 elements: 107 us in two rounds
// of K = 2, 75 us in one of K = 8), and a longer share than needed lengthens
// the chain (524288 elements: 60 us at K = 2).  32 elements a thread as 8 groups of
// 4, whose way back is half the instructions: 4194299 elements 202 us, 219 as 4
// groups of 8; above, 64 elements: 2^23 371 us against 387, 2^24 717 against 719.
void batch_inverse(const fe *in, fe *out, unsigned count, hipStream_t s) {
  if (count <= 1u << 19)
    batch_inverse_launch<1, 2>(in, out, count, s);
  else if (count <= 1u << 20)
    batch_inverse_launch<1, 8>(in, out, count, s);
  else if (count <= 1u << 21)
    batch_inverse_launch<2, 8>(in, out, count, s);
  else if (count <= 1u << 22)
    batch_inverse_launch<8, 4>(in, out, count, s);
  else
    batch_inverse_launch<8, 8>(in, out, count, s);
}

// ---------------------------------------------------------------- powers of one point
// The digit table of a scalar in device memory is made there, one thread (a host
// scalar's is made on the host and travels in the kernel arguments).  Table t + 1
// belongs to the point^(4^step) of table t.
__global__ void power_digits_kernel(const fe *point, power_digits *tables, unsigned count, unsigned digits, unsigned log_step) {
  fe x = load_fe(point);
  for (unsigned t = 0; t < count; t++) {
    power_digits_fill(tables[t], x, digits);
    for (unsigned i = 0; t + 1 < count && i < log_step; i++)
      x = mul<FrParams>(x, x);
  }
}

// out[i] = in[i] base^i.  Up to POWERS_DIRECT elements a thread forms its power
// from the digits; above, from one entry each of two tables, POWERS_FINE low
// powers and every POWERS_FINE-th one: two products an element.  65539 elements
// 47 -> 14 us, 4194299 283 -> 85 us (a prefix product of the base before); at
// 2^18 the tables' extra launch and memory cost as much as the powers save.
constexpr unsigned POWERS_LOG_FINE = 10, POWERS_FINE = 1u << POWERS_LOG_FINE;
constexpr unsigned POWERS_DIRECT = 1u << 17;

template <bool REF>
__global__ __launch_bounds__(256) void power_table_kernel(const power_digits arg, const power_digits *ref, fe *fine, fe *coarse, unsigned coarse_count,
                                                          unsigned coarse_digits) {
  const power_digits &t = REF ? *ref : arg;
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i < POWERS_FINE)
    store_fe(fine + i, power_of(t, i, POWERS_LOG_FINE / 2));
  else if (i - POWERS_FINE < coarse_count)
    store_fe(coarse + (i - POWERS_FINE), power_of(t, i - POWERS_FINE, coarse_digits, POWERS_LOG_FINE / 2));
}

template <bool REF>
__global__ __launch_bounds__(256) void multiply_by_powers_direct_kernel(const power_digits arg, const power_digits *ref, const fe *in, fe *out,
                                                                        unsigned count, unsigned digits) {
  const power_digits &t = REF ? *ref : arg;
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= count)
    return;
  const fe v = load_fe(in + i);
  store_fe(out + i, mul<FrParams>(v, power_of(t, i, digits)));
}

__global__ __launch_bounds__(256) void multiply_by_powers_kernel(const fe *fine, const fe *coarse, const fe *in, fe *out, unsigned count) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count)
    return;
  // an element, any 256 bits, times a canonical value is below 2m
  const fe v = mul_lazy<FrParams>(load_fe(in + i), load_fe(coarse + (i >> POWERS_LOG_FINE)));
  store_fe(out + i, mul<FrParams>(v, load_fe(fine + (i & (POWERS_FINE - 1)))));
}

// sum_i values[i] x^i: block b writes its tile's sum_j values[b tile + j] x^j to
// out[b], the values of a polynomial in x^tile for the next launch.  A thread
// takes every EVAL_BLOCK-th element of the tile (coalesced), by Horner's rule in
// x^EVAL_BLOCK: one product an element, beside 4 for the thread's own power of x.
constexpr unsigned EVAL_BLOCK = 256, EVAL_DIGITS = 4; // 4^EVAL_DIGITS = EVAL_BLOCK
template <unsigned K, bool REF>
__global__ __launch_bounds__(EVAL_BLOCK) void poly_eval_kernel(const power_digits arg, const power_digits *ref, const fe *values, size_t n, fe *out) {
  using F = FrParams;
  __shared__ fe wave_sum[EVAL_BLOCK / 64];
  const power_digits &t = REF ? *ref : arg;
  constexpr unsigned G = K < 8 ? K : 8; // loads in flight
  const size_t first = (size_t)blockIdx.x * (EVAL_BLOCK * K) + threadIdx.x;
  fe acc;
  // every value reduced: 4194299 elements 58 -> 62 us
  bool wide = false, again = false;
  do {
    bool seen = false;
    acc = fe_zero();
    for (unsigned g = K / G; g-- > 0;) {
      fe v[G];
#pragma unroll
      for (unsigned k = 0; k < G; k++) {
        const size_t i = first + (size_t)(g * G + k) * EVAL_BLOCK;
        v[k] = i < n ? load_fe(values + i) : fe_zero();
      }
      if (wide)
#pragma unroll
        for (unsigned k = 0; k < G; k++)
          v[k] = lazy_of_wide(v[k]);
#pragma unroll
      for (unsigned k = G; k-- > 0;) { // x^EVAL_BLOCK canonical: the product is below 2m, acc below 4m
        seen |= may_be_wide(v[k]);
        acc = K == 1 ? v[0] : add_raw(mul_lazy<F>(acc, t.p[EVAL_DIGITS][0]), v[k]);
      }
    }
    again = K > 1 && !wide && __any(seen);
    wide = again;
  } while (again);
  acc = mul_lazy<F>(acc, power_of(t, threadIdx.x, EVAL_DIGITS));
#pragma unroll
  for (unsigned off = 32; off > 0; off >>= 1) {
    fe o;
#pragma unroll
    for (int i = 0; i < 8; i++)
      o.v[i] = __shfl_xor(acc.v[i], off, 64);
    acc = add2<F>(acc, o);
  }
  if ((threadIdx.x & 63) == 0)
    wave_sum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (unsigned w = 1; w < EVAL_BLOCK / 64; w++)
      acc = add2<F>(acc, wave_sum[w]);
    store_fe(out + blockIdx.x, reduce<F>(acc));
  }
}

hipError_t poly_eval_launch(unsigned K, const power_digits &arg, const power_digits *ref, const fe *values, size_t n, fe *out, hipStream_t s) {
  const unsigned blocks = n ? grid_for(n, EVAL_BLOCK * K) : 1;
  auto launch = [&](auto kernel) { kernel<<<blocks, EVAL_BLOCK, 0, s>>>(arg, ref, values, n, out); };
  switch (K) {
  case 1:
    ref ? launch(poly_eval_kernel<1, true>) : launch(poly_eval_kernel<1, false>);
    break;
  case 2:
    ref ? launch(poly_eval_kernel<2, true>) : launch(poly_eval_kernel<2, false>);
    break;
  case 8:
    ref ? launch(poly_eval_kernel<8, true>) : launch(poly_eval_kernel<8, false>);
    break;
  default:
    ref ? launch(poly_eval_kernel<32, true>) : launch(poly_eval_kernel<32, false>);
    break;
  }
  return hipGetLastError();
}

// A scalar argument of a call over n elements: the value of a host scalar, or
// where a device one lies.  One element has the power 0 alone, whatever the
// scalar, which may then be missing.
const fe *scalar_argument(const void *p, size_t n, fe *value) {
  *value = fe_zero();
  if (n <= 1)
    return nullptr;
  if (classify_pointer(p) == mem_kind::device)
    return static_cast<const fe *>(p);
  memcpy(value, p, sizeof(fe));
  return nullptr;
}

hipError_t multiply_by_powers(const fe *in, const void *base, fe *out, unsigned n, hipMemPool_t pool, hipStream_t s) {
  const unsigned digits = power_digits_for(n);
  power_digits arg;
  fe b;
  const fe *base_ref = scalar_argument(base, n, &b);
  call_resources res(pool, s);
  power_digits *ref = nullptr;
  if (base_ref) {
    BC_TRY(res.get(&ref, 1));
    power_digits_kernel<<<1, 1, 0, s>>>(base_ref, ref, 1, digits, 0);
    BC_LAUNCH_CHECK();
  } else {
    power_digits_fill(arg, b, digits);
  }
  if (n <= POWERS_DIRECT) {
    if (ref)
      multiply_by_powers_direct_kernel<true><<<grid_for(n, 256), 256, 0, s>>>(arg, ref, in, out, n, digits);
    else
      multiply_by_powers_direct_kernel<false><<<grid_for(n, 256), 256, 0, s>>>(arg, ref, in, out, n, digits);
    return hipGetLastError();
  }
  const unsigned coarse_count = (n - 1) / POWERS_FINE + 1, coarse_digits = digits - POWERS_LOG_FINE / 2;
  fe *table = nullptr;
  BC_TRY(res.get(&table, (size_t)POWERS_FINE + coarse_count));
  const unsigned blocks = grid_for((size_t)POWERS_FINE + coarse_count, 256);
  if (ref)
    power_table_kernel<true><<<blocks, 256, 0, s>>>(arg, ref, table, table + POWERS_FINE, coarse_count, coarse_digits);
  else
    power_table_kernel<false><<<blocks, 256, 0, s>>>(arg, ref, table, table + POWERS_FINE, coarse_count, coarse_digits);
  BC_LAUNCH_CHECK();
  multiply_by_powers_kernel<<<grid_for(n, 256), 256, 0, s>>>(table, table + POWERS_FINE, in, out, n);
  return hipGetLastError();
}

// Launches of poly_eval_kernel until one value is left: 32 elements a thread
// where that fills the GPU, 8 below, and 2 where a thread's chain of products
// would set the time (65539 elements: 10 us against 13 at 8); up to EVAL_BLOCK
// * 8 elements one block does it.  65539 elements 93 -> 32 us (20 us of kernels,
// the temporary's release most of the rest), 4194299 341 -> 64 us: before, the
// powers were a prefix product, followed by an element-wise product and a sum.
hipError_t poly_evaluate(const fe *values, const void *point, void *result, size_t n, hipMemPool_t pool, hipStream_t s) {
  const unsigned K = n > (size_t)1 << 21 ? 32 : n > (size_t)1 << 17 ? 8 : 2;
  const size_t tile = (size_t)EVAL_BLOCK * K, last_max = EVAL_BLOCK * 8;
  unsigned levels = 1;
  size_t partials = 0;
  for (size_t m = n; m > last_max; levels++) {
    m = (m + tile - 1) / tile;
    partials += m;
  }
  fe x;
  const fe *point_ref = scalar_argument(point, n, &x);
  call_resources res(pool, s);
  power_digits *tables = nullptr;
  if (point_ref) {
    unsigned log_tile = 0;
    while ((size_t)1 << log_tile < tile)
      log_tile++;
    BC_TRY(res.get(&tables, levels));
    power_digits_kernel<<<1, 1, 0, s>>>(point_ref, tables, levels, EVAL_DIGITS + 1, log_tile);
    BC_LAUNCH_CHECK();
  }
  const bool in_place = on_device_of(s, result); // else it is copied: to the host, or to a GPU whose memory may not be mapped here
  fe *sums = nullptr; // the partial sums of every level, then the result to copy
  if (partials || !in_place)
    BC_TRY(res.get(&sums, partials + 1));
  fe *last = in_place ? static_cast<fe *>(result) : sums + partials;
  for (unsigned level = 0; level < levels; level++) {
    power_digits arg;
    if (!tables)
      power_digits_fill(arg, x, EVAL_DIGITS + 1);
    const power_digits *ref = tables ? tables + level : nullptr;
    if (level + 1 == levels) {
      BC_TRY(poly_eval_launch(n > 2 * EVAL_BLOCK ? 8 : n > EVAL_BLOCK ? 2 : 1, arg, ref, values, n, last, s));
      break;
    }
    BC_TRY(poly_eval_launch(K, arg, ref, values, n, sums, s));
    values = sums;
    n = (n + tile - 1) / tile;
    sums += n;
    for (size_t i = 1; !tables && i < tile; i <<= 1)
      x = mul<FrParams>(x, x);
  }
  if (!in_place)
    BC_TRY(hipMemcpyAsync(result, last, sizeof(fe), hipMemcpyDefault, s));
  return hipSuccess;
}

// ---------------------------------------------------------------- packed bits / distribute (src/pn_kernels.cu:123-160)
__global__ void set_values_from_packed_bits_kernel(fe *values, const unsigned *bits, unsigned count) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const unsigned b = (bits[i >> 5] >> (i & 31)) & 1u;
  store_fe(values + i, b ? fe_one<FrParams>() : fe_zero());
}

__global__ void distribute_values_kernel(const fe *src, fe *dst, unsigned count, unsigned stride) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  store_fe(dst + (size_t)i * stride, load_fe(src + i));
}

} // namespace bc

using namespace bc;

extern "C" {

bc_error ff_set_up(unsigned powers_of_w_coarse_log_count, unsigned powers_of_g_coarse_log_count) {
  (void)powers_of_w_coarse_log_count;
  (void)powers_of_g_coarse_log_count;
  return as_bc(ff_set_up_impl());
}

bc_error ff_tear_down() { return as_bc(ff_tear_down_impl()); }

bc_error ff_set_value(void *target, const void *value, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::set>(value, nullptr, nullptr, target, count, to_stream(stream)));
}

bc_error ff_set_value_zero(void *target, unsigned count, bc_stream stream) {
  if (count == 0)
    return bc_success;
  return as_bc(hipMemsetAsync(target, 0, sizeof(fe) * (size_t)count, to_stream(stream)));
}

bc_error ff_set_value_one(void *target, unsigned count, bc_stream stream) {
  const fe one = fe_one<FrParams>();
  return as_bc(ew_launch<ew_op::set>(&one, nullptr, nullptr, target, count, to_stream(stream)));
}

bc_error ff_ax(const void *a, const void *x, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::ax>(a, x, nullptr, result, count, to_stream(stream)));
}

bc_error ff_a_plus_x(const void *a, const void *x, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::a_plus_x>(a, x, nullptr, result, count, to_stream(stream)));
}

bc_error ff_x_plus_y(const void *x, const void *y, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::x_plus_y>(nullptr, x, y, result, count, to_stream(stream)));
}

bc_error ff_ax_plus_y(const void *a, const void *x, const void *y, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::ax_plus_y>(a, x, y, result, count, to_stream(stream)));
}

bc_error ff_x_minus_y(const void *x, const void *y, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::x_minus_y>(nullptr, x, y, result, count, to_stream(stream)));
}

bc_error ff_ax_minus_y(const void *a, const void *x, const void *y, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::ax_minus_y>(a, x, y, result, count, to_stream(stream)));
}

bc_error ff_x_minus_ay(const void *a, const void *x, const void *y, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::x_minus_ay>(a, x, y, result, count, to_stream(stream)));
}

bc_error ff_x_mul_y(const void *x, const void *y, void *result, unsigned count, bc_stream stream) {
  return as_bc(ew_launch<ew_op::x_mul_y>(nullptr, x, y, result, count, to_stream(stream)));
}

// Inclusive prefix product (src/ff.cu:104-118).
bc_error ff_grand_product(ff_grand_product_configuration cfg) {
  arena ar = arena::pool_mode(to_pool(cfg.mem_pool), to_stream(cfg.stream));
  return as_bc(prefix_product(static_cast<const fe *>(cfg.inputs), static_cast<fe *>(cfg.outputs), cfg.count, ar));
}

// outputs[i] = inputs[i] * base^i (src/ff.cu:136-163).
bc_error ff_multiply_by_powers(ff_multiply_by_powers_configuration cfg) {
  if (cfg.count == 0)
    return bc_success;
  return as_bc(multiply_by_powers(static_cast<const fe *>(cfg.inputs), cfg.base, static_cast<fe *>(cfg.outputs), cfg.count, to_pool(cfg.mem_pool),
                                  to_stream(cfg.stream)));
}

bc_error ff_inverse(ff_inverse_configuration cfg) {
  if (cfg.count == 0)
    return bc_success;
  batch_inverse(static_cast<const fe *>(cfg.inputs), static_cast<fe *>(cfg.outputs), cfg.count, to_stream(cfg.stream));
  return as_bc(hipGetLastError());
}

// sum_i values[i] * point^i (src/ff.cu:183-201); point and result may be host or device pointers.
bc_error ff_poly_evaluate(ff_poly_evaluate_configuration cfg) {
  return as_bc(poly_evaluate(static_cast<const fe *>(cfg.values), cfg.point, cfg.result, cfg.count, to_pool(cfg.mem_pool), to_stream(cfg.stream)));
}

bc_error ff_get_powers_of_w(void *target, unsigned log_degree, unsigned offset, unsigned count, bool inverse, bool bit_reversed, bc_stream stream) {
  const ff_state *st = ff_current();
  if (!st || log_degree > POW_LOG_RANGE)
    return bc_error_invalid_value;
  if (count == 0)
    return bc_success;
  powers_of_w_kernel<<<grid_for(count, 256), 256, 0, to_stream(stream)>>>(st->w, static_cast<fe *>(target), log_degree, offset, count, inverse, bit_reversed);
  return as_bc(hipGetLastError());
}

bc_error ff_get_powers_of_g(void *target, unsigned log_degree, unsigned offset, unsigned count, bool inverse, bool bit_reversed, bc_stream stream) {
  const ff_state *st = ff_current();
  if (!st || log_degree > 32)
    return bc_error_invalid_value;
  if (count == 0)
    return bc_success;
  powers_of_g_kernel<<<grid_for(count, 256), 256, 0, to_stream(stream)>>>(inverse ? st->gi : st->g, static_cast<fe *>(target), log_degree, offset, count,
                                                                          bit_reversed);
  return as_bc(hipGetLastError());
}

bc_error ff_omega_shift(const void *values, void *result, unsigned log_degree, unsigned shift, unsigned offset, unsigned count, bool inverse,
                        bc_stream stream) {
  const ff_state *st = ff_current();
  if (!st || log_degree > POW_LOG_RANGE)
    return bc_error_invalid_value;
  if (count == 0)
    return bc_success;
  omega_shift_kernel<<<grid_for(count, 256), 256, 0, to_stream(stream)>>>(st->w, static_cast<const fe *>(values), static_cast<fe *>(result), log_degree,
                                                                          shift, offset, count, inverse);
  return as_bc(hipGetLastError());
}

bc_error ff_bit_reverse(const void *values, void *result, unsigned log_count, bc_stream stream) {
  if (log_count > 31)
    return bc_error_invalid_value;
  const unsigned n = 1u << log_count;
  hipStream_t s = to_stream(stream);
  if (log_count >= BR_TILE_MIN) {
    const unsigned blocks = n >> BR_TILE_MIN;
    if (values == result)
      bit_reverse_tile_kernel<true><<<blocks, BR_SIDE * BR_SIDE, 0, s>>>(static_cast<const fe *>(values), static_cast<fe *>(result), log_count);
    else
      bit_reverse_tile_kernel<false><<<blocks, BR_SIDE * BR_SIDE, 0, s>>>(static_cast<const fe *>(values), static_cast<fe *>(result), log_count);
  } else if (values == result)
    bit_reverse_in_place_kernel<<<grid_for(n, 256), 256, 0, s>>>(static_cast<fe *>(result), log_count);
  else
    bit_reverse_kernel<<<grid_for(n, 256), 256, 0, s>>>(static_cast<const fe *>(values), static_cast<fe *>(result), log_count);
  return as_bc(hipGetLastError());
}

bc_error ff_bit_reverse_multigpu(const void **values, void **results, unsigned log_count, const bc_stream *streams, const int *device_ids,
                                 unsigned log_devices_count) {
  if (log_devices_count != 0)
    return bc_error_invalid_value;
  int prev = 0;
  BC_TRY_BC(hipGetDevice(&prev));
  BC_TRY_BC(hipSetDevice(device_ids[0]));
  bc_error e = ff_bit_reverse(values[0], results[0], log_count, streams[0]);
  (void)hipSetDevice(prev);
  return e;
}

bc_error ff_select(const void *source, void *destination, const unsigned *indexes, unsigned count, bc_stream stream) {
  if (count == 0)
    return bc_success;
  select_kernel<<<grid_for(count, 256), 256, 0, to_stream(stream)>>>(static_cast<const fe *>(source), static_cast<fe *>(destination), indexes, count);
  return as_bc(hipGetLastError());
}

bc_error ff_sort_u32(ff_sort_u32_configuration cfg) {
  arena ar = arena::pool_mode(to_pool(cfg.mem_pool), to_stream(cfg.stream));
  return as_bc(radix_sort_keys(static_cast<const uint32_t *>(cfg.values), static_cast<uint32_t *>(cfg.sorted_values), cfg.count, 32, ar));
}

bc_error pn_set_values_from_packed_bits(void *values, const void *packet_bits, unsigned count, bc_stream stream) {
  if (count == 0)
    return bc_success;
  set_values_from_packed_bits_kernel<<<grid_for(count, 256), 256, 0, to_stream(stream)>>>(static_cast<fe *>(values), static_cast<const unsigned *>(packet_bits),
                                                                                          count);
  return as_bc(hipGetLastError());
}

bc_error pn_distribute_values(const void *src, void *dst, unsigned count, unsigned stride, bc_stream stream) {
  if (count == 0)
    return bc_success;
  distribute_values_kernel<<<grid_for(count, 256), 256, 0, to_stream(stream)>>>(static_cast<const fe *>(src), static_cast<fe *>(dst), count, stride);
  return as_bc(hipGetLastError());
}

} // extern "C"
