// Extension entry points (include/bellman-amd.h).
//
// bc_amd_generator_multiples: fixed-base comb over bytes.  The table holds
// T[j][v] = v * 2^(8j) * G for 32 byte positions and v in [1, 256); a scalar
// costs at most 32 mixed additions plus one field inversion for the affine
// output.  The table is built once per device.
//
// bc_amd_msm_fold: the caller-side fold of the 254 per-bit MSM results
// (sum = 2*sum + results[i], src/bellman-cuda.h:496-505) on the device, one
// block per MSM, with the affine normalisation.
#include <mutex>

#include "common.h"
#include "curve.cuh"
#include "fold_weights.cuh"
#include "quad29.cuh"
#include "tables.h"

namespace bc {

namespace {

constexpr unsigned COMB_BYTES = 32;
constexpr unsigned COMB_ENTRIES = 256;
g1_affine *g_comb[MAX_DEVICES];
std::mutex g_comb_mutex;

__global__ __launch_bounds__(128) void comb_table_kernel(const g1_affine *base_per_byte, g1_affine *table) {
  const unsigned id = blockIdx.x * blockDim.x + threadIdx.x;
  if (id >= COMB_BYTES * COMB_ENTRIES)
    return;
  const unsigned j = id / COMB_ENTRIES, v = id % COMB_ENTRIES;
  const g1_affine b = {load_fe(&base_per_byte[j].x), load_fe(&base_per_byte[j].y)};
  g1_xyzz acc = xyzz_infinity();
  for (int bit = 7; bit >= 0; bit--) {
    acc = xyzz_dbl(acc);
    if ((v >> bit) & 1)
      acc = xyzz_add_affine(acc, b);
  }
  const g1_affine a = xyzz_to_affine(acc);
  store_fe(&table[id].x, a.x);
  store_fe(&table[id].y, a.y);
}

__global__ __launch_bounds__(128) void generator_multiples_kernel(const fe *scalars, const g1_affine *table, g1_affine *out, unsigned count) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  const fe s = load_fe(scalars + i);
  g1_xyzz acc = xyzz_infinity();
  for (unsigned j = 0; j < COMB_BYTES; j++) {
    const unsigned v = (s.v[j >> 2] >> (8 * (j & 3))) & 0xff;
    if (v)
      acc = xyzz_add_affine(acc, load_affine(table + j * COMB_ENTRIES + v));
  }
  const g1_affine a = xyzz_to_affine(acc);
  store_fe(&out[i].x, a.x);
  store_fe(&out[i].y, a.y);
}

constexpr unsigned FOLD_MAX = 64; // MSMs per fold launch
constexpr unsigned FOLD_QUADS = 128;
constexpr unsigned FOLD_BLOCK = 4 * FOLD_QUADS;

struct fold_args {
  const g1_jacobian *results[FOLD_MAX];
};

__device__ constexpr fw::table g_fold_weights = fw::make_table();

// The partial sums of one fold: S_j, and whether a result is off the curve.
constexpr unsigned FOLD_PARTS = fw::POSITIONS + 1;
struct fold_parts {
  xyzz29 sum[FOLD_PARTS]; // the last is infinity
  uint32_t off_curve;
};

constexpr unsigned PART_LEAVES = 128;
// Partial sums by 16 quads each from this many MSMs in one launch, by 64 below.
// A tree over 64 quads is 7 additions deep, but its later levels repeat their
// work in the quads that have dropped out; 16 quads take 11 additions and half
// the instructions.  The whole fold of 1, 4, 8, 24 and 64 MSMs: 314, 368, 400,
// 505 and 758 us with 64 quads, 337, 369, 382, 448 and 601 us with 16.
constexpr unsigned FOLD_MANY = 6;

// Block (j, m): S_j = R_j + sum over i >= 127 of the unit that 2^i holds at 2^j
// (fold_weights.cuh) times R_i, R the results of MSM m; sum 2^i R_i over 254
// bits is then sum 2^j S_j over 127.  A quad adds 128 / QUADS of the 128 terms
// (a few are zero), the quads' sums are joined by a tree.  27 us for one
// MSM, which saves 127 of the fold's 254 doublings of 1.8 us in sequence.
// The block after the last checks that the results lie on the curve, without
// which the units do not act.
template <unsigned QUADS> __global__ __launch_bounds__(4 * QUADS) void fold_parts_kernel(const fold_args a, fold_parts *parts) {
  using P = P29<Fq>;
  __shared__ f29 node[QUADS / 16][4];
  const g1_jacobian *r = a.results[blockIdx.y];
  fold_parts &out = parts[blockIdx.y];
  const unsigned j = blockIdx.x, q = threadIdx.x >> 2, l = quad_lane();
  if (j == fw::POSITIONS) {
    int off = 0;
    for (unsigned i = q; i < fw::BITS; i += QUADS) {
      const f29 p = quad_from_jacobian(r + i);
      const f29 s = sqr29<Fq>(p); // Y^2, X^2, Z^6, Z^4
      const f29 XXX = quad_broadcast<QUAD_X>(mul29<Fq>(s, p)), YY = quad_broadcast<QUAD_Y>(s), Z6 = quad_broadcast<QUAD_ZZZ>(s);
      const f29 d = norm29(sub29(add29(XXX, add29(Z6, add29(Z6, Z6))), YY, P::c2)); // X^3 + 3 Z^6 - Y^2 < 7 m
      off |= !quad_is_infinity(p) && !is_zero29<Fq>(d);
    }
    off = __syncthreads_or(off);
    if (q == 0) {
      quad_store_xyzz29(&out.sum[fw::POSITIONS], f29{});
      if (l == 0)
        out.off_curve = off != 0;
    }
    return;
  }
  f29 sum = f29{};
#pragma unroll 1
  for (unsigned k = q; k < PART_LEAVES; k += QUADS) { // term 0 is R_j
    const unsigned digit = k ? g_fold_weights.digit[j][k - 1] : 1u;
    f29 t = f29{};
    if (digit) {
      const f29 p = quad_from_jacobian(r + (k ? fw::POSITIONS - 1 + k : j));
      const unsigned power = (digit - 1) % 3;
      const f29 turned = mul29<Fq>(p, select29(power == 1, f29_const<Fq>(fw::beta), f29_const<Fq>(fw::beta2)));
      const f29 minus = norm29(neg29(p, P::c2));
      t = select29(l == QUAD_X && power, turned, select29(l == QUAD_Y && digit > 3, minus, p));
    }
    sum = k < QUADS ? t : quad_add(sum, t);
  }
#pragma unroll 1
  for (unsigned s = 1; s < 16; s <<= 1)
    sum = quad_add(sum, quad_from_neighbour(sum, s));
  if (QUADS > 16) {
    if (q % 16 == 0)
      node[q / 16][l] = sum;
    __syncthreads();
    if (q < 16) {
      sum = node[q % (QUADS / 16)][l];
#pragma unroll 1
      for (unsigned s = 1; s < QUADS / 16; s <<= 1)
        sum = quad_add(sum, quad_from_neighbour(sum, s));
    }
  }
  if (q == 0)
    quad_store_xyzz29(&out.sum[j], sum);
}

// One block per MSM: a binary tree over the partial sums, or over the 254
// results where there are none (no scratch memory) or a point is off the curve.
// Level j joins neighbouring nodes of 2^j positions as low + 2^(2^j) high, one
// node pair per quad of lanes, so the 127 doublings in sequence (1 + 2 + ... + 64)
// stand against only 7 additions, where Horner's rule makes 253 of each.  The
// chain is a lone wave's products one after another; a quad forms a doubling's
// in three rounds (quad29.cuh).  With the partial
// sums' launch, one MSM takes 0.31 ms and 24 take 0.45 ms; over the results
// themselves 0.51 and 0.61 ms.
__global__ __launch_bounds__(FOLD_BLOCK) void msm_fold_kernel(const fold_args a, const fold_parts *parts, g1_affine *out) {
  __shared__ f29 node[FOLD_QUADS][4];
  const g1_jacobian *r = a.results[blockIdx.x];
  const unsigned q = threadIdx.x >> 2, l = quad_lane();
  const bool whole = !parts || parts[blockIdx.x].off_curve;
  const unsigned levels = whole ? 8 : 7;
  f29 lo = f29{}, hi = f29{};
  if (!whole) {
    if (2 * q < FOLD_PARTS) {
      lo = quad_load_xyzz29(&parts[blockIdx.x].sum[2 * q]);
      hi = quad_load_xyzz29(&parts[blockIdx.x].sum[2 * q + 1]);
    }
  } else if (2 * q < fw::BITS) { // the tree has 256 leaves; the last two are infinity
    lo = quad_from_jacobian(r + 2 * q);
    hi = quad_from_jacobian(r + 2 * q + 1);
  }
  f29 sum = quad_add(lo, quad_dbl(hi));
  for (unsigned j = 1; j < levels; j++) {
    node[q][l] = sum;
    __syncthreads();
    const bool live = q < (1u << (levels - 1 - j));
    if (live) {
      lo = node[2 * q][l];
      hi = node[2 * q + 1][l];
    }
    __syncthreads();
    if (live) {
      for (unsigned k = 0; k < (1u << j); k++)
        hi = quad_dbl(hi);
      sum = quad_add(lo, hi);
    }
  }
  node[q][l] = norm29(sum);
  __syncthreads();
  if (threadIdx.x == 0) {
    const g1_affine p = xyzz_to_affine(xyzz29_to_xyzz({node[0][QUAD_X], node[0][QUAD_Y], node[0][QUAD_ZZ], node[0][QUAD_ZZZ]}));
    store_fe(&out[blockIdx.x].x, p.x);
    store_fe(&out[blockIdx.x].y, p.y);
  }
}

hipError_t comb_table(g1_affine **table) {
  std::lock_guard<std::mutex> lock(g_comb_mutex);
  const int d = device_slot();
  if (d < 0)
    return hipErrorInvalidDevice;
  if (!g_comb[d]) {
    // 2^(8j) G for j < 32, computed on the host
    g1_affine bases[COMB_BYTES];
    fe one = fe_zero(), two = fe_zero();
    one.v[0] = 1;
    two.v[0] = 2;
    g1_xyzz p = xyzz_from_affine({to_mont<Fq>(one), to_mont<Fq>(two)});
    for (unsigned j = 0; j < COMB_BYTES; j++) {
      bases[j] = xyzz_to_affine(p);
      for (int k = 0; k < 8; k++)
        p = xyzz_dbl(p);
    }
    g1_affine *dev_bases = nullptr, *t = nullptr;
    BC_TRY(hipMalloc(&dev_bases, sizeof(bases)));
    BC_TRY(hipMalloc(&t, sizeof(g1_affine) * COMB_BYTES * COMB_ENTRIES));
    BC_TRY(hipMemcpy(dev_bases, bases, sizeof(bases), hipMemcpyHostToDevice));
    comb_table_kernel<<<grid_for(COMB_BYTES * COMB_ENTRIES, 128), 128>>>(dev_bases, t);
    BC_LAUNCH_CHECK();
    BC_TRY(hipDeviceSynchronize());
    BC_TRY(hipFree(dev_bases));
    g_comb[d] = t;
  }
  *table = g_comb[d];
  return hipSuccess;
}

} // namespace

} // namespace bc

using namespace bc;

extern "C" {

bc_error bc_amd_generator_multiples(const void *scalars, void *bases, unsigned count, bc_stream stream) {
  if (count == 0)
    return bc_success;
  g1_affine *table = nullptr;
  BC_TRY_BC(comb_table(&table));
  generator_multiples_kernel<<<grid_for(count, 128), 128, 0, to_stream(stream)>>>(static_cast<const fe *>(scalars), table, static_cast<g1_affine *>(bases),
                                                                                  count);
  return as_bc(hipGetLastError());
}

bc_error bc_amd_msm_fold(const void *const *results, void *points, unsigned count, bc_stream stream) {
  if (count && (!results || !points))
    return bc_error_invalid_value;
  hipStream_t s = to_stream(stream);
  for (unsigned j = 0; j < count; j++)
    if (!results[j])
      return bc_error_invalid_value;
  // the partial sums' memory is taken and given back in stream order; without
  // any, and in a capture (whose graph would have to own it), the fold goes over
  // the results themselves
  fold_parts *parts = nullptr;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (s)
    BC_TRY_BC(hipStreamIsCapturing(s, &status));
  if (count && status == hipStreamCaptureStatusNone && pool_alloc(&parts, count < FOLD_MAX ? count : FOLD_MAX, nullptr, s) != hipSuccess) {
    (void)hipGetLastError();
    parts = nullptr;
  }
  hipError_t e = hipSuccess;
  for (unsigned base = 0; base < count && e == hipSuccess; base += FOLD_MAX) {
    const unsigned k = count - base < FOLD_MAX ? count - base : FOLD_MAX;
    fold_args a{};
    for (unsigned j = 0; j < k; j++)
      a.results[j] = static_cast<const g1_jacobian *>(results[base + j]);
    if (parts && k < FOLD_MANY)
      fold_parts_kernel<64><<<dim3(fw::POSITIONS + 1, k), 256, 0, s>>>(a, parts);
    else if (parts)
      fold_parts_kernel<16><<<dim3(fw::POSITIONS + 1, k), 64, 0, s>>>(a, parts);
    msm_fold_kernel<<<k, FOLD_BLOCK, 0, s>>>(a, parts, static_cast<g1_affine *>(points) + base);
    e = hipGetLastError();
  }
  const hipError_t freed = pool_free(parts, s);
  return as_bc(e != hipSuccess ? e : freed);
}

} // extern "C"
