// Fr NTT for gfx950, batched: a batch of transforms of any sizes and
// directions runs as one launch per pass index (per butterfly order), with
// the per-transform descriptors passed by value in the kernel arguments.  The
// plain C-ABI call is a batch of one.
//
// Semantics (src/ntt_kernels.cu:119-294, src/bellman-cuda.h:516-541):
//   bit_reversed_inputs = false: natural order in, bit-reversed order out;
//   bit_reversed_inputs = true:  bit-reversed in, natural out;
//   forward coset (log_extension_degree > 0): coefficient i is multiplied by
//   (g * omega_{n*2^e}^coset)^i before the transform, g = 7;
//   inverse: omega^-1 twiddles, then n^-1 and (with a coset) the inverse twist
//   on the natural output index; outputs canonical in [0, r).
//
// Design.  The radix-2 butterfly network of stage s pairs elements
// n/2^(s+1) apart, and block b of stage s uses w = omega_{2^(s+1)}^brev_s(b).
// One twiddle table TW[2^s + b] (n entries) therefore serves every size and
// both orders: natural->bit-reversed runs Cooley-Tukey butterflies over
// s = 0..L-1; bit-reversed->natural runs the transposed network, Gentleman-
// Sande butterflies (E,O) -> (E+O, w(E-O)) over s = L-1..0.  A pass executes a
// run of at most NTT_LOG_TILE consecutive stages [s_lo, s_hi) on LDS tiles of
// 2^NTT_LOG_TILE = 1024 elements (32 KiB, five blocks per CU): the stages'
// butterflies stay inside groups of 2^(s_hi-s_lo) elements, strided by
// 2^(L-s_hi), so a transform of 2^L takes ceil(L / 10) HBM passes (three at
// 2^24).  Tiles are mapped XCD-major so that neighbouring strided columns run
// on the same XCD and share its L2 lines.  The first twelve stages of a natural-
// order transform of 2^NTT_MFMA_MIN_LOG or more are two passes of six stages on
// the matrix cores instead (ntt_mfma.cuh): their few twiddles are shared by 32
// columns and more.
#include <algorithm>
#include <mutex>
#include <vector>

#include "batch.h"
#include "common.h"
#include "inverse.cuh"
#include "ntt.h"
#include "ntt_mfma.cuh"
#include "powers.cuh"
#include "tables.h"
#include "tuning.h"

namespace bc {

namespace {

constexpr unsigned NTT_BLOCK = (1u << NTT_LOG_TILE) / 4; // one radix-4 group per thread and step
constexpr unsigned NTT_SMALL_LOG_TILE = 9, NTT_SMALL_BLOCK = (1u << NTT_SMALL_LOG_TILE) / 2; // one butterfly per thread and stage
constexpr unsigned TWIST_FINE_BITS = 12;

struct twiddle_state {
  fe *fwd = nullptr;       // TW[2^s + b] = omega_{2^(s+1)}^brev_s(b), index 0 unused
  fe *inv = nullptr;       // inverse powers, same layout
  fe *inv_sizes = nullptr; // 2^-i, i <= NTT_MAX_LOG
  int8_t *mfma_fwd = nullptr, *mfma_inv = nullptr; // twiddle matrices (ntt_mfma.cuh)
  fe *rows_fwd = nullptr, *rows_inv = nullptr;     // [hi][t] = omega_{2^18}^(+-brev_12(hi) t), t < 64
  const fe *last_rows[2][NTT_MFMA_LAST_MAX_LOG + 1] = {}; // of the last pass, by direction and size (make_last_rows)
  unsigned log_size = 0;
  bool attributes = false;
  std::vector<fe *> retired;
};

twiddle_state g_tw[MAX_DEVICES];
std::mutex g_tw_mutex;

__global__ void twiddle_build_kernel(power_table w, fe *fwd, fe *inv, unsigned log_size) {
  const unsigned m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= (1u << log_size))
    return;
  if (m == 0) {
    store_fe(fwd, fe_one<FrParams>());
    store_fe(inv, fe_one<FrParams>());
    return;
  }
  const unsigned s = 31 - __clz(m);
  const unsigned b = m - (1u << s);
  // omega_{2^(s+1)} = omega_{2^28}^(2^(27-s))
  const unsigned e = brev_bits(b, s) << (27 - s);
  store_fe(fwd + m, table_pow(w, e));
  store_fe(inv + m, table_pow(w, inverse_exponent(e)));
}

// rows[hi][t] = omega_{2^(s_lo + log_rows)}^(+-brev(hi) t), hi < 2^s_lo, t < 2^log_rows
__global__ void row_factor_kernel(power_table w, fe *rows, unsigned s_lo, unsigned log_rows, bool inverse) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 1u << (s_lo + log_rows))
    return;
  const unsigned hi = i >> log_rows, t = i & ((1u << log_rows) - 1);
  const unsigned e = brev_bits(hi, s_lo) * t << (POW_LOG_RANGE - s_lo - log_rows);
  store_fe(rows + i, table_pow(w, inverse ? inverse_exponent(e) : e));
}

enum : uint8_t { PRE_NONE = 0, PRE_COSET = 1, PRE_ROWS = 2 };
enum : uint8_t { POST_LAZY = 0, POST_REDUCE = 1, POST_SCALE = 2, POST_TABLE = 3 };

// One transform's share of a pass launch.
struct pass_job {
  const fe *in;
  fe *out;
  const fe *aux;  // POST_SCALE: n^-1; twists: fine table, coarse table 2^12 entries later
  const fe *rows; // PRE_ROWS: [hi][row] factors
  uint32_t tile_begin; // first block of the job (a multiple of 8)
  uint8_t log_n, s_lo, s_hi;
  uint8_t log_c, log_g; // tile = 2^log_g groups x 2^(s_hi-s_lo) rows x 2^log_c columns
  uint8_t inverse, pre_table, post;
};

struct pass_table {
  uint32_t count;
  const fe *tw_fwd;
  const fe *tw_inv;
  pass_job job[NTT_MAX_JOBS];
};
static_assert(sizeof(pass_table) <= 4096, "kernel argument budget");

__device__ __forceinline__ fe twist_pow(const fe *fine, unsigned i) {
  const fe c = load_fe(fine + (1u << TWIST_FINE_BITS) + (i >> TWIST_FINE_BITS));
  const unsigned f = i & ((1u << TWIST_FINE_BITS) - 1);
  return f ? mul<FrParams>(load_fe(fine + f), c) : c;
}

template <bool GS> __global__ __launch_bounds__(NTT_BLOCK) void ntt_pass_kernel(const pass_table pt) {
  using F = FrParams;
  extern __shared__ fe tile[];
  unsigned jl = 0, jh = pt.count; // job of this block
  while (jh - jl > 1) {
    const unsigned mid = (jl + jh) >> 1;
    if (pt.job[mid].tile_begin <= blockIdx.x)
      jl = mid;
    else
      jh = mid;
  }
  const pass_job &a = pt.job[jl];
  const unsigned L = a.log_n, s_lo = a.s_lo, s_hi = a.s_hi, log_c = a.log_c, log_g = a.log_g;
  const unsigned log_t = s_hi - s_lo;
  const unsigned tiles = 1u << (L - log_t - log_c - log_g);
  unsigned tid_tile = blockIdx.x - a.tile_begin;
  if (tid_tile >= tiles)
    return; // alignment padding
  if ((tiles & 7) == 0)
    tid_tile = (tid_tile & 7) * (tiles >> 3) + (tid_tile >> 3);
  const fe *__restrict__ tw = a.inverse ? pt.tw_inv : pt.tw_fwd;
  const unsigned log_lo = L - s_hi;             // bits below the group
  const unsigned lo_tiles_log = log_lo - log_c; // tiles along the low bits
  const unsigned lo0 = (tid_tile & ((1u << lo_tiles_log) - 1)) << log_c;
  const unsigned hi0 = (tid_tile >> lo_tiles_log) << log_g;
  const unsigned elems = 1u << (log_g + log_t + log_c);
  const unsigned cmask = (1u << log_c) - 1, tmask = (1u << log_t) - 1;

  // element e of the tile <-> index of the transform
  auto index_of = [&](unsigned e) {
    const unsigned c = e & cmask, t = (e >> log_c) & tmask, g = e >> (log_c + log_t);
    return ((hi0 + g) << (L - s_lo)) | (t << log_lo) | (lo0 + c);
  };
  constexpr unsigned PER_THREAD = (1u << NTT_LOG_TILE) / NTT_BLOCK;
  if (a.pre_table && elems == (1u << NTT_LOG_TILE)) {
    // coset twist: the elements and their twists are loaded first, then the
    // products are formed
    fe v[PER_THREAD], tw[PER_THREAD];
#pragma unroll
    for (unsigned r = 0; r < PER_THREAD; r++) {
      const unsigned idx = index_of(threadIdx.x + r * NTT_BLOCK);
      v[r] = load_fe(a.in + idx);
      tw[r] = twist_pow(a.aux, GS ? brev_bits(idx, L) : idx);
    }
#pragma unroll
    for (unsigned r = 0; r < PER_THREAD; r++)
      tile[threadIdx.x + r * NTT_BLOCK] = mul_lazy<F>(v[r], tw[r]);
  } else if (a.pre_table) {
    for (unsigned e = threadIdx.x; e < elems; e += NTT_BLOCK) {
      const unsigned idx = index_of(e);
      tile[e] = mul_lazy<F>(load_fe(a.in + idx), twist_pow(a.aux, GS ? brev_bits(idx, L) : idx));
    }
  } else if (elems == (1u << NTT_LOG_TILE)) {
    // a thread's loads are all issued before the first is used
    fe v[PER_THREAD];
#pragma unroll
    for (unsigned r = 0; r < PER_THREAD; r++)
      v[r] = load_fe(a.in + index_of(threadIdx.x + r * NTT_BLOCK));
#pragma unroll
    for (unsigned r = 0; r < PER_THREAD; r++)
      tile[threadIdx.x + r * NTT_BLOCK] = v[r];
  } else {
    for (unsigned e = threadIdx.x; e < elems; e += NTT_BLOCK)
      tile[e] = load_fe(a.in + index_of(e));
  }
  __syncthreads();

  // Stages in network order (CT: s_lo..s_hi-1, GS: s_hi-1..s_lo).  An odd
  // count starts with one radix-2 step; the rest go two at a time: a thread
  // holds the 4 elements t0, t0+h/2, t0+h, t0+3h/2 (h = row distance of the
  // lower stage s) and applies stages s and s+1 in registers.
  const unsigned nst = log_t;
  unsigned done = 0;
  if (nst & 1) {
    const unsigned s = GS ? s_hi - 1 : s_lo;
    const unsigned log_h = s_hi - s - 1;
    const unsigned h = 1u << log_h;
    for (unsigned q = threadIdx.x; q < (elems >> 1); q += NTT_BLOCK) {
      const unsigned c = q & cmask;
      const unsigned r = (q >> log_c) & (tmask >> 1);
      const unsigned g = q >> (log_c + log_t - 1);
      const unsigned t0 = ((r >> log_h) << (log_h + 1)) | (r & (h - 1));
      const unsigned i0 = (((g << log_t) | t0) << log_c) | c;
      const unsigned i1 = i0 + (h << log_c);
      const unsigned b = ((hi0 + g) << (s - s_lo)) | (t0 >> (s_hi - s));
      const fe E = tile[i0], O = tile[i1];
      if (!GS) {
        // CT tile values are < 4m; each output is < 4m again
        const fe wo = s != 0 ? mul_lazy<F>(O, load_fe(tw + (1u << s) + b)) : reduce2<F>(O);
        const fe e = reduce2<F>(E);
        tile[i0] = add_raw(e, wo);
        tile[i1] = sub_raw2<F>(e, wo);
      } else {
        // GS tile values stay < 2m
        tile[i0] = add2<F>(E, O);
        tile[i1] = s != 0 ? mul_lazy<F>(sub_raw2<F>(E, O), load_fe(tw + (1u << s) + b)) : sub2<F>(E, O);
      }
    }
    __syncthreads();
    done = 1;
  }
  for (; done < nst; done += 2) {
    // the lower-numbered stage of the pair
    const unsigned s = GS ? s_hi - 2 - done : s_lo + done;
    const unsigned log_h = s_hi - s - 1; // >= 1
    const unsigned h = 1u << log_h, hh = h >> 1;
    for (unsigned q = threadIdx.x; q < (elems >> 2); q += NTT_BLOCK) {
      const unsigned c = q & cmask;
      const unsigned u = (q >> log_c) & (tmask >> 2);
      const unsigned g = q >> (log_c + log_t - 2);
      const unsigned t0 = ((u >> (log_h - 1)) << (log_h + 1)) | (u & (hh - 1));
      const unsigned i0 = (((g << log_t) | t0) << log_c) | c;
      const unsigned i1 = i0 + (hh << log_c), i2 = i0 + (h << log_c), i3 = i2 + (hh << log_c);
      const unsigned b = ((hi0 + g) << (s - s_lo)) | (t0 >> (s_hi - s));
      const fe *tw_s1 = tw + (2u << s) + 2 * b; // stage s+1 twiddles of blocks 2b, 2b+1
      // the step's twiddles are loaded ahead of the tile reads (for s = 0,
      // TW[1] = 1 is loaded and not used)
      const fe wa = load_fe(tw + (1u << s) + b), wb0 = load_fe(tw_s1), wb1 = load_fe(tw_s1 + 1);
      fe x0 = tile[i0], x1 = tile[i1], x2 = tile[i2], x3 = tile[i3];
      if (!GS) {
        // values < 4m in and out: the odd inputs of a butterfly go through a
        // twiddle product (< 2m), the even ones through one reduction (< 2m)
        if (s != 0) {
          x2 = mul_lazy<F>(x2, wa);
          x3 = mul_lazy<F>(x3, wa);
        } else {
          x2 = reduce2<F>(x2);
          x3 = reduce2<F>(x3);
        }
        x0 = reduce2<F>(x0);
        x1 = reduce2<F>(x1);
        const fe y0 = reduce2<F>(add_raw(x0, x2)), y2 = reduce2<F>(sub_raw2<F>(x0, x2));
        const fe y1 = mul_lazy<F>(add_raw(x1, x3), wb0);
        const fe y3 = mul_lazy<F>(sub_raw2<F>(x1, x3), wb1);
        tile[i0] = add_raw(y0, y1);
        tile[i1] = sub_raw2<F>(y0, y1);
        tile[i2] = add_raw(y2, y3);
        tile[i3] = sub_raw2<F>(y2, y3);
      } else {
        // values < 2m in and out; differences that feed a product skip the reduction
        const fe y0 = add2<F>(x0, x1), y1 = mul_lazy<F>(sub_raw2<F>(x0, x1), wb0);
        const fe y2 = add2<F>(x2, x3), y3 = mul_lazy<F>(sub_raw2<F>(x2, x3), wb1);
        fe z2, z3;
        if (s != 0) {
          z2 = mul_lazy<F>(sub_raw2<F>(y0, y2), wa);
          z3 = mul_lazy<F>(sub_raw2<F>(y1, y3), wa);
        } else {
          z2 = sub2<F>(y0, y2);
          z3 = sub2<F>(y1, y3);
        }
        tile[i0] = add2<F>(y0, y2);
        tile[i1] = add2<F>(y1, y3);
        tile[i2] = z2;
        tile[i3] = z3;
      }
    }
    __syncthreads();
  }

  const unsigned post = a.post;
  const fe scale = post == POST_SCALE ? load_fe(a.aux) : fe_zero();
  for (unsigned e = threadIdx.x; e < elems; e += NTT_BLOCK) {
    const unsigned c = e & cmask, t = (e >> log_c) & tmask, g = e >> (log_c + log_t);
    const unsigned idx = ((hi0 + g) << (L - s_lo)) | (t << log_lo) | (lo0 + c);
    fe v = tile[e];
    switch (post) {
    case POST_REDUCE:
      v = reduce4<F>(v); // CT tiles hold values < 4m
      break;
    case POST_SCALE:
      v = mul<F>(v, scale);
      break;
    case POST_TABLE:
      v = mul<F>(v, twist_pow(a.aux, GS ? idx : brev_bits(idx, L)));
      break;
    default:
      break;
    }
    store_fe(a.out + idx, v);
  }
}

// A pass of a launch too small to fill the GPU.  Its time is the chain of one
// thread's products, barriers and loads, so a thread forms one radix-2 butterfly
// a stage (tiles of at most 512 elements for 256 threads, one wave per SIMD)
// where a radix-4 step of the kernel above has four products in a row, and the
// next stage's twiddle is loaded during the current one.  2^12 elements 29 ->
// 17 us, 2^17 42 -> 31 us.
template <bool GS> __global__ __launch_bounds__(NTT_SMALL_BLOCK) void ntt_small_pass_kernel(const pass_table pt) {
  using F = FrParams;
  __shared__ fe tile[2 * NTT_SMALL_BLOCK];
  unsigned jl = 0, jh = pt.count; // job of this block
  while (jh - jl > 1) {
    const unsigned mid = (jl + jh) >> 1;
    if (pt.job[mid].tile_begin <= blockIdx.x)
      jl = mid;
    else
      jh = mid;
  }
  const pass_job &a = pt.job[jl];
  const unsigned L = a.log_n, s_lo = a.s_lo, s_hi = a.s_hi, log_c = a.log_c, log_g = a.log_g;
  const unsigned log_t = s_hi - s_lo, log_lo = L - s_hi;
  const unsigned t = blockIdx.x - a.tile_begin;
  if (t >= 1u << (L - log_t - log_c - log_g))
    return; // alignment padding
  const fe *__restrict__ tw = a.inverse ? pt.tw_inv : pt.tw_fwd;
  const unsigned lo0 = (t & ((1u << (log_lo - log_c)) - 1)) << log_c, hi0 = (t >> (log_lo - log_c)) << log_g;
  const unsigned elems = 1u << (log_g + log_t + log_c), cmask = (1u << log_c) - 1, tmask = (1u << log_t) - 1;
  auto index_of = [&](unsigned e) {
    const unsigned c = e & cmask, row = (e >> log_c) & tmask, g = e >> (log_c + log_t);
    return ((hi0 + g) << (L - s_lo)) | (row << log_lo) | (lo0 + c);
  };
  // the thread's butterfly of stage s: elements i0, i1 and its block b
  const unsigned q = threadIdx.x, c = q & cmask, r = (q >> log_c) & (tmask >> 1), g = q >> (log_c + log_t - 1);
  const bool active = q < (elems >> 1);
  auto twiddle = [&](unsigned s) {
    const unsigned log_h = s_hi - s - 1, b = ((hi0 + g) << (s - s_lo)) | (r >> log_h);
    return active ? load_fe(tw + (1u << s) + b) : fe_zero();
  };
  fe w = twiddle(GS ? s_hi - 1 : s_lo);
#pragma unroll
  for (unsigned k = 0; k < 2; k++) {
    const unsigned e = threadIdx.x + k * NTT_SMALL_BLOCK;
    if (e < elems) {
      const unsigned idx = index_of(e);
      fe v = load_fe(a.in + idx);
      if (a.pre_table)
        v = mul_lazy<F>(v, twist_pow(a.aux, GS ? brev_bits(idx, L) : idx));
      tile[e] = v;
    }
  }
  __syncthreads();
  for (unsigned k = 0; k < log_t; k++) {
    const unsigned s = GS ? s_hi - 1 - k : s_lo + k;
    const fe next = k + 1 < log_t ? twiddle(GS ? s - 1 : s + 1) : w;
    if (active) {
      const unsigned log_h = s_hi - s - 1;
      const unsigned t0 = ((r >> log_h) << (log_h + 1)) | (r & ((1u << log_h) - 1));
      const unsigned i0 = (((g << log_t) | t0) << log_c) | c, i1 = i0 + (1u << (log_h + log_c));
      const fe E = tile[i0], O = tile[i1];
      if (!GS) {
        // CT tile values are < 4m; each output is < 4m again
        const fe wo = s != 0 ? mul_lazy<F>(O, w) : reduce2<F>(O);
        const fe e = reduce2<F>(E);
        tile[i0] = add_raw(e, wo);
        tile[i1] = sub_raw2<F>(e, wo);
      } else {
        // GS tile values stay < 2m
        tile[i0] = add2<F>(E, O);
        tile[i1] = s != 0 ? mul_lazy<F>(sub_raw2<F>(E, O), w) : sub2<F>(E, O);
      }
    }
    w = next;
    __syncthreads();
  }
  const unsigned post = a.post;
  const fe scale = post == POST_SCALE ? load_fe(a.aux) : fe_zero();
#pragma unroll
  for (unsigned k = 0; k < 2; k++) {
    const unsigned e = threadIdx.x + k * NTT_SMALL_BLOCK;
    if (e >= elems)
      continue;
    const unsigned idx = index_of(e);
    fe v = tile[e];
    if (post == POST_REDUCE)
      v = reduce4<F>(v);
    else if (post == POST_SCALE)
      v = mul<F>(v, scale);
    else if (post == POST_TABLE)
      v = mul<F>(v, twist_pow(a.aux, GS ? idx : brev_bits(idx, L)));
    store_fe(a.out + idx, v);
  }
}

// A pass of six stages on the matrix cores, natural to bit-reversed order: tiles
// of 64 rows x 32 columns, a quad of rows a thread and step, three radix-4 steps.
// A wave's quads share their twiddles (its two halves in the last step), whose
// matrices depend on the pass's block hi alone, so they come from L2.  The first
// step takes its quads from memory and the last returns them there; in between
// they change hands through LDS, in two arrays of 16-byte halves (lanes on
// consecutive columns then meet no bank conflict).
// The blocks of stages 12..17 are too many for matrices of their own.  Scaling
// row t of block hi by omega_{2^18}^(brev(hi) t) first makes every block's
// network that of block 0 (PRE_ROWS; a row's 32 columns share the factor).
// Bound by memory at 2^24: 0.29 ms for 1.07 GB (3.7 TB/s, where a copy reaches
// 5.2), where six stages of VALU butterflies take 0.56-0.60 ms; at 2^20 23 us,
// one round of blocks, so its loads, steps and stores follow one another.
__global__ __launch_bounds__(mf::BLOCK, 4) void ntt_mfma_kernel(const pass_table pt, const int8_t *mfma_fwd, const int8_t *mfma_inv, int two16) {
  using F = FrParams;
  extern __shared__ fe tile[];
  u32x4 *lds = reinterpret_cast<u32x4 *>(tile); // [2][mf::TILE]
  fe *multiples = tile + mf::TILE;
  unsigned jl = 0, jh = pt.count; // job of this block
  while (jh - jl > 1) {
    const unsigned mid = (jl + jh) >> 1;
    if (pt.job[mid].tile_begin <= blockIdx.x)
      jl = mid;
    else
      jh = mid;
  }
  const pass_job &a = pt.job[jl];
  const unsigned L = a.log_n, s_lo = a.s_lo, log_lo = L - s_lo - mf::STAGES;
  const unsigned tiles = 1u << (L - mf::STAGES - mf::LOG_COLS);
  unsigned t = blockIdx.x - a.tile_begin;
  if (t >= tiles)
    return; // alignment padding
  if ((tiles & 7) == 0)
    t = (t & 7) * (tiles >> 3) + (t >> 3);
  mf::make_multiples(multiples);
  const unsigned hi = t >> (log_lo - mf::LOG_COLS), lo0 = (t << mf::LOG_COLS) & ((1u << log_lo) - 1);
  const unsigned c = threadIdx.x & (mf::COLS - 1), u = threadIdx.x >> mf::LOG_COLS, lane = threadIdx.x & 63;
  const size_t base = ((size_t)hi << (L - s_lo)) + lo0 + c;
  const unsigned group = s_lo == mf::STAGES ? 1 + hi : 0;
  const v4i *matrices = reinterpret_cast<const v4i *>((a.inverse ? mfma_inv : mfma_fwd) +
                                                      (size_t)group * mf::GROUP_BLOCKS * mf::PER_BLOCK * mf::MATRIX_BYTES) + lane;
  auto block_matrices = [&](unsigned block) { return matrices + block * (mf::PER_BLOCK * mf::MATRIX_BYTES / sizeof(v4i)); };
  auto put = [&](unsigned row, const fe &v) {
    lds[row * mf::COLS + c] = u32x4{v.v[0], v.v[1], v.v[2], v.v[3]};
    lds[mf::TILE + row * mf::COLS + c] = u32x4{v.v[4], v.v[5], v.v[6], v.v[7]};
  };
  auto take = [&](unsigned row) {
    const u32x4 p = lds[row * mf::COLS + c], q = lds[mf::TILE + row * mf::COLS + c];
    fe v;
    v.v[0] = p.x, v.v[1] = p.y, v.v[2] = p.z, v.v[3] = p.w;
    v.v[4] = q.x, v.v[5] = q.y, v.v[6] = q.z, v.v[7] = q.w;
    return v;
  };
  fe x[4];
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = load_fe(a.in + base + ((size_t)(u + 16 * i) << log_lo));
  if (a.pre_table == PRE_COSET) {
#pragma unroll
    for (unsigned i = 0; i < 4; i++)
      x[i] = mul_lazy<F>(x[i], twist_pow(a.aux, (unsigned)(base + ((size_t)(u + 16 * i) << log_lo))));
  } else if (a.pre_table == PRE_ROWS) {
    fe w[4];
#pragma unroll
    for (unsigned i = 0; i < 4; i++)
      w[i] = load_fe(a.rows + hi * mf::ROWS + u + 16 * i);
#pragma unroll
    for (unsigned i = 0; i < 4; i++)
      x[i] = mul_lazy<F>(x[i], w[i]);
  }
  // the transform's inputs and what this kernel leaves are below 4r, products (of any
  // 256 bits and a lazy value) below 3r: all are taken 2r off, as the matrix products
  // need |x| < 2.64 r
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = mf::add_offset(x[i], mf::offset(-2, 1));
  __syncthreads(); // `multiples`
  mf::radix4(x, block_matrices(0), block_matrices(0), multiples, two16);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    put(u + 16 * i, x[i]);
  __syncthreads();
  const unsigned row2 = (u >> 2) * 16 + (u & 3);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = take(row2 + 4 * i);
  const unsigned block2 = __builtin_amdgcn_readfirstlane(1 + (u >> 2));
  mf::radix4(x, block_matrices(block2), block_matrices(block2), multiples, two16);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    put(row2 + 4 * i, x[i]); // the rows this thread took
  __syncthreads();
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = take(4 * u + i);
  const unsigned block3 = __builtin_amdgcn_readfirstlane(5 + (u & ~1u));
  mf::radix4(x, block_matrices(block3), block_matrices(block3 + 1), multiples, two16);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    store_fe(a.out + base + ((size_t)(4 * u + i) << log_lo), mf::add_offset(x[i], mf::offset(2, -1)));
}

// The last pass of 6..10 stages, natural to bit-reversed order: tiles of 2048
// neighbouring elements, whole blocks hi of the pass.  Scaling element t of block
// hi by omega_n^(brev(hi) t) first (a table as large as the transform, read
// once) makes every block's network that of block 0, so the first six stages run
// on the matrix cores as above (rows: the top six bits of t, columns: the lower
// bits and the blocks); the rest are VALU butterflies with the first few
// twiddles of the table.  Against the VALU pass: 2^20 94 -> 82 us for the whole
// transform, 2^22 352 -> 324, 2^24 1.38 -> 1.30 ms; its time is a product an
// element, half the bytes again for the factors, and at 2^20 one round of blocks.
__global__ __launch_bounds__(mf::BLOCK, 4) void ntt_mfma_last_kernel(const pass_table pt, const int8_t *mfma_fwd, const int8_t *mfma_inv, int two16) {
  using F = FrParams;
  extern __shared__ fe tile[];
  u32x4 *lds = reinterpret_cast<u32x4 *>(tile); // [2][mf::LAST_HALF]
  fe *multiples = tile + mf::LAST_HALF;
  unsigned jl = 0, jh = pt.count; // job of this block
  while (jh - jl > 1) {
    const unsigned mid = (jl + jh) >> 1;
    if (pt.job[mid].tile_begin <= blockIdx.x)
      jl = mid;
    else
      jh = mid;
  }
  const pass_job &a = pt.job[jl];
  const unsigned L = a.log_n, rest = L - a.s_lo - mf::STAGES; // VALU stages
  const unsigned t = blockIdx.x - a.tile_begin;
  if (t >= 1u << (L - mf::STAGES - mf::LOG_COLS))
    return; // alignment padding
  mf::make_multiples(multiples);
  const unsigned c = threadIdx.x & (mf::COLS - 1), u = threadIdx.x >> mf::LOG_COLS, lane = threadIdx.x & 63;
  const size_t base = (size_t)t * mf::TILE;
  const v4i *matrices = reinterpret_cast<const v4i *>(a.inverse ? mfma_inv : mfma_fwd) + lane;
  auto block_matrices = [&](unsigned block) { return matrices + block * (mf::PER_BLOCK * mf::MATRIX_BYTES / sizeof(v4i)); };
  auto put = [&](unsigned slot, const fe &v) {
    lds[slot] = u32x4{v.v[0], v.v[1], v.v[2], v.v[3]};
    lds[mf::LAST_HALF + slot] = u32x4{v.v[4], v.v[5], v.v[6], v.v[7]};
  };
  auto take = [&](unsigned slot) {
    const u32x4 p = lds[slot], q = lds[mf::LAST_HALF + slot];
    fe v;
    v.v[0] = p.x, v.v[1] = p.y, v.v[2] = p.z, v.v[3] = p.w;
    v.v[4] = q.x, v.v[5] = q.y, v.v[6] = q.z, v.v[7] = q.w;
    return v;
  };
  // element e of the tile: block e >> (6 + rest), row, low bits
  auto slot_of = [&](unsigned e) {
    const unsigned low = e & ((1u << rest) - 1), row = (e >> rest) & (mf::ROWS - 1), g = e >> (mf::STAGES + rest);
    return row * mf::LAST_ROW + (g << rest | low);
  };
  fe x[4];
  {
    fe w[4];
#pragma unroll
    for (unsigned i = 0; i < 4; i++) {
      const size_t idx = base + threadIdx.x + i * mf::BLOCK;
      x[i] = load_fe(a.in + idx);
      w[i] = load_fe(a.rows + idx);
    }
#pragma unroll
    for (unsigned i = 0; i < 4; i++)
      put(slot_of(threadIdx.x + i * mf::BLOCK), mf::add_offset(mul_lazy<F>(x[i], w[i]), mf::offset(0, 1)));
  }
  __syncthreads();
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = take((u + 16 * i) * mf::LAST_ROW + c);
  mf::radix4(x, block_matrices(0), block_matrices(0), multiples, two16);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    put((u + 16 * i) * mf::LAST_ROW + c, x[i]);
  __syncthreads();
  const unsigned row2 = (u >> 2) * 16 + (u & 3);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = take((row2 + 4 * i) * mf::LAST_ROW + c);
  const unsigned block2 = __builtin_amdgcn_readfirstlane(1 + (u >> 2));
  mf::radix4(x, block_matrices(block2), block_matrices(block2), multiples, two16);
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    put((row2 + 4 * i) * mf::LAST_ROW + c, x[i]);
  __syncthreads();
#pragma unroll
  for (unsigned i = 0; i < 4; i++)
    x[i] = take((4 * u + i) * mf::LAST_ROW + c);
  const unsigned block3 = __builtin_amdgcn_readfirstlane(5 + (u & ~1u));
  mf::radix4(x, block_matrices(block3), block_matrices(block3 + 1), multiples, two16);
#pragma unroll
  for (unsigned i = 0; i < 4; i++) // below 4r again
    put((4 * u + i) * mf::LAST_ROW + c, mf::add_offset(x[i], mf::offset(2, -1)));
  __syncthreads();

  // stages 6..: a lane per row, the column pairs and quads of its row by wave
  const fe *__restrict__ tw = a.inverse ? pt.tw_inv : pt.tw_fwd;
  const unsigned slot0 = lane * mf::LAST_ROW, wave = threadIdx.x >> 6;
  unsigned k = 0;
  if (rest & 1) {
    const unsigned log_h = rest - 1;
    const unsigned b = lane;
    const fe w = load_fe(tw + mf::ROWS + b);
#pragma unroll
    for (unsigned i = 0; i < 2; i++) {
      const unsigned v = wave + 8 * i; // of 16 pairs
      const unsigned i0 = slot0 + (((v >> log_h) << (log_h + 1)) | (v & ((1u << log_h) - 1))), i1 = i0 + (1u << log_h);
      const fe e = reduce2<F>(take(i0)), wo = mul_lazy<F>(take(i1), w);
      put(i0, add_raw(e, wo));
      put(i1, sub_raw2<F>(e, wo));
    }
    __syncthreads();
    k = 1;
  }
  for (; k < rest; k += 2) {
    const unsigned log_hh = rest - 2 - k, hh = 1u << log_hh; // distance at stage 6 + k + 1
    const unsigned low0 = ((wave >> log_hh) << (log_hh + 2)) | (wave & (hh - 1));
    const unsigned b = lane << k | ((low0 & ((1u << rest) - 1)) >> (rest - k));
    const unsigned i0 = slot0 + low0, i1 = i0 + hh, i2 = i1 + hh, i3 = i2 + hh;
    const fe *tw_s1 = tw + (2u << (mf::STAGES + k)) + 2 * b;
    const fe wa = load_fe(tw + (1u << (mf::STAGES + k)) + b), wb0 = load_fe(tw_s1), wb1 = load_fe(tw_s1 + 1);
    // as the radix-4 step of ntt_pass_kernel<false>
    const fe x0 = reduce2<F>(take(i0)), x1 = reduce2<F>(take(i1)), x2 = mul_lazy<F>(take(i2), wa), x3 = mul_lazy<F>(take(i3), wa);
    const fe y0 = reduce2<F>(add_raw(x0, x2)), y2 = reduce2<F>(sub_raw2<F>(x0, x2));
    const fe y1 = mul_lazy<F>(add_raw(x1, x3), wb0);
    const fe y3 = mul_lazy<F>(sub_raw2<F>(x1, x3), wb1);
    put(i0, add_raw(y0, y1));
    put(i1, sub_raw2<F>(y0, y1));
    put(i2, add_raw(y2, y3));
    put(i3, sub_raw2<F>(y2, y3));
    __syncthreads();
  }
  const unsigned post = a.post;
  const fe scale = post == POST_SCALE ? load_fe(a.aux) : fe_zero();
#pragma unroll
  for (unsigned i = 0; i < 4; i++) {
    const unsigned e = threadIdx.x + i * mf::BLOCK;
    const size_t idx = base + e;
    fe v = take(slot_of(e));
    if (post == POST_REDUCE)
      v = reduce4<F>(v);
    else if (post == POST_SCALE)
      v = mul<F>(v, scale);
    else
      v = mul<F>(v, twist_pow(a.aux, brev_bits((unsigned)idx, L)));
    store_fe(a.out + idx, v);
  }
}

// fine[j] = alpha^j (j < 2^12), coarse[j] = scale * alpha^(j << 12), so that
// twist(i) = fine[i mod 2^12] * coarse[i >> 12] = scale * alpha^i (fine[0] is
// skipped).  The digit table of alpha comes from the host, so an entry is a chain
// of at most 10 products: 6.6 us at 2^20 elements, where square-and-multiply in the
// thread took 16 us.
__global__ void twist_table_kernel(fe *fine, fe *coarse, const power_digits alpha, fe scale, unsigned coarse_count, unsigned coarse_digits) {
  const unsigned j = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned nf = 1u << TWIST_FINE_BITS;
  if (j < nf)
    store_fe(fine + j, power_of(alpha, j, TWIST_FINE_BITS / 2));
  else if (j - nf < coarse_count)
    store_fe(coarse + (j - nf), mul<FrParams>(scale, power_of(alpha, j - nf, coarse_digits, TWIST_FINE_BITS / 2)));
}

struct pass_plan {
  unsigned s_lo, s_hi;
  bool mfma;               // ntt_mfma_kernel, or ntt_mfma_last_kernel with
  const fe *last = nullptr; // its row factors
};

// Passes of a launch of ntt_small_pass_kernel: as few as its tiles allow, balanced.
std::vector<pass_plan> plan_small_passes(unsigned L) {
  std::vector<pass_plan> p;
  const unsigned passes = (L + NTT_SMALL_LOG_TILE - 1) / NTT_SMALL_LOG_TILE;
  for (unsigned i = 0, s = 0; i < passes; i++) {
    const unsigned len = L / passes + (i < L % passes ? 1 : 0);
    p.push_back({s, s + len, false});
    s += len;
  }
  return p;
}

// Stage runs of the HBM passes.  Large natural-order transforms start on the
// matrix cores, whatever the tuning table names (2^24: 1.28 ms against 2.2 ms in
// named passes); else ceil(L / NTT_LOG_TILE) passes, balanced, or a first pass of
// the named stage count and the rest balanced over the remaining ones.
std::vector<pass_plan> plan_passes(unsigned L, bool bitrev_in, const fe *last_rows) {
  std::vector<pass_plan> p;
  unsigned passes = ntt_passes(L), s = 0;
  if (!bitrev_in && L >= NTT_MFMA_MIN_LOG) {
    // a third pass where a pass of VALU butterflies would follow it anyway
    const unsigned mfma_stages = L >= NTT_MFMA_ROWS_MIN_LOG ? mf::ROWS_STAGE + mf::STAGES : mf::ROWS_STAGE;
    for (; s < mfma_stages; s += mf::STAGES)
      p.push_back({s, s + mf::STAGES, true});
    passes = ntt_passes(L - s);
    if (last_rows) {
      p.push_back({s, L, true, last_rows});
      return p;
    }
  } else if (const unsigned first = passes >= 2 ? ntt_first_pass(L) : 0; first && ntt_split_valid(L, first)) {
    p.push_back({0, first, false});
    s = first;
    passes--;
  }
  const unsigned rest = L - s;
  for (unsigned i = 0; i < passes; i++) {
    const unsigned len = rest / passes + (i < rest % passes ? 1 : 0);
    p.push_back({s, s + len, false});
    s += len;
  }
  return p;
}

fe inverse_power_of_two(unsigned L) {
  using F = FrParams;
  const fe two_inv = bc::inverse<F>(add<F>(fe_one<F>(), fe_one<F>()));
  fe r = fe_one<F>();
  for (unsigned i = 0; i < L; i++)
    r = mul<F>(r, two_inv);
  return r;
}

// The row factors of the last pass for every size up to 2^log_size that has none
// yet, made with the twiddles of that size and not by the transforms, which then
// neither allocate nor wait.  They save a transform 6 to 13 %, so they leave an
// eighth of the GPU's memory to the caller; without its table a transform's
// last stages are a VALU pass, to the same result.
hipError_t make_last_rows(twiddle_state &t, const ff_state &ff, unsigned log_size, hipStream_t stream) {
  struct made {
    const fe **slot;
    fe *rows;
  };
  std::vector<made> tables;
  hipError_t e = hipSuccess;
  for (unsigned L = NTT_MFMA_MIN_LOG; L <= std::min(log_size, NTT_MFMA_LAST_MAX_LOG) && e == hipSuccess; L++) {
    if (!ntt_mfma_last(L))
      continue;
    const unsigned s_lo = L >= NTT_MFMA_ROWS_MIN_LOG ? mf::ROWS_STAGE + mf::STAGES : mf::ROWS_STAGE;
    for (int inverse = 0; inverse < 2 && e == hipSuccess; inverse++) {
      if (t.last_rows[inverse][L])
        continue;
      size_t free = 0, total = 0;
      fe *f = nullptr;
      if (hipMemGetInfo(&free, &total) != hipSuccess || free < total / 8 + (sizeof(fe) << L) || hipMalloc(&f, sizeof(fe) << L) != hipSuccess) {
        (void)hipGetLastError();
        continue;
      }
      tables.push_back({&t.last_rows[inverse][L], f});
      row_factor_kernel<<<grid_for((size_t)1 << L, 256), 256, 0, stream>>>(ff.w, f, s_lo, L - s_lo, inverse != 0);
      e = hipGetLastError();
    }
  }
  // other streams may use a table as soon as it is published
  if (!tables.empty() && e == hipSuccess)
    e = hipStreamSynchronize(stream);
  for (const made &m : tables)
    if (e == hipSuccess)
      *m.slot = m.rows;
    else
      (void)hipFree(m.rows);
  return e;
}

} // namespace

// Twiddles for 2^max_log_n and kernel attributes of the current device.  Growing
// the tables synchronises `stream`; older tables stay alive until ntt_tear_down
// because in-flight work may still read them.
hipError_t ntt_prepare(unsigned max_log_n, hipStream_t stream, ntt_tables *out) {
  std::lock_guard<std::mutex> lock(g_tw_mutex);
  const int d = device_slot();
  if (d < 0)
    return hipErrorInvalidDevice;
  twiddle_state &t = g_tw[d];
  if (!t.attributes) {
    const int bytes = (int)(sizeof(fe) << NTT_LOG_TILE);
    BC_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&ntt_pass_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    BC_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&ntt_pass_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    BC_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&ntt_mfma_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)mf::LDS_BYTES));
    BC_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&ntt_mfma_last_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)mf::LAST_LDS_BYTES));
    t.attributes = true;
  }
  if (!t.inv_sizes) {
    std::vector<fe> sizes(NTT_MAX_LOG + 1);
    for (unsigned i = 0; i <= NTT_MAX_LOG; i++)
      sizes[i] = inverse_power_of_two(i);
    fe *d = nullptr;
    BC_TRY(hipMalloc(&d, sizeof(fe) * sizes.size()));
    BC_TRY(hipMemcpy(d, sizes.data(), sizeof(fe) * sizes.size(), hipMemcpyHostToDevice));
    t.inv_sizes = d;
  }
  if (t.log_size < max_log_n) {
    const ff_state *ff = ff_current();
    if (!ff)
      return hipErrorNotInitialized;
    const unsigned log_size = std::max(max_log_n, 12u);
    fe *f = nullptr, *i = nullptr;
    BC_TRY(hipMalloc(&f, sizeof(fe) << log_size));
    BC_TRY(hipMalloc(&i, sizeof(fe) << log_size));
    twiddle_build_kernel<<<grid_for(1u << log_size, 256), 256, 0, stream>>>(ff->w, f, i, log_size);
    BC_LAUNCH_CHECK();
    // other streams may use the tables as soon as they are published
    BC_TRY(hipStreamSynchronize(stream));
    if (t.fwd) {
      t.retired.push_back(t.fwd);
      t.retired.push_back(t.inv);
    }
    t.fwd = f;
    t.inv = i;
    t.log_size = log_size;
    BC_TRY(make_last_rows(t, *ff, log_size, stream));
  }
  if (!t.mfma_fwd && max_log_n >= NTT_MFMA_MIN_LOG) {
    int8_t *m = nullptr;
    BC_TRY(hipMalloc(&m, 2 * mf::TABLE_BYTES));
    const unsigned rows = mf::TABLE_BYTES / 32;
    mf::matrix_kernel<<<grid_for(rows, 256), 256, 0, stream>>>(t.fwd, m);
    BC_LAUNCH_CHECK();
    mf::matrix_kernel<<<grid_for(rows, 256), 256, 0, stream>>>(t.inv, m + mf::TABLE_BYTES);
    BC_LAUNCH_CHECK();
    BC_TRY(hipStreamSynchronize(stream));
    t.mfma_fwd = m;
    t.mfma_inv = m + mf::TABLE_BYTES;
  }
  if (!t.rows_fwd && max_log_n >= NTT_MFMA_ROWS_MIN_LOG) {
    const ff_state *ff = ff_current();
    if (!ff)
      return hipErrorNotInitialized;
    fe *f = nullptr;
    BC_TRY(hipMalloc(&f, 2 * sizeof(fe) * mf::ROW_FACTORS));
    for (int inv = 0; inv < 2; inv++) {
      row_factor_kernel<<<grid_for(mf::ROW_FACTORS, 256), 256, 0, stream>>>(ff->w, f + inv * mf::ROW_FACTORS, mf::ROWS_STAGE, mf::STAGES, inv != 0);
      BC_LAUNCH_CHECK();
    }
    BC_TRY(hipStreamSynchronize(stream));
    t.rows_fwd = f;
    t.rows_inv = f + mf::ROW_FACTORS;
  }
  if (out) {
    *out = ntt_tables{t.fwd, t.inv, t.inv_sizes, t.mfma_fwd, t.mfma_inv, t.rows_fwd, t.rows_inv, {}, t.log_size};
    std::copy(&t.last_rows[0][0], &t.last_rows[0][0] + sizeof(t.last_rows) / sizeof(fe *), &out->last_rows[0][0]);
  }
  return hipSuccess;
}

hipError_t ntt_prepare_jobs(const ntt_job *jobs, unsigned count, hipStream_t stream) {
  unsigned max_log = 0;
  for (unsigned j = 0; j < count; j++)
    max_log = std::max(max_log, jobs[j].log_n);
  if (max_log == 0)
    return hipSuccess;
  return ntt_prepare(max_log, stream, nullptr);
}

hipError_t ntt_batch_device(const ntt_job *jobs, unsigned count, arena &ar, bool small_passes) {
  using F = FrParams;
  hipStream_t stream = ar.stream();
  if (count == 0)
    return hipSuccess;
  if (count > NTT_MAX_JOBS)
    return hipErrorInvalidValue;
  unsigned max_log = 0;
  for (unsigned j = 0; j < count; j++) {
    const ntt_job &q = jobs[j];
    if (!ntt_job_valid(q))
      return hipErrorInvalidValue;
    max_log = std::max(max_log, q.log_n);
  }
  ntt_tables tt{};
  BC_TRY(ntt_prepare(max_log, stream, &tt));

  // per-job twist tables: forward coset -> rho^i; inverse -> n^-1 * rho^-i
  std::vector<fe *> twist(count, nullptr);
  for (unsigned j = 0; j < count; j++) {
    const ntt_job &q = jobs[j];
    if (!q.log_ext)
      continue;
    const unsigned L = q.log_n;
    const unsigned coarse_count = L > TWIST_FINE_BITS ? 1u << (L - TWIST_FINE_BITS) : 1u;
    fe seven = fe_zero();
    seven.v[0] = F::generator;
    const fe g = to_mont<F>(seven);
    const fe w_big = pow_u64<F>(fe_const<F>(F::omega), 1ull << (F::omega_log_order - L - q.log_ext));
    fe rho = mul<F>(g, pow_u64<F>(w_big, q.coset));
    if (q.inverse)
      rho = bc::inverse<F>(rho);
    const unsigned coarse_digits = power_digits_for(coarse_count);
    power_digits digits;
    power_digits_fill(digits, rho, TWIST_FINE_BITS / 2 + coarse_digits);
    const unsigned entries = (1u << TWIST_FINE_BITS) + coarse_count;
    BC_TRY(ar.get(&twist[j], entries));
    twist_table_kernel<<<grid_for(entries, 64), 64, 0, stream>>>(twist[j], twist[j] + (1u << TWIST_FINE_BITS), digits,
                                                                q.inverse ? inverse_power_of_two(L) : fe_one<F>(), coarse_count, coarse_digits);
    BC_LAUNCH_CHECK();
  }

  // a launch that cannot fill the GPU takes the small passes, whatever the tuning
  // table names for the large ones (2^12: 17 us against 28 us)
  uint64_t elements = 0;
  for (unsigned j = 0; j < count; j++)
    elements += 1ull << jobs[j].log_n;
  const bool small = small_passes && max_log <= 2 * NTT_SMALL_LOG_TILE && elements <= NTT_SMALL_ELEMENTS;
  const unsigned log_tile = small ? NTT_SMALL_LOG_TILE : NTT_LOG_TILE;

  std::vector<std::vector<pass_plan>> plans(count);
  unsigned max_passes = 0;
  for (unsigned j = 0; j < count; j++) {
    if (small) {
      plans[j] = plan_small_passes(jobs[j].log_n);
    } else {
      const unsigned L = jobs[j].log_n;
      plans[j] = plan_passes(L, jobs[j].bitrev_in, ntt_mfma_last(L) ? tt.last_rows[jobs[j].inverse][L] : nullptr);
    }
    max_passes = std::max(max_passes, (unsigned)plans[j].size());
  }
  for (unsigned k = 0; k < max_passes; k++) {
    // butterfly order and kernel: Cooley-Tukey, Gentleman-Sande, Cooley-Tukey on the matrix cores (and its last pass)
    for (int form = 0; form < 4; form++) {
      const int gs = form == 1;
      const bool mfma = form >= 2, last = form == 3;
      pass_table pt{};
      pt.tw_fwd = tt.fwd;
      pt.tw_inv = tt.inv;
      uint32_t blocks = 0;
      size_t lds = 0;
      for (unsigned j = 0; j < count; j++) {
        const ntt_job &q = jobs[j];
        const unsigned np = (unsigned)plans[j].size();
        if ((int)q.bitrev_in != gs || k >= np)
          continue;
        const pass_plan pp = q.bitrev_in ? plans[j][np - 1 - k] : plans[j][k];
        if (pp.mfma != mfma || (pp.last != nullptr) != last)
          continue;
        const unsigned L = q.log_n;
        const unsigned log_t = pp.s_hi - pp.s_lo;
        const unsigned log_lo = L - pp.s_hi, log_hi = pp.s_lo;
        const unsigned room = log_tile - log_t;
        const unsigned log_c = std::min(log_lo, room);
        const unsigned log_g = log_c == log_lo ? std::min(room - log_c, log_hi) : 0;
        pass_job &a = pt.job[pt.count++];
        a.in = k == 0 ? q.in : q.out;
        a.out = q.out;
        a.log_n = (uint8_t)L;
        a.s_lo = (uint8_t)pp.s_lo;
        a.s_hi = (uint8_t)pp.s_hi;
        a.log_c = (uint8_t)log_c;
        a.log_g = (uint8_t)log_g;
        a.inverse = q.inverse ? 1 : 0;
        a.pre_table = (k == 0 && q.log_ext && !q.inverse) ? PRE_COSET : PRE_NONE;
        a.aux = twist[j];
        if (last) {
          a.rows = pp.last;
        } else if (mfma && pp.s_lo == mf::ROWS_STAGE) {
          a.pre_table = PRE_ROWS;
          a.rows = q.inverse ? tt.rows_inv : tt.rows_fwd;
        }
        if (k == np - 1) {
          if (!q.inverse)
            a.post = POST_REDUCE;
          else if (q.log_ext)
            a.post = POST_TABLE;
          else {
            a.post = POST_SCALE;
            a.aux = tt.inv_sizes + L;
          }
        } else {
          a.post = POST_LAZY;
        }
        a.tile_begin = blocks;
        const uint32_t tiles = mfma ? 1u << (L - mf::STAGES - mf::LOG_COLS) : 1u << (L - log_t - log_c - log_g);
        blocks += (tiles + 7) & ~7u;
        lds = std::max(lds, sizeof(fe) << (log_g + log_t + log_c));
      }
      if (pt.count == 0)
        continue;
      if (last)
        ntt_mfma_last_kernel<<<blocks, mf::BLOCK, mf::LAST_LDS_BYTES, stream>>>(pt, tt.mfma_fwd, tt.mfma_inv, 1 << 16);
      else if (mfma)
        ntt_mfma_kernel<<<blocks, mf::BLOCK, mf::LDS_BYTES, stream>>>(pt, tt.mfma_fwd, tt.mfma_inv, 1 << 16);
      else if (small && gs)
        ntt_small_pass_kernel<true><<<blocks, NTT_SMALL_BLOCK, 0, stream>>>(pt);
      else if (small)
        ntt_small_pass_kernel<false><<<blocks, NTT_SMALL_BLOCK, 0, stream>>>(pt);
      else if (gs)
        ntt_pass_kernel<true><<<blocks, NTT_BLOCK, lds, stream>>>(pt);
      else
        ntt_pass_kernel<false><<<blocks, NTT_BLOCK, lds, stream>>>(pt);
      BC_LAUNCH_CHECK();
    }
  }
  for (fe *p : twist)
    if (p)
      BC_TRY(ar.put(p));
  return hipSuccess;
}

hipError_t ntt_tear_down_impl() {
  std::lock_guard<std::mutex> lock(g_tw_mutex);
  const int d = device_slot();
  if (d < 0)
    return hipErrorInvalidDevice;
  twiddle_state &t = g_tw[d];
  BC_TRY(hipDeviceSynchronize());
  for (fe *p : t.retired)
    BC_TRY(hipFree(p));
  if (t.fwd) {
    BC_TRY(hipFree(t.fwd));
    BC_TRY(hipFree(t.inv));
  }
  if (t.inv_sizes)
    BC_TRY(hipFree(t.inv_sizes));
  if (t.mfma_fwd)
    BC_TRY(hipFree(t.mfma_fwd));
  if (t.rows_fwd)
    BC_TRY(hipFree(t.rows_fwd));
  for (auto &direction : t.last_rows)
    for (const fe *p : direction)
      if (p)
        BC_TRY(hipFree(const_cast<fe *>(p)));
  t = twiddle_state{};
  return hipSuccess;
}

hipError_t ntt_set_up_impl() {
  if (!ff_current())
    return hipErrorNotInitialized;
  BC_TRY(ntt_prepare(20, nullptr, nullptr));
  return hipDeviceSynchronize();
}

// Host-pointer handling of ntt_execute_async (src/ntt.cu:155-231): inputs and
// outputs may each be device, pinned or pageable memory.  Temporaries are
// released on every return path.
hipError_t ntt_execute(const ntt_configuration &c) {
  hipStream_t s = to_stream(c.stream);
  const unsigned L = c.log_values_count;
  // checked before anything is allocated or copied
  if (!ntt_shape_valid(L, c.log_extension_degree, c.coset_index) || !c.inputs || !c.outputs)
    return hipErrorInvalidValue;
  call_resources res(to_pool(c.mem_pool), s);
  const size_t bytes = sizeof(fe) << L;
  const bool in_host = classify_pointer(c.inputs) != mem_kind::device;
  const bool out_host = classify_pointer(c.outputs) != mem_kind::device;
  fe *d_in = static_cast<fe *>(c.inputs);
  fe *d_out = static_cast<fe *>(c.outputs);
  fe *staged_in = nullptr;
  if (in_host)
    BC_TRY(res.get(&staged_in, (size_t)1 << L));
  if (out_host && !in_host && !c.can_overwrite_inputs)
    BC_TRY(res.get(&d_out, (size_t)1 << L));
  const ntt_job probe{d_in, d_out, L, c.bit_reversed_inputs, c.inverse, c.log_extension_degree, c.coset_index};
  // only a coset transform has temporaries (releasing an unused block costs the
  // host 8 us, a third of a small transform)
  const size_t block_bytes = c.log_extension_degree ? ntt_footprint(probe) : 0;
  char *block = nullptr;
  if (block_bytes)
    BC_TRY(res.get(&block, block_bytes));
  if (in_host) {
    BC_TRY(hipMemcpyAsync(staged_in, c.inputs, bytes, hipMemcpyHostToDevice, s));
    if (c.h2d_copy_finished.handle)
      BC_TRY(hipEventRecord(to_event(c.h2d_copy_finished), s));
    if (c.h2d_copy_finished_callback)
      BC_TRY(hipLaunchHostFunc(s, c.h2d_copy_finished_callback, c.h2d_copy_finished_callback_data));
    d_in = staged_in;
  }
  if (out_host && (in_host || c.can_overwrite_inputs))
    d_out = d_in; // transform in place in the staging copy (or the caller's device inputs)
  const ntt_job job{d_in, d_out, L, c.bit_reversed_inputs, c.inverse, c.log_extension_degree, c.coset_index};
  arena ar = arena::bump_mode(block, block_bytes, s);
  BC_TRY(ntt_batch_device(&job, 1, ar));
  if (out_host) {
    BC_TRY(hipMemcpyAsync(c.outputs, d_out, bytes, hipMemcpyDeviceToHost, s));
    if (c.d2h_copy_finished.handle)
      BC_TRY(hipEventRecord(to_event(c.d2h_copy_finished), s));
    if (c.d2h_copy_finished_callback)
      BC_TRY(hipLaunchHostFunc(s, c.d2h_copy_finished_callback, c.d2h_copy_finished_callback_data));
  }
  return hipSuccess;
}

} // namespace bc

using namespace bc;

extern "C" {

bc_error ntt_set_up() { return as_bc(ntt_set_up_impl()); }

bc_error ntt_execute_async(ntt_configuration configuration) { return as_bc(ntt_execute(configuration)); }

bc_error ntt_execute_async_multigpu(const ntt_configuration *configurations, const int *dev_ids, unsigned log_n_devs) {
  if (log_n_devs != 0)
    return bc_error_invalid_value;
  int prev = 0;
  BC_TRY_BC(hipGetDevice(&prev));
  BC_TRY_BC(hipSetDevice(dev_ids[0]));
  const hipError_t e = ntt_execute(configurations[0]);
  (void)hipSetDevice(prev);
  return as_bc(e);
}

bc_error ntt_tear_down() { return as_bc(ntt_tear_down_impl()); }

} // extern "C"
