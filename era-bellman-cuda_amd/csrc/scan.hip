// Device-wide scans and reductions, replacing the reference's cub calls
// (src/bellman-cuda-cub.cu:30-64): u32 exclusive sum and Fr inclusive prefix
// product (grand product).
#include "device.cuh"
#include "scan.h"

namespace bc {

constexpr unsigned SCAN_BLOCK = 256;

// ---------------- u32 exclusive sum ----------------
// Reduce-then-scan over tiles: one launch sums every tile, one block scans the
// tile sums, one launch scans every tile from its prefix (three launches up to
// U32_TILE * U32_TOTALS entries; the tile sums of larger inputs are scanned
// recursively).  A thread owns U32_ITEMS consecutive entries (four 16-byte
// loads and stores when aligned), so a tile needs one block-wide scan of the
// thread sums: wave shuffles and one LDS exchange of the wave totals.
constexpr unsigned U32_BLOCK = 256;
constexpr unsigned U32_ITEMS = 16;
constexpr unsigned U32_TILE = U32_BLOCK * U32_ITEMS;
constexpr unsigned U32_TOTALS_BLOCK = 1024;
constexpr unsigned U32_TOTALS = U32_TOTALS_BLOCK * U32_ITEMS; // most tile sums one block scans

// exclusive prefix of v over the block (blockDim.x = 64 * waves, waves <= 16);
// *total receives the block's sum.  sh holds one word per wave.
__device__ __forceinline__ uint32_t block_exclusive_u32(uint32_t v, uint32_t *sh, uint32_t *total) {
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (unsigned off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, 64);
    if (lane >= off)
      x += y;
  }
  if (lane == 63)
    sh[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (unsigned w = 0; w < waves; w++) {
    const uint32_t t = sh[w];
    before += w < wave ? t : 0u;
    all += t;
  }
  *total = all;
  return before + x - v;
}

// the `count` (<= U32_ITEMS) entries of a thread from `first`; 16-byte loads
// when all U32_ITEMS are in range and aligned
__device__ __forceinline__ void load_items(const uint32_t *in, size_t first, size_t n, unsigned count, uint32_t (&v)[U32_ITEMS]) {
  const uint32_t *p = in + first;
  if (count == U32_ITEMS && first + U32_ITEMS <= n && ((uintptr_t)p & 15) == 0) {
#pragma unroll
    for (unsigned q = 0; q < U32_ITEMS / 4; q++) {
      const uint4 w = reinterpret_cast<const uint4 *>(p)[q];
      v[4 * q] = w.x;
      v[4 * q + 1] = w.y;
      v[4 * q + 2] = w.z;
      v[4 * q + 3] = w.w;
    }
    return;
  }
#pragma unroll
  for (unsigned k = 0; k < U32_ITEMS; k++)
    v[k] = k < count && first + k < n ? p[k] : 0u;
}

__global__ __launch_bounds__(U32_BLOCK) void scan_u32_reduce_kernel(const uint32_t *in, uint32_t *tile_sums, size_t n) {
  __shared__ uint32_t sh[U32_BLOCK / 64];
  uint32_t v[U32_ITEMS];
  load_items(in, (size_t)blockIdx.x * U32_TILE + (size_t)threadIdx.x * U32_ITEMS, n, U32_ITEMS, v);
  uint32_t sum = 0;
#pragma unroll
  for (unsigned k = 0; k < U32_ITEMS; k++)
    sum += v[k];
#pragma unroll
  for (unsigned off = 32; off > 0; off >>= 1)
    sum += __shfl_xor(sum, off, 64);
  if ((threadIdx.x & 63) == 0)
    sh[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (unsigned w = 0; w < U32_BLOCK / 64; w++)
      t += sh[w];
    tile_sums[blockIdx.x] = t;
  }
}

// Block b scans entries [b * BLOCK * items, +BLOCK * items) from prefix[b]
// (0 without a prefix), `items` (<= U32_ITEMS) consecutive entries per thread.
template <unsigned BLOCK>
__global__ __launch_bounds__(BLOCK) void scan_u32_tile_kernel(const uint32_t *in, uint32_t *out, const uint32_t *prefix, size_t n, unsigned items) {
  __shared__ uint32_t sh[BLOCK / 64];
  const size_t first = (size_t)blockIdx.x * BLOCK * items + (size_t)threadIdx.x * items;
  uint32_t v[U32_ITEMS];
  load_items(in, first, n, items, v);
  uint32_t sum = 0;
#pragma unroll
  for (unsigned k = 0; k < U32_ITEMS; k++)
    sum += v[k];
  uint32_t total;
  uint32_t run = (prefix ? prefix[blockIdx.x] : 0u) + block_exclusive_u32(sum, sh, &total);
  uint32_t *p = out + first;
  if (items == U32_ITEMS && first + U32_ITEMS <= n && ((uintptr_t)p & 15) == 0) {
#pragma unroll
    for (unsigned q = 0; q < U32_ITEMS / 4; q++) {
      uint4 w;
      w.x = run;
      run += v[4 * q];
      w.y = run;
      run += v[4 * q + 1];
      w.z = run;
      run += v[4 * q + 2];
      w.w = run;
      run += v[4 * q + 3];
      reinterpret_cast<uint4 *>(p)[q] = w;
    }
    return;
  }
#pragma unroll
  for (unsigned k = 0; k < U32_ITEMS; k++) {
    if (k < items && first + k < n)
      p[k] = run;
    run += v[k];
  }
}

// out[i] = sum_{j<i} in[j]; in and out may alias.
hipError_t scan_u32_exclusive(const uint32_t *in, uint32_t *out, size_t n, arena &ar) {
  hipStream_t stream = ar.stream();
  if (n == 0)
    return hipSuccess;
  if (n <= U32_TOTALS) {
    const unsigned items = (unsigned)((n + U32_TOTALS_BLOCK - 1) / U32_TOTALS_BLOCK);
    scan_u32_tile_kernel<U32_TOTALS_BLOCK><<<1, U32_TOTALS_BLOCK, 0, stream>>>(in, out, nullptr, n, items);
    return hipGetLastError();
  }
  const size_t tiles = (n + U32_TILE - 1) / U32_TILE;
  uint32_t *sums = nullptr;
  BC_TRY(ar.get(&sums, tiles));
  scan_u32_reduce_kernel<<<(unsigned)tiles, U32_BLOCK, 0, stream>>>(in, sums, n);
  BC_LAUNCH_CHECK();
  BC_TRY(scan_u32_exclusive(sums, sums, tiles, ar));
  scan_u32_tile_kernel<U32_BLOCK><<<(unsigned)tiles, U32_BLOCK, 0, stream>>>(in, out, sums, n, U32_ITEMS);
  BC_LAUNCH_CHECK();
  return ar.put(sums);
}

// ---------------- Fr inclusive prefix product ----------------
// A product is about 0.5 us of a SIMD's time whatever the wave's lanes hold, so
// a block that scans a tile has four waves, one per SIMD, and a scan of few
// elements is spread over the CUs: tiles of PP_TILE elements are scanned, the
// tile products are scanned, and a second launch multiplies every tile by the
// product before it (65539 elements 37 -> 31 us, of which the 16 products
// in sequence of a tile are 8).  That is 4.5 products and 128 bytes an element.
// Above PP_TILES_MAX elements a thread instead takes PP_CHUNK consecutive ones:
// one launch multiplies up every chunk, the chunk products are scanned as above,
// and one launch walks every chunk again from the product before it: 2.6
// products and 100 bytes an element (4194299 elements 212 -> 163 us; at 2^20
// the two are equal).
constexpr unsigned PP_WAVES = SCAN_BLOCK / 64;
constexpr unsigned PP_TILE = SCAN_BLOCK * 4;
constexpr unsigned PP_CHUNK = 8;
constexpr unsigned PP_TILES_MAX = 1u << 20;

__device__ __forceinline__ fe shfl_up_fe(const fe &a, unsigned off) {
  fe r;
#pragma unroll
  for (int i = 0; i < 8; i++)
    r.v[i] = __shfl_up(a.v[i], off, 64);
  return r;
}

// Reduces a thread's elements if one of the wave's may not be lazy.
template <unsigned K> __device__ __forceinline__ void make_lazy(fe (&v)[K]) {
  bool wide = false;
#pragma unroll
  for (unsigned k = 0; k < K; k++)
    wide |= may_be_wide(v[k]);
  if (__any(wide))
#pragma unroll
    for (unsigned k = 0; k < K; k++)
      v[k] = lazy_of_wide(v[k]);
}

// Scans tiles of SCAN_BLOCK * K elements, K consecutive ones a thread; the
// product of a whole tile goes to tile_products (if any).
template <unsigned K>
__global__ __launch_bounds__(SCAN_BLOCK) void prefix_product_tile_kernel(const fe *in, fe *out, fe *tile_products, size_t n) {
  using F = FrParams;
  __shared__ fe wave_product[PP_WAVES];
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const size_t first = ((size_t)blockIdx.x * SCAN_BLOCK + threadIdx.x) * K;
  fe v[K];
#pragma unroll
  for (unsigned k = 0; k < K; k++)
    v[k] = first + k < n ? load_fe(in + first + k) : fe_one<F>();
  make_lazy(v);
#pragma unroll
  for (unsigned k = 1; k < K; k++)
    v[k] = mul_lazy<F>(v[k - 1], v[k]);
  fe incl = v[K - 1]; // of the wave's lanes up to this one
  for (unsigned off = 1; off < 64; off <<= 1) {
    const fe y = shfl_up_fe(incl, off);
    const fe xy = mul_lazy<F>(y, incl);
    if (lane >= off)
      incl = xy;
  }
  if (lane == 63)
    wave_product[wave] = incl;
  __syncthreads();
  // everything before the thread's elements: the waves before, then the lanes before
  fe before = shfl_up_fe(incl, 1);
  if (wave > 0) {
    fe w = wave_product[0];
    for (unsigned i = 1; i < wave; i++)
      w = mul_lazy<F>(w, wave_product[i]);
    before = lane > 0 ? mul_lazy<F>(w, before) : w;
  }
#pragma unroll
  for (unsigned k = 0; k < K; k++) {
    if (threadIdx.x > 0)
      v[k] = mul_lazy<F>(before, v[k]);
    v[k] = reduce<F>(v[k]);
    if (first + k < n)
      store_fe(out + first + k, v[k]);
  }
  if (tile_products && threadIdx.x == SCAN_BLOCK - 1)
    store_fe(tile_products + blockIdx.x, v[K - 1]);
}

// multiplies tile t >= 1 by the product of the tiles [0, t)
__global__ __launch_bounds__(SCAN_BLOCK) void prefix_product_fixup_kernel(fe *out, const fe *tiles_inclusive, size_t n) {
  const fe m = load_fe(tiles_inclusive + blockIdx.x);
  const size_t i = (size_t)(blockIdx.x + 1) * PP_TILE + threadIdx.x;
#pragma unroll
  for (unsigned k = 0; k < PP_TILE / SCAN_BLOCK; k++) {
    const size_t j = i + k * SCAN_BLOCK;
    if (j < n)
      store_fe(out + j, mul<FrParams>(m, load_fe(out + j)));
  }
}

// The chunk's elements are all loaded before the first product: its lines are
// then fetched once although neighbouring lanes are a chunk apart.
__device__ __forceinline__ void load_chunk(const fe *in, size_t first, size_t n, fe (&v)[PP_CHUNK]) {
#pragma unroll
  for (unsigned k = 0; k < PP_CHUNK; k++)
    v[k] = first + k < n ? load_fe(in + first + k) : fe_one<FrParams>();
  make_lazy(v);
}

__global__ __launch_bounds__(SCAN_BLOCK) void prefix_product_chunk_kernel(const fe *in, fe *products, size_t n) {
  const size_t c = (size_t)blockIdx.x * SCAN_BLOCK + threadIdx.x, first = c * PP_CHUNK;
  if (first >= n)
    return;
  fe v[PP_CHUNK];
  load_chunk(in, first, n, v);
  fe acc = v[0];
#pragma unroll
  for (unsigned k = 1; k < PP_CHUNK; k++)
    acc = mul_lazy<FrParams>(acc, v[k]);
  store_fe(products + c, acc);
}

// scanned[c]: the product of c's tile of chunks up to and including chunk c;
// tiles[t]: the product of the tiles up to and including t
__global__ __launch_bounds__(SCAN_BLOCK) void prefix_product_apply_kernel(const fe *in, fe *out, const fe *scanned, const fe *tiles, size_t n) {
  using F = FrParams;
  const size_t c = (size_t)blockIdx.x * SCAN_BLOCK + threadIdx.x, first = c * PP_CHUNK;
  if (first >= n)
    return;
  fe v[PP_CHUNK];
  load_chunk(in, first, n, v);
  fe acc = v[0];
  if (c > 0) {
    const size_t tile = (c - 1) / PP_TILE;
    fe before = load_fe(scanned + (c - 1));
    if (tile > 0)
      before = mul_lazy<F>(load_fe(tiles + (tile - 1)), before);
    acc = mul_lazy<F>(before, acc);
  }
#pragma unroll
  for (unsigned k = 0; k < PP_CHUNK; k++) {
    if (k > 0)
      acc = mul_lazy<F>(acc, v[k]);
    if (first + k < n)
      store_fe(out + first + k, reduce<F>(acc));
  }
}

// out[i] = prod_{j<=i} in[j]; in and out may alias.
hipError_t prefix_product(const fe *in, fe *out, size_t n, arena &ar) {
  hipStream_t stream = ar.stream();
  if (n == 0)
    return hipSuccess;
  if (n <= PP_TILE) {
    if (n <= SCAN_BLOCK)
      prefix_product_tile_kernel<1><<<1, SCAN_BLOCK, 0, stream>>>(in, out, nullptr, n);
    else
      prefix_product_tile_kernel<4><<<1, SCAN_BLOCK, 0, stream>>>(in, out, nullptr, n);
    return hipGetLastError();
  }
  // the chunk products are n / 8 elements; a pool without them still has the tile
  // products' n / 1024
  bool chunked = n > PP_TILES_MAX;
  size_t items = 0, tiles = 0; // elements or chunk products to scan in tiles
  fe *temp = nullptr;
  for (;;) {
    items = chunked ? (n + PP_CHUNK - 1) / PP_CHUNK : n;
    tiles = (items + PP_TILE - 1) / PP_TILE;
    const hipError_t e = ar.get(&temp, tiles + (chunked ? items : 0));
    if (e == hipSuccess)
      break;
    if (e != hipErrorOutOfMemory || !chunked)
      return e;
    (void)hipGetLastError();
    chunked = false;
  }
  fe *tile_products = temp, *chunk_products = temp + tiles;
  if (chunked) {
    prefix_product_chunk_kernel<<<grid_for(items, SCAN_BLOCK), SCAN_BLOCK, 0, stream>>>(in, chunk_products, n);
    BC_LAUNCH_CHECK();
  }
  prefix_product_tile_kernel<4><<<(unsigned)tiles, SCAN_BLOCK, 0, stream>>>(chunked ? chunk_products : in, chunked ? chunk_products : out, tile_products, items);
  BC_LAUNCH_CHECK();
  BC_TRY(prefix_product(tile_products, tile_products, tiles, ar));
  if (chunked)
    prefix_product_apply_kernel<<<grid_for(items, SCAN_BLOCK), SCAN_BLOCK, 0, stream>>>(in, out, chunk_products, tile_products, n);
  else
    prefix_product_fixup_kernel<<<(unsigned)(tiles - 1), SCAN_BLOCK, 0, stream>>>(out, tile_products, n);
  BC_LAUNCH_CHECK();
  return ar.put(temp);
}

} // namespace bc
