// Pippenger G1 MSM for gfx950, batched: every phase is one launch over all the
// MSMs of a batch (job tables travel by value in the kernel arguments, so a
// batch is a fixed launch sequence with no device-side tables to set up).  The
// plain C-ABI call is a batch of one.
//
// Contract (src/bellman-cuda.h:477-506, src/msm.cu, src/msm_kernels.cu):
//   scalars are Montgomery Fr; window width c(log n) and W = ceil(254/c) as
//   src/msm.cu:12-59; a scalar s >= r - s is replaced by r - s with a global
//   sign; signed c-bit digits with borrow lie in [0, 2^(c-1)]
//   (src/msm_kernels.cu:36-75).  The output is 254 Jacobian points, one per
//   result bit: result[w*c + j] = sum of the buckets of window w whose digit
//   has bit j set (j < c-1), and the top-digit bucket for j = c-1 and for bit
//   253 (src/msm.cu:354-414, src/msm_kernels.cu:269-299).  The caller folds
//   them as sum = 2*sum + result[i].
//
// Pipeline:
//   1. digits:     one thread per scalar writes, for each window, the key
//                  (the window-local bucket d - 1, or 2^(c-1) for a zero
//                  digit) and the value sign | point index;
//   2. sort:       one stable segmented radix sort of all (key, value) pairs
//                  of the batch, each window a segment (c key bits: two passes
//                  of <= 11 bits up to c = 22; per-tile LDS histograms,
//                  wave-ballot ranking, no global atomics, so heavy buckets
//                  cost nothing extra);
//   3. accumulate: the sorted entries of a job are cut into chunks of
//                  `piece` entries, one per thread; a thread adds its chunk's
//                  points with XYZZ mixed additions into one running sum per
//                  bucket it meets, so every lane does the same work and a
//                  heavy bucket (e.g. digit 1 of window 0 when many scalars
//                  are 1) is spread over many threads; the same pass records
//                  each bucket's run [start, end) of sorted entries;
//   4. bucket sums: a bucket's partial sums lie in consecutive slots; one launch
//                  adds them into the windows, a thread a bucket of up to a few
//                  (4..32, small_pieces), a wave of quads a listed bucket of up to
//                  64, and a block of quads every 512 sums of a larger one, whose
//                  chunks a second launch joins;
//   5. per-bit reduction: windows are split recursively into low/high halves
//                  of their index bits (sums split across threads, then folded,
//                  or by quads of lanes) until they hold at most 8 bits; then a
//                  block per window forms its per-bit sums;
//   6. gather:     254 Jacobian results per job.
#include <algorithm>
#include <functional>
#include <mutex>
#include <vector>

#include "batch.h"
#include "common.h"
#include "curve.cuh"
#include "curve29.cuh"
#include "msm.h"
#include "quad29.cuh"
#include "scan.h"
#include "sort.h"

namespace bc {

unsigned msm_window_bits(unsigned log_n) {
  switch (log_n) {
  case 14:
    return 13;
  case 15:
  case 16:
  case 17:
  case 18:
  case 19:
    return 15;
  case 20:
  case 21:
    return 16;
  case 22:
    return 17;
  case 23:
    return 19;
  case 24:
  case 25:
    return 20;
  case 26:
    return 22;
  default:
    return log_n > 3 ? log_n : 3;
  }
}

namespace {

constexpr uint32_t SIGN = 0x80000000u;
constexpr unsigned MSM_BLOCK = 256;
constexpr unsigned ACC_BLOCK = 64;
constexpr unsigned DIGITS_BLOCK = 1024; // threads of a block that also counts (4 points each)
constexpr uint64_t SPLIT_THREADS = 1u << 17; // two waves per SIMD
// First-digit counters of one digits block.  Measured at 2^24: with 15 KiB of
// counters (c = 17) counting in the digits kernel saved 0.18 ms over the
// sort's own count; with 27 KiB (c = 20) it saved nothing.
constexpr size_t DIGITS_MAX_LDS = 20 * 1024;
// Counting takes a block per 4096 points, so it pays once the tiles give every
// CU a block; below, one point a thread on all CUs and the sort's own count are
// faster: 2^12 points 120 -> 9 us (and 5 us for the count), four chunks of 2^16
// 402 -> 32 (and 17) us.  With DIGITS_BLOCK threads a tile instead of 256 the
// counting form takes 61 us instead of 104 at 2^20.
constexpr uint64_t DIGITS_MIN_TILES = 256;

struct job_desc {
  const g1_affine *bases;
  const fe *scalars;
  uint32_t entry_begin;  // first (key, value) pair of the job (a launch holds < 2^31)
  uint32_t digit_block;  // first block of the job in the digits launch
  uint32_t table_begin;  // the job's counts in the sort's first-pass table
  uint32_t bucket_begin; // first batch-global bucket
  uint32_t top_begin;    // first top-digit slot
  uint32_t chunk_begin;  // first accumulation chunk of the job
  uint32_t slot_begin;   // first partial-sum slot of the job
  uint32_t stride;       // fixed-base table: points per window block (0: plain bases)
  uint16_t piece;        // sorted entries per accumulation chunk
  uint8_t log_n;         // 2^log_n scalars
  uint8_t c;             // window bits
  uint8_t Wd;            // digit windows of a scalar, ceil(254 / c)
  uint8_t W;             // bucket windows: Wd, or 1 over a fixed-base table
  uint8_t small;         // partial sums of a bucket that one thread of the gather adds
};

static_assert(MSM_MAX_JOBS <= SEG_MAX_GROUPS, "one sort segment group per job");

struct job_table {
  uint32_t count;
  job_desc job[MSM_MAX_JOBS];
};
static_assert(sizeof(job_table) <= 4096, "kernel argument budget");

// Index of the last job whose `begin` field is <= v (fields ascend with the job index).
template <class Begin> __device__ __forceinline__ unsigned find_job(const job_table &t, uint32_t v, Begin begin) {
  unsigned lo = 0, hi = t.count;
  while (hi - lo > 1) {
    const unsigned mid = (lo + hi) >> 1;
    if (begin(t.job[mid]) <= v)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

struct by_digit_block {
  __device__ uint32_t operator()(const job_desc &d) const { return d.digit_block; }
};
struct by_bucket {
  __device__ uint32_t operator()(const job_desc &d) const { return d.bucket_begin; }
};
struct by_entry {
  __device__ uint32_t operator()(const job_desc &d) const { return d.entry_begin; }
};
struct by_chunk {
  __device__ uint32_t operator()(const job_desc &d) const { return d.chunk_begin; }
};

__global__ void fill_u32_kernel(uint32_t *p, size_t n, uint32_t v) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = v;
}

hipError_t fill_u32(uint32_t *p, size_t n, uint32_t v, hipStream_t s) {
  if (n == 0)
    return hipSuccess;
  fill_u32_kernel<<<grid_for(n, MSM_BLOCK), MSM_BLOCK, 0, s>>>(p, n, v);
  return hipGetLastError();
}

// 1. signed digits.  Entry (w, i) of a job gets the window-local key d - 1
// (2^(c-1), after every bucket, for d = 0) and value = sign << 31 | i.  Block k
// of a job takes points [k block_points, (k+1) block_points).  With
// `first_table`, block_points = SEG_TILE, so a block holds tile k of every
// window's sort segment: it also counts the sort's first digit (key bits
// [0, bits0)) per window in LDS and writes the tile's counts to the first-pass
// table, and the sort need not read the entries to count them; DIGITS_BLOCK
// threads share the tile.  Without it a block takes MSM_BLOCK points, one per
// thread.  A scalar is loaded one point ahead of its digits.
__global__ __launch_bounds__(DIGITS_BLOCK) void digits_kernel(const job_table jobs, uint64_t *__restrict__ entries, uint32_t *__restrict__ first_table,
                                                           unsigned bits0, uint32_t block_points) {
  using F = FrParams;
  // [Wd][2^min(c, bits0)] 16-bit counts (a tile has SEG_TILE entries), two per
  // word: digit d of window w is half d & 1 of word (w nd + d) / 2
  extern __shared__ uint32_t hist[];
  // blocks are dealt round-robin to the 8 XCDs; block ids are remapped so each
  // XCD takes a contiguous range of tiles, and the counts that neighbouring
  // tiles write side by side into the table meet in one L2
  const uint32_t per_xcd = gridDim.x >> 3;
  const uint32_t blk = blockIdx.x < (per_xcd << 3) ? (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
  const job_desc &jd = jobs.job[find_job(jobs, blk, by_digit_block())];
  const uint32_t k = blk - jd.digit_block, n = 1u << jd.log_n, c = jd.c, Wd = jd.Wd;
  const uint32_t top = 1u << (c - 1);
  const unsigned dbits = c < bits0 ? c : bits0; // keys are below 2^c
  const uint32_t nd = 1u << dbits;
  auto count = [&](uint32_t w, uint32_t d, uint32_t v) {
    const uint32_t slot = w * nd + d;
    atomicAdd(&hist[slot >> 1], v << ((slot & 1) << 4));
  };
  if (first_table) {
    for (uint32_t i = threadIdx.x; i < (Wd * nd + 1) / 2; i += blockDim.x)
      hist[i] = 0;
    __syncthreads();
  }
  const uint32_t p1 = min(n, (k + 1) * block_points);
  uint32_t i = k * block_points + threadIdx.x;
  fe next = i < p1 ? load_fe(jd.scalars + i) : fe_zero();
  for (; i < p1; i += blockDim.x) {
    const fe pos = from_mont<F>(next);
    if (i + blockDim.x < p1)
      next = load_fe(jd.scalars + i + blockDim.x);
    fe neg;
    sub_limbs(neg, fe_const<F>(F::m), pos); // r - s (r for s = 0)
    const uint32_t global_sign = lt(pos, neg) ? 0u : SIGN;
    const fe kk = global_sign ? neg : pos;
    uint32_t borrow = 0;
    for (unsigned w = 0; w < Wd; w++) {
      uint32_t d = extract_bits(kk, w * c, c) + borrow;
      uint32_t sign = global_sign;
      borrow = 0;
      if (d > top) {
        d = (top << 1) - d;
        borrow = 1;
        sign ^= SIGN;
      }
      const uint32_t key = d ? d - 1 : top;
      // key low, point reference high: point i, or [2^(c w)] point i of a fixed-base table
      const uint32_t point = jd.stride ? w * jd.stride + i : i;
      entries[jd.entry_begin + ((uint64_t)w << jd.log_n) + i] = (uint64_t)(sign | point) << 32 | key;
      if (first_table) {
        // zero digits (often most lanes of a wave in the high windows) are
        // counted once per wave instead of once per lane
        const uint64_t zeros = __ballot(d == 0);
        if (d != 0)
          count(w, key & (nd - 1), 1u);
        else if ((threadIdx.x & 63) == (unsigned)__ffsll((unsigned long long)zeros) - 1)
          count(w, top & (nd - 1), (uint32_t)__popcll(zeros));
      }
    }
  }
  if (first_table) {
    __syncthreads();
    // window w, digit d of tile k (digits at or above 2^c count nothing): the
    // table is [window][digit][tile] over the windows' segments, or, for a
    // fixed-base job's single segment (windows of whole tiles, n >= SEG_TILE),
    // [digit][w tiles + k]
    const uint32_t tiles = (n + SEG_TILE - 1) / SEG_TILE;
    for (uint32_t j = threadIdx.x; j < (Wd << bits0); j += blockDim.x) {
      const uint32_t w = j >> bits0, d = j & ((1u << bits0) - 1), slot = w * nd + d;
      const uint64_t at = jd.stride ? (uint64_t)d * Wd * tiles + w * tiles + k : (uint64_t)j * tiles + k;
      first_table[jd.table_begin + at] = d < nd ? (hist[slot >> 1] >> ((slot & 1) << 4)) & 0xffffu : 0u;
    }
  }
}

// 3. accumulation over equal chunks of the sorted entries.  Chunk k of a job
// is its entries [k piece, (k+1) piece); one thread adds the chunk's points
// into a running XYZZ sum and stores the sum at slot(b, k) = slot_begin +
// (b - bucket_begin) + k whenever the bucket b it was adding to ends inside the
// chunk, and at the chunk's end.  Along the sorted entries neither b nor k
// decreases, so every (chunk, bucket) pair has a slot of its own and a
// bucket's sums occupy consecutive slots.  All threads of a wave do the same
// number of additions whatever the bucket sizes (cutting buckets into pieces
// instead leaves a wave waiting for its longest piece).  The thread that holds
// a bucket's first (last) sorted entry also records where the bucket's run
// starts (ends), from the keys before and after it, so no separate pass over
// the sorted entries is needed.

// Buckets of up to d.small partial sums are summed by one thread of the gather,
// those of up to MEDIUM_PIECES by a wave of quads, larger ones by blocks of quads
// in chunks of HEAVY_CHUNK.  The additions of a thread take 7 us each in
// sequence, so the line (a rule on the job alone) lies at twice the sums of an
// average bucket, where few buckets are left to the waves; a witness has some:
// the window where its small scalars end (13 sums at 2^12 points), the top
// window (9 at 2^20, 15 at 2^24).  At 2^12 points the gather takes 23 us instead
// of 112 for 12 us more of waves.
uint8_t small_pieces(const job_desc &d) {
  const uint64_t entries_per_bucket = ((uint64_t)(d.stride ? d.Wd : 1u) << d.log_n) >> (d.c - 1);
  return (uint8_t)std::min<uint64_t>(4 + 2 * (entries_per_bucket / d.piece), 32);
}
constexpr uint32_t MEDIUM_PIECES = 64;
constexpr unsigned HEAVY_BLOCK = 256;
constexpr unsigned HEAVY_QUADS = HEAVY_BLOCK / 4;
constexpr unsigned HEAVY_CHUNK = HEAVY_QUADS * 8;
constexpr unsigned LISTED_BLOCKS = 512;
static_assert(HEAVY_BLOCK == MSM_BLOCK, "one launch for both");

// Work lists of the buckets that the gather does not sum itself: medium buckets,
// (bucket, chunk) pairs of heavy ones, and heavy buckets of several chunks.
// count[0..2] are their lengths.  Their order varies from run to run; what is
// summed in which order does not.
struct piece_lists {
  uint32_t *count, *medium, *several;
  uint2 *chunks;
};

// piece_offset[b], piece_count[b]: the slots of bucket b's sums, from its run
// [start, end) of sorted entries (empty buckets have none).
__global__ void bucket_slots_kernel(const job_table jobs, const uint32_t *start, const uint32_t *end, uint32_t *piece_offset, uint32_t *piece_count,
                                    unsigned nb, const piece_lists lists) {
  const unsigned b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb)
    return;
  const job_desc &jd = jobs.job[find_job(jobs, b, by_bucket())];
  const uint32_t s0 = start[b], e0 = end[b];
  uint32_t np = 0, off = 0;
  if (e0 > s0) {
    const uint32_t k0 = (s0 - jd.entry_begin) / jd.piece, k1 = (e0 - 1 - jd.entry_begin) / jd.piece;
    off = jd.slot_begin + (b - jd.bucket_begin) + k0;
    np = k1 - k0 + 1;
  }
  piece_offset[b] = off;
  piece_count[b] = np;
  if (np > MEDIUM_PIECES) {
    const uint32_t chunks = (np + HEAVY_CHUNK - 1) / HEAVY_CHUNK;
    const uint32_t at = atomicAdd(lists.count + 1, chunks);
    for (uint32_t k = 0; k < chunks; k++)
      lists.chunks[at + k] = make_uint2(b, k);
    if (chunks > 1)
      lists.several[atomicAdd(lists.count + 2, 1u)] = b;
  }
  // one atomic per wave: the top window's buckets are all medium, side by side
  const bool medium = np > jd.small && np <= MEDIUM_PIECES;
  const uint64_t mask = __ballot(medium);
  if (medium) {
    const unsigned lane = threadIdx.x & 63, before = __popcll(mask & ((1ull << lane) - 1)), leader = (unsigned)__ffsll((unsigned long long)mask) - 1;
    uint32_t at = 0;
    if (before == 0)
      at = atomicAdd(lists.count, (uint32_t)__popcll(mask));
    lists.medium[__shfl(at, leader, 64) + before] = b;
  }
}

__global__ __launch_bounds__(ACC_BLOCK) void accumulate_kernel(const job_table jobs, const uint64_t *__restrict__ sorted, uint32_t chunks,
                                                               xyzz29 *__restrict__ partials, uint32_t *__restrict__ run_start,
                                                               uint32_t *__restrict__ run_end) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= chunks)
    return;
  const job_desc &jd = jobs.job[find_job(jobs, t, by_chunk())];
  const g1_affine *__restrict__ bases = jd.bases;
  const uint32_t k = t - jd.chunk_begin, top = 1u << (jd.c - 1);
  const uint32_t begin = jd.entry_begin + k * jd.piece;
  const uint32_t job_end = jd.entry_begin + ((uint32_t)jd.Wd << jd.log_n);
  const uint32_t end = begin + jd.piece < job_end ? begin + jd.piece : job_end;
  // sort segments: every window, or all of a fixed-base job's entries;
  // (e - entry_begin) & seg_mask is 0 exactly at a segment's first entry
  const uint32_t seg_mask = jd.stride ? 0xffffffffu : (1u << jd.log_n) - 1;
  xyzz29 *slots = partials + (jd.slot_begin + k - jd.bucket_begin); // + batch-global bucket
  constexpr uint32_t NONE = 0xffffffffu;
  uint32_t cur = NONE;
  // the running sum in the 29-bit-limb form (infinity while `empty`)
  xyzz29 acc{};
  bool empty = true;
  // software pipeline: entries three ahead, their points one ahead (a zero
  // digit's point is not loaded; a second point in flight cost the registers
  // of the third wave per SIMD); indexes past the chunk repeat its last entry
  const uint32_t last = end - 1;
  auto point_of = [&](uint64_t ent, const g1_affine &keep) {
    return (uint32_t)ent != top ? load_affine(bases + ((uint32_t)(ent >> 32) & ~SIGN)) : keep;
  };
  uint64_t ent0 = sorted[begin], ent1 = sorted[min(begin + 1, last)], ent2 = sorted[min(begin + 2, last)];
  // bucket b occupies [run_start[b], run_end[b]) of the sorted entries; a run
  // is recorded by the chunk that holds its first (last) entry.  The chunk's
  // first bucket continues a run when the entry before it, in the same
  // segment, has its key; its last bucket continues into the next chunk alike.
  const bool starts_segment = ((begin - jd.entry_begin) & seg_mask) == 0;
  const bool continued = !starts_segment && (uint32_t)sorted[begin - 1] == (uint32_t)ent0;
  const bool next_starts_segment = end == job_end || ((end - jd.entry_begin) & seg_mask) == 0;
  const uint32_t key_after = next_starts_segment ? NONE : (uint32_t)sorted[end];
  uint32_t last_e = 0, cur_key = NONE;
  g1_affine pt0 = point_of(ent0, g1_affine{});
  for (uint32_t e = begin; e < end; e++) {
    const uint64_t ent3 = sorted[min(e + 3, last)];
    const g1_affine pt1 = point_of(ent1, pt0);
    const uint32_t key = (uint32_t)ent0;
    if (key != top) { // zero digits add nothing
      const uint32_t b = jd.bucket_begin + (jd.stride ? 0u : (e - jd.entry_begin) >> jd.log_n) * top + key;
      if (b != cur) {
        if (cur != NONE) {
          run_end[cur] = last_e + 1;
          store_xyzz29_raw(slots + cur, empty ? xyzz29_infinity() : acc);
        }
        if (e != begin || !continued)
          run_start[b] = e;
        empty = true;
        cur = b;
        cur_key = key;
      }
      xyzz29_add_affine(acc, empty, pt0, ((uint32_t)(ent0 >> 32) & SIGN) != 0, bases + ((uint32_t)(ent0 >> 32) & ~SIGN));
      last_e = e;
    }
    ent0 = ent1;
    ent1 = ent2;
    ent2 = ent3;
    pt0 = pt1;
  }
  if (cur != NONE) {
    if (last_e + 1 != end || key_after != cur_key)
      run_end[cur] = last_e + 1;
    store_xyzz29_raw(slots + cur, empty ? xyzz29_infinity() : acc);
  }
}

// The top digit of window w: the last digit window tops out below B = 2^(c-1) (a
// fixed-base job's single bucket window takes every window's digits, up to B).
__device__ __forceinline__ uint32_t top_digit(const job_desc &jd, uint32_t w) {
  return 1u << (w == jd.W - 1 && !jd.stride ? jd.c - (jd.Wd * jd.c - 254) - 1 : jd.c - 1);
}

// Heavy buckets are reduced in chunks of HEAVY_CHUNK partial sums, one block
// per chunk: a quad of lanes (quad29.cuh) sums every HEAVY_QUADS-th sum, then a
// tree in LDS; the chunk's sum overwrites the chunk's first slot when the bucket
// has several, whose sums a second kernel adds.  There are few such
// buckets, so the additions in sequence set the time: 13 by quads, at 2.7 us
// each, where a thread per point takes 14 at 7 us (2^12 points, 512 sums: 98 -> 41 us).

// the sum of `n` points (not 0), `stride` apart, in every quad's lanes of quad 0
__device__ __forceinline__ f29 heavy_block_sum(const xyzz29 *base, uint32_t n, uint32_t stride, f29 (&sh)[HEAVY_QUADS][4]) {
  const unsigned q = threadIdx.x >> 2, l = quad_lane();
  f29 acc = f29{}; // infinity
  if (q < n)
    acc = quad_load_xyzz29(base + (size_t)q * stride);
  for (uint32_t i = q + HEAVY_QUADS; i < n; i += HEAVY_QUADS)
    acc = quad_add(acc, quad_load_xyzz29(base + (size_t)i * stride));
  unsigned half = HEAVY_QUADS / 2;
  while (half >= n && half > 0) // the upper halves hold nothing
    half >>= 1;
  for (; half > 0; half >>= 1) {
    sh[q][l] = acc;
    __syncthreads();
    if (q < half && q + half < n)
      acc = quad_add(acc, sh[q + half][l]);
    __syncthreads();
  }
  return acc;
}

// where the sum of bucket b goes: slot d of its window, or the window's top when
// d is its top digit (the bucket's digit d is at least 1)
__device__ __forceinline__ g1_xyzz *bucket_destination(const job_desc &jd, uint32_t b, g1_xyzz *A, g1_xyzz *tops) {
  const uint32_t B = 1u << (jd.c - 1);
  const uint32_t local = b - jd.bucket_begin, w = local >> (jd.c - 1), d = (local & (B - 1)) + 1;
  return d == top_digit(jd, w) ? tops + jd.top_begin + w : A + jd.bucket_begin + w * B + d;
}

// one quad: its sum to the bucket's place, added to what is there with `add`
__device__ __forceinline__ void quad_store_bucket(g1_xyzz *dst, const f29 &sum, bool add) {
  quad_store_xyzz(dst, add ? quad_add(quad_load_xyzz(dst), sum) : sum);
}

// 4a. one block per chunk of a heavy bucket, then one wave per medium bucket: a
// quad sums every 16th partial sum and the quads' sums meet in a tree over the
// wave (grid-stride over both lists by `blocks` blocks).  The chunk of a bucket
// of several goes to its first slot, every other sum to the bucket's place.
__device__ __forceinline__ void sum_listed(const job_table &jobs, xyzz29 *partials, const piece_lists &lists, const uint32_t *piece_offset,
                                           const uint32_t *piece_count, g1_xyzz *A, g1_xyzz *tops, bool add, uint32_t blocks,
                                           f29 (&sh)[HEAVY_QUADS][4]) {
  const uint32_t chunks = lists.count[1], medium = lists.count[0];
  for (uint32_t c = blockIdx.x; c < chunks; c += blocks) {
    const uint2 ch = lists.chunks[c];
    const uint32_t np = piece_count[ch.x], first = ch.y * HEAVY_CHUNK, left = np - first; // sums from the chunk start
    xyzz29 *base = partials + piece_offset[ch.x] + first;
    const f29 sum = heavy_block_sum(base, left < HEAVY_CHUNK ? left : HEAVY_CHUNK, 1, sh);
    if (threadIdx.x < 4) {
      if (np > HEAVY_CHUNK)
        quad_store_xyzz29(base, sum);
      else
        quad_store_bucket(bucket_destination(jobs.job[find_job(jobs, ch.x, by_bucket())], ch.x, A, tops), sum, add);
    }
  }
  const unsigned q = (threadIdx.x & 63) >> 2;
  for (uint32_t m = blockIdx.x * (HEAVY_BLOCK / 64) + (threadIdx.x >> 6); m < medium; m += blocks * (HEAVY_BLOCK / 64)) {
    const uint32_t b = lists.medium[m], np = piece_count[b];
    const xyzz29 *base = partials + piece_offset[b];
    f29 acc = f29{};
    if (q < np)
      acc = quad_load_xyzz29(base + q);
    for (uint32_t i = q + 16; i < np; i += 16)
      acc = quad_add(acc, quad_load_xyzz29(base + i));
    for (uint32_t off = 8; off > 0; off >>= 1)
      if (off < np) // the sums off.. of a smaller bucket are infinity
        acc = quad_add(acc, quad_from_neighbour(acc, off));
    if (q == 0)
      quad_store_bucket(bucket_destination(jobs.job[find_job(jobs, b, by_bucket())], b, A, tops), acc, add);
  }
}

// 4b. one block per heavy bucket of several chunks (grid-stride): the sum of its chunks' sums
__global__ __launch_bounds__(HEAVY_BLOCK) void heavy_final_kernel(const job_table jobs, const xyzz29 *partials, const piece_lists lists,
                                                                  const uint32_t *piece_offset, const uint32_t *piece_count, g1_xyzz *A,
                                                                  g1_xyzz *tops, bool add) {
  __shared__ f29 sh[HEAVY_QUADS][4];
  const uint32_t count = lists.count[2];
  for (uint32_t h = blockIdx.x; h < count; h += gridDim.x) {
    const uint32_t b = lists.several[h];
    const f29 sum = heavy_block_sum(partials + piece_offset[b], (piece_count[b] + HEAVY_CHUNK - 1) / HEAVY_CHUNK, HEAVY_CHUNK, sh);
    if (threadIdx.x < 4)
      quad_store_bucket(bucket_destination(jobs.job[find_job(jobs, b, by_bucket())], b, A, tops), sum, add);
  }
}

// Level-0 windows: A[bucket_begin + w*2^(c-1) + k] for k in [0, 2^(c-1)) holds
// bucket k of window w (k = 0 and the top digit hold infinity); tops[top_begin + w]
// holds the bucket of the window's top digit (2^(c-1), or 2^top_signed in the last window).
// With `add`, the buckets of this launch are added to what A and tops already
// hold (the chunks of one MSM accumulate into the same windows).
// One bucket of the gather: where its sum goes and which partial sums make
// it.  With `first`, the window's infinity stores are made here.
struct gather_item {
  g1_xyzz *dst;
  uint32_t off, np; // its partial sums
  bool live;        // false: nothing to store for this bucket
};

__device__ __forceinline__ gather_item gather_prepare(const job_table &jobs, uint32_t t, const uint32_t *__restrict__ piece_offset,
                                                      const uint32_t *__restrict__ piece_count, g1_xyzz *__restrict__ A,
                                                      g1_xyzz *__restrict__ tops, bool add, bool first) {
  const job_desc &jd = jobs.job[find_job(jobs, t, by_bucket())];
  const uint32_t B = 1u << (jd.c - 1);
  const uint32_t local = t - jd.bucket_begin, w = local >> (jd.c - 1), k = local & (B - 1);
  const uint32_t top = top_digit(jd, w);
  // slot k of a window holds bucket k; slot 0 also hands the bucket of digit B
  // to the window's top when that is its top digit, and the top digit's own
  // slot in the last window hands it there instead
  const bool to_top = k == 0 ? top == B : k == top;
  if ((k == 0 || k == top) && !add && first)
    store_xyzz(A + t, xyzz_infinity());
  gather_item g{nullptr, 0, 0, false};
  if (k == 0 && !to_top)
    return g;
  // bucket of digit d is batch bucket bucket_begin + w B + d - 1
  const uint32_t d = k == 0 ? B : k;
  const uint32_t b = jd.bucket_begin + w * B + d - 1;
  g.np = piece_count[b];
  g.off = piece_offset[b];
  g.dst = to_top ? tops + jd.top_begin + w : A + t;
  g.live = g.np <= jd.small && !(add && g.np == 0); // larger ones are stored by sum_listed; nothing of this launch to add
  return g;
}

__device__ __forceinline__ bool gather_sums(const gather_item &g) { return g.live && g.np >= 2; }

__device__ __forceinline__ void gather_finish(const gather_item &g, const xyzz29 *__restrict__ partials, bool add) {
  // the partial sums are on 29-bit limbs; the window arrays take the library's format
  xyzz29 acc = xyzz29_infinity();
  bool empty = true;
  if (g.np != 0) {
    acc = load_xyzz29(partials + g.off);
    empty = xyzz29_is_infinity(acc);
    for (uint32_t q = 1; q < g.np; q++)
      xyzz29_accumulate29(acc, empty, load_xyzz29(partials + g.off + q));
  }
  if (add)
    xyzz29_accumulate(acc, empty, load_xyzz(g.dst));
  store_xyzz29(g.dst, acc, empty);
}

// A thread per bucket.  With LIST, for launches whose buckets are much smaller
// than the accumulation chunks (2^24 at c = 20: one bucket in six spans two
// chunks), a thread copies a bucket of at most one partial sum at once and, in
// a wave where few buckets have more, lists those in LDS; the block's threads
// then sum the listed buckets, one per thread, so the additions run in waves
// whose lanes all add (0.84 -> 0.63 ms): with a bucket per lane throughout,
// almost every wave made 63 lanes wait for one lane's addition.  Where most
// buckets span several chunks (2^24 at c = 17) the list saves nothing and its
// block barriers keep finished waves resident (0.26 -> 0.29 ms), so such
// launches sum every bucket in place.
constexpr unsigned GATHER_LIST_MAX_LANES = 16; // a wave lists when at most this many of its lanes add

// The first `listed_blocks` blocks sum the listed buckets: these take a wave or
// a block for 50 us of additions in sequence, which as a launch of their own
// before the gather left the GPU nearly idle.  Both launches and this one: 67 +
// 168 -> 189 us at 2^20 points, 61 + 242 -> 245 us for 24 MSMs of 2^12..2^17, 51 +
// 23 -> 58 us at 2^12, 95 + 530 -> 590 us at 2^24.
template <bool LIST>
__global__ __launch_bounds__(MSM_BLOCK) void bucket_gather_kernel(const job_table jobs, uint32_t nb, xyzz29 *partials, const piece_lists lists,
                                                                  const uint32_t *__restrict__ piece_offset,
                                                                  const uint32_t *__restrict__ piece_count, g1_xyzz *__restrict__ A,
                                                                  g1_xyzz *__restrict__ tops, bool add, uint32_t listed_blocks) {
  __shared__ f29 sh[HEAVY_QUADS][4];
  if (blockIdx.x < listed_blocks) {
    sum_listed(jobs, partials, lists, piece_offset, piece_count, A, tops, add, listed_blocks, sh);
    return;
  }
  const uint32_t t = (blockIdx.x - listed_blocks) * MSM_BLOCK + threadIdx.x;
  if (!LIST) {
    if (t < nb) {
      const gather_item g = gather_prepare(jobs, t, piece_offset, piece_count, A, tops, add, true);
      if (g.live)
        gather_finish(g, partials, add);
    }
    return;
  }
  __shared__ uint32_t list[MSM_BLOCK];
  __shared__ uint32_t listed;
  if (threadIdx.x == 0)
    listed = 0;
  __syncthreads();
  gather_item g{nullptr, 0, 0, false};
  if (t < nb)
    g = gather_prepare(jobs, t, piece_offset, piece_count, A, tops, add, true);
  const bool sums = gather_sums(g);
  const bool in_place = __popcll(__ballot(sums)) > GATHER_LIST_MAX_LANES;
  if (g.live && (!sums || in_place))
    gather_finish(g, partials, add);
  else if (sums)
    list[atomicAdd(&listed, 1u)] = t;
  __syncthreads();
  if (threadIdx.x < listed)
    gather_finish(gather_prepare(jobs, list[threadIdx.x], piece_offset, piece_count, A, tops, add, false), partials, add);
}

// 5. one split level for every job whose windows are still wider than one bit.
// Segment: X windows of width s at A -> 2X windows of width t = ceil(s/2) at out;
// lo[u] = sum_v A[v*2^t + u] (2^hs terms), hi[v] = sum_u A[v*2^t + u] (2^t terms).
// Output part p holds the terms == p (mod D_lo) of lo and (mod D) of hi, with
// D = D_lo * 2^(t-hs), so every thread sums about the same number of terms.
struct split_seg {
  const g1_xyzz *A;
  g1_xyzz *out;
  uint32_t X, s, D_lo, D;
  uint32_t thread_begin;
};

struct split_table {
  uint32_t count;
  split_seg seg[MSM_MAX_JOBS];
};

template <class Table> __device__ __forceinline__ unsigned find_seg(const Table &t, uint32_t v) {
  unsigned lo = 0, hi = t.count;
  while (hi - lo > 1) {
    const unsigned mid = (lo + hi) >> 1;
    if (t.seg[mid].thread_begin <= v)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// PREFETCH: the next term is loaded before the current one is added (64 more
// VGPRs: two waves per SIMD instead of three).  It pays when the launch is too
// small to fill the GPU (2^24 at c = 17: 123 K threads, 0.27 -> 0.20 ms) and
// costs when it is large (2^24 at c = 20: 1.7 M threads, 1.44 -> 1.50 ms).
constexpr uint32_t SPLIT_PREFETCH_BELOW = 1u << 19;

template <bool PREFETCH> __global__ __launch_bounds__(ACC_BLOCK) void split_kernel(const split_table segs, uint32_t total) {
  const uint32_t id_all = blockIdx.x * blockDim.x + threadIdx.x;
  if (id_all >= total)
    return;
  const split_seg &sg = segs.seg[find_seg(segs, id_all)];
  const uint32_t id = id_all - sg.thread_begin;
  const unsigned s = sg.s, t = (s + 1) >> 1, hs = s - t;
  const uint32_t per_part = (2 * sg.X) << t;
  uint32_t part = id / per_part;
  const uint32_t rem = id % per_part;
  uint32_t j = rem & ((1u << t) - 1), x = rem >> (t + 1);
  const uint32_t half = (rem >> t) & 1;
  if (half) {
    // Half-1 sums run along a row (consecutive u); the threads of this half
    // are renumbered so that neighbouring lanes take neighbouring parts of
    // one row and their loads are contiguous: (part, x, j) -> L -> (x, j, part)
    // with part fastest.  D is a power of two.
    const uint32_t log_d = __builtin_ctz(sg.D);
    const uint32_t L = ((part * sg.X + x) << t) + j;
    part = L & (sg.D - 1);
    j = (L >> log_d) & ((1u << t) - 1);
    x = L >> (log_d + t);
  }
  const g1_xyzz *src = sg.A + ((size_t)x << s);
  // terms q = first, first + step, ... < limit at src[(q << t) | j] (low half)
  // or src[(j << t) | q] (high half)
  const bool lo = half == 0;
  const uint32_t first = part, step = lo ? sg.D_lo : sg.D, limit = lo ? (1u << hs) : (1u << t);
  const bool active = lo ? part < sg.D_lo : j < (1u << hs);
  auto term = [&](uint32_t q) { return src + (lo ? ((q << t) | j) : ((j << t) | q)); };
  // the sum in the 29-bit-limb radix; `empty` marks infinity
  xyzz29 acc;
  bool empty = true;
  if (active && first < limit) {
    xyzz29_accumulate(acc, empty, load_xyzz(term(first)));
    if (PREFETCH) {
      uint32_t q = first + step;
      if (q < limit) {
        g1_xyzz cur = load_xyzz(term(q));
        for (q += step; q < limit; q += step) {
          const g1_xyzz next = load_xyzz(term(q));
          xyzz29_accumulate(acc, empty, cur);
          cur = next;
        }
        xyzz29_accumulate(acc, empty, cur);
      }
    } else {
      for (uint32_t q = first + step; q < limit; q += step)
        xyzz29_accumulate(acc, empty, load_xyzz(term(q)));
    }
  }
  store_xyzz29(sg.out + (size_t)part * per_part + ((2 * x + half) << t) + j, acc, empty);
}

// out[i] += out[i + half] for i < half, per segment, while that is
// FOLD_THREADS_MIN additions or more; quads take over below, FOLD_QUADS_MAX of
// them (a wave per SIMD) where the parts allow.
constexpr uint64_t FOLD_THREADS_MIN = 1u << 17;
constexpr uint32_t FOLD_QUADS_MAX = 1u << 14;

struct fold_seg {
  g1_xyzz *out;
  uint32_t half;
  uint32_t thread_begin;
};

struct fold_table {
  uint32_t count;
  fold_seg seg[MSM_MAX_JOBS];
};

__global__ __launch_bounds__(ACC_BLOCK) void fold_kernel(const fold_table segs, uint32_t total) {
  const uint32_t id_all = blockIdx.x * blockDim.x + threadIdx.x;
  if (id_all >= total)
    return;
  const fold_seg &sg = segs.seg[find_seg(segs, id_all)];
  const uint32_t i = id_all - sg.thread_begin;
  // the sum on 29-bit limbs, as in the split kernel
  xyzz29 acc;
  bool empty = true;
  xyzz29_accumulate(acc, empty, load_xyzz(sg.out + i));
  xyzz29_accumulate(acc, empty, load_xyzz(sg.out + i + sg.half));
  store_xyzz29(sg.out + i, acc, empty);
}

// The rest of a level's parts, by quads of lanes (quad29.cuh): Q quads share an
// output, a quad adds every Q-th of its D parts, then the quads' sums meet in a
// tree over the wave.  A level's fold has few outputs (2816 at 2^12 points), so
// additions in sequence set its time: one launch of D / Q + log2 Q additions by
// quads, at 2.7 us, replaces log2 D launches of one at 7 us each.
struct quad_fold_seg {
  g1_xyzz *out;
  uint32_t outputs, D, Q;
  uint32_t thread_begin; // a multiple of 64
};

struct quad_fold_table {
  uint32_t count;
  quad_fold_seg seg[MSM_MAX_JOBS];
};

__global__ __launch_bounds__(ACC_BLOCK) void quad_fold_kernel(const quad_fold_table segs) {
  const uint32_t id_all = blockIdx.x * ACC_BLOCK + threadIdx.x;
  const quad_fold_seg &sg = segs.seg[find_seg(segs, id_all)];
  const uint32_t quad = (id_all - sg.thread_begin) >> 2;
  const uint32_t i = quad / sg.Q, q = quad % sg.Q;
  if (i >= sg.outputs)
    return; // padding; a wave serves one segment, an output's quads leave together
  f29 acc = quad_load_xyzz(sg.out + (size_t)q * sg.outputs + i);
  for (uint32_t part = q + sg.Q; part < sg.D; part += sg.Q)
    acc = quad_add(acc, quad_load_xyzz(sg.out + (size_t)part * sg.outputs + i));
  for (uint32_t off = sg.Q >> 1; off > 0; off >>= 1)
    acc = quad_add(acc, quad_from_neighbour(acc, off));
  if (q == 0)
    quad_store_xyzz(sg.out + i, acc);
}

// A whole split level by quads, for small levels: Q quads share an output sum
// (Q << (t - hs) in the high half, whose sums are longer), a quad adds every Q-th
// term, and the quads' sums meet in a tree over the wave, so the level needs no
// parts and no folds.  A thread per part adds in half the SIMD time, a quad in
// under half the latency: at 2^12 points (90 K terms) 34 us against 51 us for
// parts and their fold, at 2^18 (557 K terms) 167 us against 115 us.
constexpr uint64_t QUAD_SPLIT_TERMS = 1u << 18; // levels of fewer terms
struct quad_split_seg {
  const g1_xyzz *A;
  g1_xyzz *out;
  uint32_t X, s, Q;
  uint32_t thread_begin; // a multiple of 64
};

struct quad_split_table {
  uint32_t count;
  quad_split_seg seg[MSM_MAX_JOBS];
};

__global__ __launch_bounds__(ACC_BLOCK) void quad_split_kernel(const quad_split_table segs) {
  const uint32_t id_all = blockIdx.x * ACC_BLOCK + threadIdx.x;
  const quad_split_seg &sg = segs.seg[find_seg(segs, id_all)];
  const unsigned s = sg.s, t = (s + 1) >> 1, hs = s - t;
  // a window's half takes Q << t quads (a multiple of 16: a wave has one half)
  const uint32_t quad = (id_all - sg.thread_begin) >> 2, per_half = sg.Q << t;
  const uint32_t x = quad / (2 * per_half), half = (quad / per_half) & 1, in_half = quad % per_half;
  const uint32_t Q = half ? sg.Q << (t - hs) : sg.Q, j = in_half / Q, q = in_half % Q;
  const g1_xyzz *src = sg.A + ((size_t)x << s);
  // terms q, q + Q, ... at src[(term << t) | j] (low half, 2^hs of them) or src[(j << t) | term] (high half, 2^t)
  const uint32_t terms = half ? 1u << t : 1u << hs;
  auto term = [&](uint32_t i) { return src + (half ? (j << t) | i : (i << t) | j); };
  f29 acc = quad_load_xyzz(term(q));
  for (uint32_t i = q + Q; i < terms; i += Q)
    acc = quad_add(acc, quad_load_xyzz(term(i)));
  for (uint32_t off = Q >> 1; off > 0; off >>= 1)
    acc = quad_add(acc, quad_from_neighbour(acc, off));
  if (q == 0) {
    g1_xyzz *out = sg.out + ((size_t)(2 * x + half) << t) + j;
    quad_store_xyzz(out, acc);
    if (half && hs < t) // the high child has one bit less: its upper half is infinity
      quad_store_xyzz(out + (1u << hs), f29{});
  }
}

// Windows of s <= BITS_WIDTH bits, a block each, down to their per-bit sums:
// bits[x s + j] = the sum of the points of window x whose index has bit j set.
// In round r the lists of 2^(s - r) points at offsets 0 and 2^j, j >= s - r, are
// halved, L[i] += L[i + half]; the upper half of the list at 0 becomes the list
// at 2^(s - r - 1), the sum of bit s - r - 1.  About 2 2^s additions by quads, in
// s rounds of one LDS barrier, replace the splits and folds of the last three
// levels (nine launches).
constexpr unsigned BITS_WIDTH = 8;
constexpr unsigned BITS_BLOCK = 256, BITS_QUADS = BITS_BLOCK / 4;

struct bits_seg {
  const g1_xyzz *A;
  g1_xyzz *bits;
  uint32_t s;
  uint32_t thread_begin; // first window (block) of the job
};

struct bits_table {
  uint32_t count;
  bits_seg seg[MSM_MAX_JOBS];
};

__global__ __launch_bounds__(BITS_BLOCK) void bits_kernel(const bits_table segs) {
  __shared__ f29 pts[1u << BITS_WIDTH][4];
  const bits_seg &sg = segs.seg[find_seg(segs, blockIdx.x)];
  const uint32_t x = blockIdx.x - sg.thread_begin, s = sg.s;
  const unsigned quad = threadIdx.x >> 2, l = quad_lane();
  for (uint32_t i = quad; i < (1u << s); i += BITS_QUADS)
    pts[i][l] = quad_load_xyzz(sg.A + ((size_t)x << s) + i);
  __syncthreads();
  for (uint32_t r = 0; r < s; r++) {
    const uint32_t log_half = s - 1 - r;
    for (uint32_t k = quad; k < ((r + 1) << log_half); k += BITS_QUADS) {
      const uint32_t list = k >> log_half, i = k & ((1u << log_half) - 1);
      const uint32_t at = (list == 0 ? 0u : 1u << (s - list)) + i;
      pts[at][l] = quad_add(pts[at][l], pts[at + (1u << log_half)][l]);
    }
    __syncthreads();
  }
  if (quad < s)
    quad_store_xyzz(sg.bits + (size_t)x * s + quad, pts[1u << quad][l]);
}

// 6. bit i = w*c + j of a job is its window's top bucket (j == c-1 or i == 253),
// else the bit's sum in the window reached by following the splits: a width-s
// window x holds bits [0, t) in child 2x and [t, s) in child 2x+1, t = ceil(s/2),
// down to the BITS_WIDTH bits whose sums bits_kernel left.
// A job over a fixed-base table has one window: bits [0, c) as above, the
// bits above are infinity (its fold is the same point).
struct result_desc {
  const g1_xyzz *bits;
  const g1_xyzz *tops;
  g1_jacobian *out;
  uint32_t c;
  uint32_t single; // one bucket window (fixed-base table)
};

struct result_table {
  uint32_t count;
  result_desc job[MSM_MAX_JOBS];
};

__global__ void result_kernel(const result_table jobs) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 254 * jobs.count)
    return;
  const result_desc &rd = jobs.job[t / 254];
  const uint32_t i = t % 254, c = rd.c;
  if (rd.single && i >= c) {
    store_fe(&rd.out[i].x, fe_zero());
    store_fe(&rd.out[i].y, fe_one<Fq>());
    store_fe(&rd.out[i].z, fe_zero());
    return;
  }
  const uint32_t w = i / c;
  uint32_t j = i % c;
  g1_xyzz v;
  if (j == c - 1 || (i == 253 && !rd.single)) {
    v = load_xyzz(rd.tops + w);
  } else {
    uint32_t x = w, s = c - 1;
    while (s > BITS_WIDTH) {
      const uint32_t half = (s + 1) >> 1;
      if (j < half) {
        x = 2 * x;
      } else {
        x = 2 * x + 1;
        j -= half;
      }
      s = half;
    }
    v = load_xyzz(rd.bits + (size_t)x * s + j);
  }
  const g1_jacobian r = xyzz_to_jacobian(v);
  store_fe(&rd.out[i].x, r.x);
  store_fe(&rd.out[i].y, r.y);
  store_fe(&rd.out[i].z, r.z);
}

} // namespace

namespace {

// Both are functions of the job alone, so a job's sums are the same alone and in
// any batch.
//
// Parts D_lo of the low half of a split level (X windows of `width` bits): each
// split thread adds 2^hs / D_lo terms: 16 where that leaves SPLIT_THREADS
// threads, else 8 (2^20 points: 187 -> 109 us of splits for 28 us more of folds;
// at 2^18 four terms cost 49 us more of folds than they save of splits).
uint32_t split_parts(uint32_t X, unsigned width) {
  const unsigned hs = width - (width + 1) / 2;
  const uint64_t level_terms = (uint64_t)(2 * X) << width;
  const unsigned terms = level_terms / 16 >= SPLIT_THREADS ? 16 : 8;
  return (1u << hs) > terms ? (1u << hs) / terms : 1u;
}

bool split_by_quads(uint32_t X, unsigned width) { return (uint64_t)(2 * X) << width < QUAD_SPLIT_TERMS; }

// Quads per low-half sum of such a level: up to a wave per SIMD, and no more
// than 4, whose tree is a small part of the additions.
uint32_t split_quads(uint32_t X, unsigned width) {
  uint32_t Q = 1;
  while (Q < 4 && ((uint64_t)(2 * X) * 2 * Q << ((width + 1) / 2)) <= FOLD_QUADS_MAX)
    Q *= 2;
  return Q;
}

} // namespace

// Points (of 128 bytes) the reduction of one job's windows keeps: the windows
// (in parts) of every split level and the per-bit sums.
uint64_t msm_split_points(unsigned c, unsigned windows) {
  uint64_t total = 0;
  uint32_t X = windows;
  unsigned width = c - 1;
  for (; width > BITS_WIDTH; width = (width + 1) / 2, X *= 2) {
    const unsigned t = (width + 1) / 2, hs = width - t;
    const uint64_t D = split_by_quads(X, width) ? 1 : (uint64_t)split_parts(X, width) << (t - hs);
    total += D * (2 * (uint64_t)X << t);
  }
  return total + (uint64_t)X * width;
}

namespace {

// Per-launch job table and totals of a batch (window buckets, top slots, ...).
struct batch_layout {
  job_table jt{};
  uint64_t entries = 0, nb = 0, chunks = 0, slots = 0;
  uint32_t tops_total = 0, max_np = 0;
};

hipError_t layout_batch(const msm_job *jobs, unsigned count, batch_layout *out) {
  if (count == 0 || count > MSM_MAX_JOBS)
    return hipErrorInvalidValue;
  batch_layout &bl = *out;
  job_table &jt = bl.jt;
  jt.count = count;
  uint64_t entries = 0, nb64 = 0, chunks = 0, slots = 0;
  uint32_t tops_total = 0, max_np = 0;
  for (unsigned j = 0; j < count; j++) {
    const unsigned c = jobs[j].c;
    if (c < 3 || c > 24 || jobs[j].log_n > 28 || jobs[j].piece == 0 || jobs[j].piece > MSM_MAX_PIECE || !jobs[j].bases || !jobs[j].scalars ||
        !jobs[j].results)
      return hipErrorInvalidValue;
    // a fixed-base table holds ceil(254 / c) blocks of `stride` >= 2^log_n
    // points, indexed below 2^31 (the entry's top bit is the sign)
    const uint64_t wd = (254 - 1) / c + 1;
    if (jobs[j].stride && (jobs[j].stride < (1ull << jobs[j].log_n) || wd * jobs[j].stride >= (1ull << 31)))
      return hipErrorInvalidValue;
    job_desc &d = jt.job[j];
    const uint32_t n = 1u << jobs[j].log_n;
    d.bases = jobs[j].bases;
    d.scalars = jobs[j].scalars;
    d.log_n = (uint8_t)jobs[j].log_n;
    d.c = (uint8_t)c;
    d.Wd = (uint8_t)wd;
    d.W = jobs[j].stride ? 1 : d.Wd;
    d.stride = jobs[j].stride;
    d.piece = (uint16_t)jobs[j].piece;
    d.small = small_pieces(d);
    if (entries + (uint64_t)d.Wd * n >= (1ull << 31))
      return hipErrorInvalidValue;
    d.entry_begin = (uint32_t)entries;
    d.bucket_begin = (uint32_t)nb64;
    d.top_begin = tops_total;
    d.chunk_begin = (uint32_t)chunks;
    d.slot_begin = (uint32_t)slots;
    const uint64_t job_chunks = ((uint64_t)d.Wd * n + d.piece - 1) / d.piece, job_buckets = (uint64_t)d.W << (c - 1);
    entries += (uint64_t)d.Wd * n;
    nb64 += job_buckets;
    tops_total += d.W;
    chunks += job_chunks;
    slots += job_buckets + job_chunks; // slot(b, k) <= (buckets - 1) + (chunks - 1)
    // a bucket holds at most n entries, or Wd n in a fixed-base job's single window
    const uint64_t bucket_max = (uint64_t)(d.stride ? d.Wd : 1u) * n;
    max_np = std::max<uint32_t>(max_np, (uint32_t)((bucket_max + d.piece - 1) / d.piece + 1));
  }
  if (entries >= (1ull << 31) || nb64 >= (1ull << 31) || slots >= (1ull << 32))
    return hipErrorInvalidValue;
  bl.entries = entries;
  bl.nb = nb64;
  bl.chunks = chunks;
  bl.slots = slots;
  bl.tops_total = tops_total;
  bl.max_np = max_np;
  return hipSuccess;
}

// Steps 1-4 for every job of the layout: the jobs' points are sorted into
// buckets, summed, and stored (or, with `add`, added) into the level-0 window
// array A (bl.nb buckets) and the top-digit slots `tops` (bl.tops_total).
// Every temporary it takes from `ar` is returned before it ends.
hipError_t accumulate_phase(batch_layout &bl, unsigned count, arena &ar, g1_xyzz *A, g1_xyzz *tops, bool add) {
  hipStream_t s = ar.stream();
  job_table &jt = bl.jt;
  const uint64_t entries = bl.entries, chunks = bl.chunks, slots = bl.slots;
  const uint32_t nb = (uint32_t)bl.nb, max_np = bl.max_np;

  // 1-2. digits, sort, bucket runs
  uint32_t *offsets = nullptr, *counts = nullptr;
  uint64_t *sorted = nullptr; // (key, point reference) pairs, sorted by key within each window
  // offsets, counts and the lists' lengths are cleared together
  BC_TRY(ar.get(&offsets, 2 * (uint64_t)nb + 3));
  counts = offsets + nb;
  BC_TRY(ar.get(&sorted, entries));
  {
    uint64_t *digits = nullptr;
    BC_TRY(ar.get(&digits, entries));
    seg_group groups[MSM_MAX_JOBS];
    unsigned key_bits = 0; // local keys are <= 2^(c-1)
    bool unaligned = false; // a fixed-base job whose windows are not whole sort tiles
    for (unsigned j = 0; j < count; j++) {
      // a sort segment per window, or one over all of a fixed-base job's entries
      const job_desc &d = jt.job[j];
      groups[j] = d.stride ? seg_group{d.entry_begin, (uint32_t)d.Wd << d.log_n, 1u} : seg_group{d.entry_begin, 1u << d.log_n, d.W};
      key_bits = std::max<unsigned>(key_bits, d.c);
      unaligned |= d.stride != 0 && (1u << d.log_n) < SEG_TILE;
    }
    // the digits kernel counts the sort's first digit when its per-window
    // counters fit DIGITS_MAX_LDS; otherwise the sort counts them itself
    seg_first_pass fp;
    BC_TRY(segmented_sort_first_pass(groups, count, key_bits, &fp));
    size_t lds = 0; // 16-bit counters per digit window, two per word
    for (unsigned j = 0; j < count; j++)
      lds = std::max(lds, sizeof(uint32_t) * ((((size_t)jt.job[j].Wd << std::min<unsigned>(jt.job[j].c, fp.bits)) + 1) / 2));
    uint32_t *first_table = nullptr;
    // (the digits kernel counts per window tile: a fixed-base job's single
    // segment qualifies when its windows are whole tiles)
    uint64_t tiles = 0;
    for (unsigned j = 0; j < count; j++)
      tiles += ((1u << jt.job[j].log_n) + SEG_TILE - 1) / SEG_TILE;
    if (fp.bits > 0 && lds <= DIGITS_MAX_LDS && fp.table_entries < (1ull << 32) && !unaligned && tiles >= DIGITS_MIN_TILES) {
      BC_TRY(ar.get(&first_table, fp.table_entries));
      for (unsigned j = 0; j < count; j++)
        jt.job[j].table_begin = (uint32_t)fp.table_begin[j];
    }
    const uint32_t block_points = first_table ? SEG_TILE : MSM_BLOCK;
    uint32_t blocks = 0;
    for (unsigned j = 0; j < count; j++) {
      jt.job[j].digit_block = blocks;
      blocks += ((1u << jt.job[j].log_n) + block_points - 1) / block_points;
    }
    digits_kernel<<<blocks, first_table ? DIGITS_BLOCK : MSM_BLOCK, first_table ? lds : 0, s>>>(jt, digits, first_table, fp.bits, block_points);
    BC_LAUNCH_CHECK();
    BC_TRY(segmented_sort_kv(digits, sorted, groups, count, key_bits, ar, first_table));
    if (first_table)
      BC_TRY(ar.put(first_table));
    BC_TRY(ar.put(digits));
  }

  // 3. accumulation over chunks of the sorted entries, which also records each
  // bucket's run [offsets[b], counts[b]) (empty buckets keep [0, 0))
  uint32_t *piece_count = nullptr, *piece_offset = nullptr;
  piece_lists lists{counts + nb, nullptr, nullptr, nullptr};
  xyzz29 *partials = nullptr; // on 29-bit limbs, 144 B each
  BC_TRY(ar.get(&piece_count, nb));
  BC_TRY(ar.get(&piece_offset, nb));
  BC_TRY(ar.get(&partials, slots));
  // a chunk has more than MEDIUM_PIECES of the sums, a bucket of several HEAVY_CHUNK
  BC_TRY(ar.get(&lists.medium, nb));
  BC_TRY(ar.get(&lists.chunks, slots / MEDIUM_PIECES + 1));
  BC_TRY(ar.get(&lists.several, slots / HEAVY_CHUNK + 1));
  BC_TRY(fill_u32(offsets, 2 * (uint64_t)nb + 3, 0, s));
  accumulate_kernel<<<grid_for(chunks, ACC_BLOCK), ACC_BLOCK, 0, s>>>(jt, sorted, (uint32_t)chunks, partials, offsets, counts);
  BC_LAUNCH_CHECK();
  bucket_slots_kernel<<<grid_for(nb, MSM_BLOCK), MSM_BLOCK, 0, s>>>(jt, offsets, counts, piece_offset, piece_count, nb, lists);
  BC_LAUNCH_CHECK();

  // 4. the buckets' sums into the level-0 windows; where none has more than 4
  // partial sums, none is listed
  const uint32_t listed_blocks = max_np > 4 ? LISTED_BLOCKS : 0;
  const uint32_t gather_blocks = listed_blocks + grid_for(nb, MSM_BLOCK);
  // the listing gather when most buckets lie in jobs whose buckets average at
  // most a quarter of a chunk
  uint64_t small_buckets = 0;
  for (unsigned j = 0; j < count; j++) {
    const job_desc &d = jt.job[j];
    const uint64_t job_buckets = (uint64_t)d.W << (d.c - 1);
    const uint64_t entries_per_bucket = ((uint64_t)(d.stride ? d.Wd : 1u) << d.log_n) >> (d.c - 1);
    if (4 * entries_per_bucket <= d.piece)
      small_buckets += job_buckets;
  }
  if (2 * small_buckets >= nb)
    bucket_gather_kernel<true>
        <<<gather_blocks, MSM_BLOCK, 0, s>>>(jt, nb, partials, lists, piece_offset, piece_count, A, tops, add, listed_blocks);
  else
    bucket_gather_kernel<false>
        <<<gather_blocks, MSM_BLOCK, 0, s>>>(jt, nb, partials, lists, piece_offset, piece_count, A, tops, add, listed_blocks);
  BC_LAUNCH_CHECK();
  if (max_np > HEAVY_CHUNK) {
    heavy_final_kernel<<<256, HEAVY_BLOCK, 0, s>>>(jt, partials, lists, piece_offset, piece_count, A, tops, add);
    BC_LAUNCH_CHECK();
  }
  for (void *p : {(void *)lists.several, (void *)lists.chunks, (void *)lists.medium})
    BC_TRY(ar.put(p));
  for (void *p : {(void *)partials, (void *)piece_offset, (void *)piece_count, (void *)sorted, (void *)offsets})
    BC_TRY(ar.put(p));
  return hipSuccess;
}

// Steps 5-6: the per-bit results of every job from its windows in A and tops.
hipError_t reduce_phase(const batch_layout &bl, const msm_job *jobs, unsigned count, arena &ar, g1_xyzz *A, g1_xyzz *tops) {
  hipStream_t s = ar.stream();
  const job_table &jt = bl.jt;
  // 5. split levels, all jobs together
  std::vector<g1_xyzz *> cur(count), level_buffers;
  std::vector<uint32_t> width(count), X(count);
  for (unsigned j = 0; j < count; j++) {
    cur[j] = A + jt.job[j].bucket_begin;
    width[j] = jt.job[j].c - 1;
    X[j] = jt.job[j].W;
  }
  for (;;) {
    split_table st{};
    quad_split_table qs{};
    std::vector<uint32_t> per_part, parts;
    uint64_t points = 0, threads = 0, quad_threads = 0;
    unsigned wide = 0;
    for (unsigned j = 0; j < count; j++) {
      if (width[j] <= BITS_WIDTH)
        continue;
      wide++;
      const unsigned t = (width[j] + 1) / 2, hs = width[j] - t;
      const uint32_t sums = (2 * X[j]) << t;
      if (split_by_quads(X[j], width[j])) {
        const uint32_t Q = split_quads(X[j], width[j]);
        qs.seg[qs.count++] = {cur[j], nullptr, X[j], width[j], Q, (uint32_t)quad_threads};
        quad_threads += 4ull * Q * sums;
        points += sums;
      } else {
        const uint32_t D_lo = split_parts(X[j], width[j]), D = D_lo << (t - hs);
        st.seg[st.count++] = {cur[j], nullptr, X[j], width[j], D_lo, D, (uint32_t)threads};
        per_part.push_back(sums);
        parts.push_back(D);
        threads += (uint64_t)D * sums;
        points += (uint64_t)D * sums;
      }
    }
    if (wide == 0)
      break;
    if (threads >= (1ull << 32) || quad_threads >= (1ull << 32))
      return hipErrorInvalidValue;
    g1_xyzz *next = nullptr;
    BC_TRY(ar.get(&next, points));
    level_buffers.push_back(next);
    for (unsigned j = 0, k = 0, q = 0; j < count; j++) {
      if (width[j] <= BITS_WIDTH)
        continue;
      const unsigned t = (width[j] + 1) / 2;
      const uint32_t sums = (2 * X[j]) << t;
      const bool quads = split_by_quads(X[j], width[j]);
      cur[j] = next;
      if (quads)
        qs.seg[q++].out = next;
      else
        st.seg[k].out = next;
      next += quads ? sums : (uint64_t)sums * st.seg[k++].D;
      X[j] *= 2;
      width[j] = t;
    }
    if (qs.count) {
      quad_split_kernel<<<(unsigned)(quad_threads / ACC_BLOCK), ACC_BLOCK, 0, s>>>(qs);
      BC_LAUNCH_CHECK();
    }
    if (st.count == 0)
      continue;
    if (threads < SPLIT_PREFETCH_BELOW)
      split_kernel<true><<<grid_for(threads, ACC_BLOCK), ACC_BLOCK, 0, s>>>(st, (uint32_t)threads);
    else
      split_kernel<false><<<grid_for(threads, ACC_BLOCK), ACC_BLOCK, 0, s>>>(st, (uint32_t)threads);
    BC_LAUNCH_CHECK();
    // rounds that halve the parts, a thread per sum, while they fill the GPU
    // (again a rule on the job alone), then quads
    for (;;) {
      fold_table ft{};
      uint32_t fthreads = 0;
      for (unsigned k = 0; k < st.count; k++) {
        const uint64_t half = (uint64_t)(parts[k] / 2) * per_part[k];
        if (half < FOLD_THREADS_MIN)
          continue;
        fold_seg &fs = ft.seg[ft.count++];
        fs.out = st.seg[k].out;
        fs.half = (uint32_t)half;
        fs.thread_begin = fthreads;
        fthreads += fs.half;
        parts[k] /= 2;
      }
      if (ft.count == 0)
        break;
      fold_kernel<<<grid_for(fthreads, ACC_BLOCK), ACC_BLOCK, 0, s>>>(ft, fthreads);
      BC_LAUNCH_CHECK();
    }
    quad_fold_table qt{};
    uint32_t qthreads = 0;
    for (unsigned k = 0; k < st.count; k++) {
      if (parts[k] < 2)
        continue;
      quad_fold_seg &qf = qt.seg[qt.count++];
      qf.out = st.seg[k].out;
      qf.outputs = per_part[k];
      qf.D = parts[k];
      qf.Q = 1;
      while (qf.Q < 8 && 2 * qf.Q < qf.D && 2 * qf.Q * qf.outputs <= FOLD_QUADS_MAX)
        qf.Q *= 2;
      qf.thread_begin = qthreads;
      qthreads += (4 * qf.Q * qf.outputs + 63) & ~63u;
    }
    if (qt.count) {
      quad_fold_kernel<<<qthreads / ACC_BLOCK, ACC_BLOCK, 0, s>>>(qt);
      BC_LAUNCH_CHECK();
    }
  }

  bits_table bt{};
  uint32_t windows = 0;
  uint64_t sums = 0;
  for (unsigned j = 0; j < count; j++)
    sums += (uint64_t)X[j] * width[j];
  g1_xyzz *bits = nullptr;
  BC_TRY(ar.get(&bits, sums));
  level_buffers.push_back(bits);
  bt.count = count;
  for (unsigned j = 0; j < count; j++) {
    bt.seg[j] = {cur[j], bits, width[j], windows};
    cur[j] = bits;
    bits += X[j] * width[j];
    windows += X[j];
  }
  bits_kernel<<<windows, BITS_BLOCK, 0, s>>>(bt);
  BC_LAUNCH_CHECK();

  // 6. results
  result_table rt{};
  rt.count = count;
  for (unsigned j = 0; j < count; j++)
    rt.job[j] = {cur[j], tops + jt.job[j].top_begin, jobs[j].results, jt.job[j].c, jt.job[j].stride ? 1u : 0u};
  result_kernel<<<grid_for(254 * count, 256), 256, 0, s>>>(rt);
  BC_LAUNCH_CHECK();
  while (!level_buffers.empty()) {
    BC_TRY(ar.put(level_buffers.back()));
    level_buffers.pop_back();
  }
  return hipSuccess;
}

} // namespace

namespace {

// Fixed-base table: thread i writes [2^(c w)] P_i for every window w, by c
// doublings from the window before and one inversion per entry.
__global__ __launch_bounds__(MSM_BLOCK) void fixed_base_kernel(const g1_affine *bases, uint32_t n, unsigned c, unsigned windows, g1_affine *table) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  const g1_affine p = load_affine(bases + i);
  store_fe(&table[i].x, p.x);
  store_fe(&table[i].y, p.y);
  g1_xyzz acc = xyzz_from_affine(p);
  for (unsigned w = 1; w < windows; w++) {
    for (unsigned k = 0; k < c; k++)
      acc = xyzz_dbl(acc);
    const g1_affine a = xyzz_to_affine(acc);
    g1_affine *dst = table + (size_t)w * n + i;
    store_fe(&dst->x, a.x);
    store_fe(&dst->y, a.y);
  }
}

} // namespace

hipError_t msm_fixed_base_table(const g1_affine *bases, unsigned log_n, unsigned c, g1_affine *table, hipStream_t s) {
  const uint64_t windows = (254 - 1) / (c ? c : 1) + 1;
  if (!bases || !table || c < 3 || c > 24 || log_n > 28 || (windows << log_n) >= (1ull << 31))
    return hipErrorInvalidValue;
  const uint32_t n = 1u << log_n;
  fixed_base_kernel<<<grid_for(n, MSM_BLOCK), MSM_BLOCK, 0, s>>>(bases, n, c, (unsigned)windows, table);
  return hipGetLastError();
}

hipError_t msm_batch_device(const msm_job *jobs, unsigned count, arena &ar) {
  if (count == 0)
    return hipSuccess;
  batch_layout bl;
  BC_TRY(layout_batch(jobs, count, &bl));
  // the windows are taken first: they outlive every temporary of the accumulation
  g1_xyzz *A = nullptr, *tops = nullptr;
  BC_TRY(ar.get(&A, bl.nb));
  BC_TRY(ar.get(&tops, bl.tops_total));
  BC_TRY(accumulate_phase(bl, count, ar, A, tops, false));
  BC_TRY(reduce_phase(bl, jobs, count, ar, A, tops));
  BC_TRY(ar.put(tops));
  BC_TRY(ar.put(A));
  return hipSuccess;
}

namespace {

// Host inputs are copied in chunks: chunk k+1 moves over PCIe while chunk k is
// accumulated (src/msm.cu:160-195 copies growing chunks on side streams for the
// same purpose).  Every chunk pays for the sort and the bucket sums again, so
// chunks pay once the copy they hide is longer: pinned scalars in one, two and
// four chunks take 0.91 / 1.05 / 1.60 ms at 2^18, 2.29 / 2.23 / 2.64 at 2^20,
// 4.17 / 3.70 / 4.02 at 2^21, 7.79 / 6.78 / 6.53 at 2^22.
unsigned host_chunk_log(unsigned L) { return L >= 22 ? L - 2 : L >= 20 ? L - 1 : L; }
// Out-of-memory back-off: at most this many halvings of the chunk.
constexpr unsigned MSM_BACKOFF_HALVINGS = 8;

// One MSM of 2^L points accumulated chunk by chunk into the same windows, then
// reduced once.  inputs_of(k) names chunk k's bases and scalars (and waits for
// them to arrive); consumed(k) runs after chunk k's kernels are enqueued.
hipError_t msm_chunked_device(const msm_job &full, unsigned chunk_log, arena &ar,
                              const std::function<hipError_t(unsigned, const g1_affine **, const fe **)> &inputs_of,
                              const std::function<hipError_t(unsigned)> &consumed) {
  msm_job chunk = full;
  chunk.log_n = chunk_log;
  chunk.piece = msm_plain_piece(chunk_log);
  batch_layout bl;
  BC_TRY(layout_batch(&chunk, 1, &bl));
  g1_xyzz *A = nullptr, *tops = nullptr;
  BC_TRY(ar.get(&A, bl.nb));
  BC_TRY(ar.get(&tops, bl.tops_total));
  const unsigned K = 1u << (full.log_n - chunk_log);
  for (unsigned k = 0; k < K; k++) {
    BC_TRY(inputs_of(k, &bl.jt.job[0].bases, &bl.jt.job[0].scalars));
    BC_TRY(accumulate_phase(bl, 1, ar, A, tops, k > 0));
    BC_TRY(consumed(k));
  }
  BC_TRY(reduce_phase(bl, &chunk, 1, ar, A, tops));
  BC_TRY(ar.put(tops));
  BC_TRY(ar.put(A));
  return hipSuccess;
}

// One attempt of msm_execute with chunks of 2^chunk_log points.  Every
// allocation is made before any work is enqueued, so an out-of-memory return
// leaves the stream as it was.
hipError_t msm_execute_chunks(const msm_configuration &cfg, unsigned chunk_log, bool bases_host, bool scalars_host, bool results_host) {
  hipStream_t s = to_stream(cfg.stream);
  call_resources res(to_pool(cfg.mem_pool), s);
  const unsigned L = cfg.log_scalars_count;
  const size_t chunk_n = (size_t)1 << chunk_log;
  const unsigned K = 1u << (L - chunk_log);
  const bool copying = bases_host || scalars_host;
  // staging: two slots per copied input (chunk k uses slot k % 2)
  fe *s_slot[2] = {nullptr, nullptr};
  g1_affine *b_slot[2] = {nullptr, nullptr};
  for (unsigned i = 0; i < std::min(K, 2u); i++) {
    if (scalars_host)
      BC_TRY(res.get(&s_slot[i], chunk_n));
    if (bases_host)
      BC_TRY(res.get(&b_slot[i], chunk_n));
  }
  g1_jacobian *d_results = static_cast<g1_jacobian *>(cfg.results);
  if (results_host)
    BC_TRY(res.get(&d_results, 254));
  const msm_job full{static_cast<const g1_affine *>(cfg.bases), static_cast<const fe *>(cfg.scalars), d_results, L, msm_window_bits(L),
                     msm_plain_piece(L)};
  msm_job chunk = full;
  chunk.log_n = chunk_log;
  chunk.piece = msm_plain_piece(chunk_log);
  const size_t bytes = msm_footprint(chunk);
  char *block = nullptr;
  BC_TRY(res.get(&block, bytes));
  arena ar = arena::bump_mode(block, bytes, s);

  // Copies run on their own stream: chunk k's copy is enqueued right after chunk
  // k - 1's kernels (so a pageable copy, which holds the host thread, overlaps
  // them), into slot k % 2 once chunk k - 2 has been consumed.  A single copy runs
  // on the call's stream, unless a callback follows it, which would hold up the
  // kernels there.
  const bool own_stream = copying && (K > 1 || cfg.h2d_copy_finished_callback);
  hipStream_t cs = s;
  std::vector<hipEvent_t> loaded(K), freed(2);
  auto enqueue_copy = [&](unsigned k) -> hipError_t {
    if (k >= 2)
      BC_TRY(hipStreamWaitEvent(cs, freed[k % 2], 0));
    const size_t off = (size_t)k * chunk_n;
    if (scalars_host)
      BC_TRY(hipMemcpyAsync(s_slot[k % 2], static_cast<const fe *>(cfg.scalars) + off, sizeof(fe) * chunk_n, hipMemcpyHostToDevice, cs));
    if (bases_host)
      BC_TRY(hipMemcpyAsync(b_slot[k % 2], static_cast<const g1_affine *>(cfg.bases) + off, sizeof(g1_affine) * chunk_n, hipMemcpyHostToDevice, cs));
    if (own_stream)
      BC_TRY(hipEventRecord(loaded[k], cs));
    if (k + 1 == K) {
      // after the last copy, on the copy stream (src/msm.cu:183-191)
      if (cfg.h2d_copy_finished.handle)
        BC_TRY(hipEventRecord(to_event(cfg.h2d_copy_finished), cs));
      if (cfg.h2d_copy_finished_callback)
        BC_TRY(hipLaunchHostFunc(cs, cfg.h2d_copy_finished_callback, cfg.h2d_copy_finished_callback_data));
    }
    return hipSuccess;
  };
  if (own_stream) {
    BC_TRY(res.stream(&cs));
    for (auto &e : loaded)
      BC_TRY(res.event(&e));
    for (auto &e : freed)
      BC_TRY(res.event(&e));
    // the staging memory belongs to `s` until the copy stream is ordered after its allocation
    hipEvent_t ready = nullptr;
    BC_TRY(res.event(&ready));
    BC_TRY(hipEventRecord(ready, s));
    BC_TRY(hipStreamWaitEvent(cs, ready, 0));
  }
  if (copying)
    BC_TRY(enqueue_copy(0));
  auto inputs_of = [&](unsigned k, const g1_affine **b, const fe **sc) -> hipError_t {
    const size_t off = (size_t)k * chunk_n;
    if (own_stream)
      BC_TRY(hipStreamWaitEvent(s, loaded[k], 0));
    *b = bases_host ? b_slot[k % 2] : full.bases + off;
    *sc = scalars_host ? s_slot[k % 2] : full.scalars + off;
    return hipSuccess;
  };
  auto consumed = [&](unsigned k) -> hipError_t {
    if (!own_stream || k + 1 >= K)
      return hipSuccess;
    BC_TRY(hipEventRecord(freed[k % 2], s));
    return enqueue_copy(k + 1);
  };
  BC_TRY(msm_chunked_device(full, chunk_log, ar, inputs_of, consumed));
  res.streams_joined(); // `s` has waited for every copy; it need not for the callback
  if (results_host) {
    BC_TRY(hipMemcpyAsync(cfg.results, d_results, sizeof(g1_jacobian) * 254, hipMemcpyDeviceToHost, s));
    if (cfg.d2h_copy_finished.handle)
      BC_TRY(hipEventRecord(to_event(cfg.d2h_copy_finished), s));
    if (cfg.d2h_copy_finished_callback)
      BC_TRY(hipLaunchHostFunc(s, cfg.d2h_copy_finished_callback, cfg.d2h_copy_finished_callback_data));
  }
  return hipSuccess;
}

} // namespace

// msm_execute_async (src/msm.cu:419-460): bases, scalars and results may each
// be device, pinned or pageable memory.  Device-resident inputs run as one
// chunk; host inputs are copied in chunks overlapped with the accumulation of
// the chunk before.  When the pool cannot supply the temporaries, the call is
// planned again with chunks of half the size (as src/msm.cu:442-459 does), at
// most MSM_BACKOFF_HALVINGS times.  Chunked and unchunked calls give the same
// per-bit results as points (their Jacobian coordinates may differ).
hipError_t msm_execute(const msm_configuration &cfg) {
  const unsigned L = cfg.log_scalars_count;
  if (L > 28 || !cfg.bases || !cfg.scalars || !cfg.results)
    return hipErrorInvalidValue;
  const bool bases_host = classify_pointer(cfg.bases) != mem_kind::device;
  const bool scalars_host = classify_pointer(cfg.scalars) != mem_kind::device;
  const bool results_host = classify_pointer(cfg.results) != mem_kind::device;
  unsigned chunk_log = bases_host || scalars_host ? host_chunk_log(L) : L;
  const unsigned min_log = L > MSM_BACKOFF_HALVINGS ? L - MSM_BACKOFF_HALVINGS : 0;
  for (;;) {
    const hipError_t e = msm_execute_chunks(cfg, chunk_log, bases_host, scalars_host, results_host);
    if (e != hipErrorOutOfMemory || chunk_log <= min_log)
      return e;
    (void)hipGetLastError();
    chunk_log--;
  }
}

namespace {

// Device memory of the no-allocation entry point: one array per GPU, held
// from the library's load until the process ends, shared by every call on
// that GPU (calls that overlap on one GPU race on it).  On the host the name
// `scratch` is only a stand-in for the symbol; its device address on each
// GPU comes from hipGetSymbolAddress, resolved once per device with that
// device current.
constexpr size_t MSM_NO_ALLOC_BYTES = (size_t)192 << 20;
static __device__ __align__(256) unsigned char scratch[MSM_NO_ALLOC_BYTES];

std::mutex g_scratch_mu;
void *g_scratch[MAX_DEVICES];

hipError_t scratch_address(void **ptr) {
  const int d = device_slot();
  if (d < 0)
    return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[d]) {
    void *p = nullptr;
    BC_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch[d] = p;
  }
  *ptr = g_scratch[d];
  return hipSuccess;
}

// The plain call's device path (same window width, chunk length and kernels,
// hence the same per-bit results) over the static array instead of a pool
// block.  Bases, scalars and results must be device memory, and the job's
// footprint must fit the array; nothing is allocated.
hipError_t msm_execute_no_alloc(const msm_configuration &cfg) {
  const unsigned L = cfg.log_scalars_count;
  if (L > 28 || !cfg.bases || !cfg.scalars || !cfg.results)
    return hipErrorInvalidValue;
  for (const void *p : {cfg.bases, cfg.scalars, cfg.results})
    if (classify_pointer(p) != mem_kind::device)
      return hipErrorInvalidValue;
  const msm_job job{static_cast<const g1_affine *>(cfg.bases), static_cast<const fe *>(cfg.scalars), static_cast<g1_jacobian *>(cfg.results), L,
                    msm_window_bits(L), msm_plain_piece(L)};
  if (msm_footprint(job) > MSM_NO_ALLOC_BYTES)
    return hipErrorInvalidValue;
  void *base = nullptr;
  BC_TRY(scratch_address(&base));
  arena ar = arena::bump_mode(base, MSM_NO_ALLOC_BYTES, to_stream(cfg.stream));
  auto inputs_of = [&](unsigned, const g1_affine **b, const fe **sc) -> hipError_t {
    *b = job.bases;
    *sc = job.scalars;
    return hipSuccess;
  };
  auto consumed = [](unsigned) -> hipError_t { return hipSuccess; };
  return msm_chunked_device(job, L, ar, inputs_of, consumed);
}

} // namespace

} // namespace bc

using namespace bc;

extern "C" {

// Also resolves the current device's address of the no-allocation array.
bc_error msm_set_up() {
  void *p = nullptr;
  return as_bc(scratch_address(&p));
}

bc_error bc_amd_msm_execute_no_alloc(msm_configuration configuration) { return as_bc(msm_execute_no_alloc(configuration)); }

bc_error bc_amd_msm_fixed_base_table(const void *bases, unsigned log_count, unsigned window_bits, void *table, bc_stream stream) {
  return as_bc(msm_fixed_base_table(static_cast<const g1_affine *>(bases), log_count, window_bits, static_cast<g1_affine *>(table), to_stream(stream)));
}

bc_error msm_execute_async(msm_configuration configuration) { return as_bc(msm_execute(configuration)); }

bc_error msm_tear_down() { return bc_success; }

} // extern "C"
