// Internal NTT interface shared by the plain C ABI path and the batched /
// serving layer.
#pragma once

#include "common.h"
#include "field.cuh"

namespace bc {

constexpr unsigned NTT_MAX_LOG = 28;
constexpr unsigned NTT_MAX_JOBS = 64;
// Stages per HBM pass of VALU butterflies at most (tiles of 2^10 elements, 32 KiB
// of LDS): five blocks share a CU, so one block's loads and stores overlap the
// others' butterflies.  Against tiles of 2^9..2^12 elements it is the fastest of
// these passes wherever they fill the GPU (2^24: 1.80 ms in three
// passes against 2.27 ms in two passes of 2^12-element tiles); launches of
// NTT_SMALL_ELEMENTS and less, and natural-order transforms from
// NTT_MFMA_MIN_LOG on, take passes of their own.
constexpr unsigned NTT_LOG_TILE = 10;

// Smallest natural-order transform whose first twelve stages run on the matrix
// cores (two passes of six).  Against the VALU passes alone: 2^24 1.73 -> 1.46 ms,
// 2^20 120 -> 95 us, 2^18 47 -> 43 us; at 2^17 the third pass costs what they save.
constexpr unsigned NTT_MFMA_MIN_LOG = 18;
// Smallest one with a third such pass (five to ten stages are then left for one
// VALU pass; below, the one VALU pass takes them all): 2^23 731 -> 688 us, 2^24
// 1.46 -> 1.38 ms.
constexpr unsigned NTT_MFMA_ROWS_MIN_LOG = 23;

// Launches of at most this many elements run one butterfly per thread and stage
// (a wave per SIMD); at 2^18 that takes 46 us, the larger passes 43 to 47 us.
constexpr uint64_t NTT_SMALL_ELEMENTS = 1u << 17;

// Transforms whose last pass (6..10 stages, one launch) starts on the matrix
// cores.  Its row factors are a table of 2^log_n elements per direction, so it is
// kept to tables of 512 MB: for all sizes 56 MB a direction to 2^20, 760 MB to 2^24,
// beside twiddles of 32 and 512 MB.
constexpr unsigned NTT_MFMA_LAST_MAX_LOG = 24;
inline bool ntt_mfma_last(unsigned log_n) {
  return log_n >= NTT_MFMA_MIN_LOG && log_n <= NTT_MFMA_LAST_MAX_LOG && log_n != NTT_MFMA_ROWS_MIN_LOG;
}

inline unsigned ntt_passes(unsigned log_n) { return (log_n + NTT_LOG_TILE - 1) / NTT_LOG_TILE; }

// A first pass of `first` stages is valid for a size of two or more passes
// when the remaining stages fit the remaining passes.
inline bool ntt_split_valid(unsigned log_n, unsigned first) {
  const unsigned passes = ntt_passes(log_n);
  return passes >= 2 && first >= 1 && first <= NTT_LOG_TILE && log_n - first <= (passes - 1) * NTT_LOG_TILE;
}

struct ntt_job {
  const fe *in; // device, may equal out
  fe *out;      // device
  unsigned log_n;
  bool bitrev_in;
  bool inverse;
  unsigned log_ext; // coset LDE: 0 = plain transform
  unsigned coset;
};

// Shape of a transform that every entry point accepts: 2^1..2^NTT_MAX_LOG
// elements, an extended domain of at most 2^NTT_MAX_LOG (compared without a
// sum that could wrap), and a coset index below 2^log_ext.
inline bool ntt_shape_valid(unsigned log_n, unsigned log_ext, unsigned coset) {
  return log_n != 0 && log_n <= NTT_MAX_LOG && log_ext <= NTT_MAX_LOG - log_n && (log_ext == 0 || coset < (1u << log_ext));
}

inline bool ntt_job_valid(const ntt_job &q) { return ntt_shape_valid(q.log_n, q.log_ext, q.coset) && q.in && q.out; }

struct ntt_tables {
  const fe *fwd, *inv, *inv_sizes;
  const int8_t *mfma_fwd, *mfma_inv;
  const fe *rows_fwd, *rows_inv;
  const fe *last_rows[2][NTT_MFMA_LAST_MAX_LOG + 1]; // by direction and size; null: VALU passes
  unsigned log_size;
};

// Twiddle tables for sizes up to 2^max_log_n and kernel attributes of the
// current device.  May allocate and synchronise `stream` (not capturable);
// afterwards every batch of transforms up to that size is capturable.
hipError_t ntt_prepare(unsigned max_log_n, hipStream_t stream, ntt_tables *out);

// The same for the largest of these jobs.
hipError_t ntt_prepare_jobs(const ntt_job *jobs, unsigned count, hipStream_t stream);

// Up to NTT_MAX_JOBS transforms, one launch per pass index and butterfly
// order; temporaries (coset twist tables) come from `ar`.  `small_passes` false:
// also a launch that cannot fill the GPU takes the passes that the tuning table
// names (the autotuner times those).
hipError_t ntt_batch_device(const ntt_job *jobs, unsigned count, arena &ar, bool small_passes = true);

} // namespace bc
