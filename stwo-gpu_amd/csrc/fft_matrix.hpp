// Host-side interface of the matrix-core FFT passes (fft_matrix.hip).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace sh {
namespace fft {

// Column groups per block of a pass over n_groups groups at each of `tiles` tiles, `fill` blocks at
// a time on the chip.  A block's first group waits for its matrices and values with nothing to
// compute, about 0.3 groups' worth, so blocks walk over many groups; but every block lasts as long
// as the longest, so what counts is the rounds that the chip needs times a block's length.  A fixed
// number of rounds left 36 groups in blocks of 32 and 4, with the long blocks on half of the XCDs
// (forward pass of 72 columns of log 20 at blowup 8: 1490 us, 1020 at 12 groups a block), and
// blocks of 4 at 4.5 rounds (its middle pass at blowup 2: 304 us, 279 at 18).  At one tile the
// blocks of one long round read far apart: past 12 rounds of single groups (columns beyond the
// caches) a block takes at most a quarter of them (16384 columns of log 12: 129 us at 4 groups a
// block, 139 at 16; 4096 columns: 34 at 4, one round, and 37 at 1).
inline uint32_t groups_per_block(uint64_t n_groups, uint64_t tiles, uint32_t fill) {
  const uint64_t alone = (n_groups * tiles + fill - 1) / fill;
  const uint64_t most = tiles == 1 && alone > 12 ? alone / 4 : 32;
  uint64_t best = 1, best_cost = ~0ull;
  for (uint64_t p = 1; p <= most && p <= 32; p++) {
    const uint64_t chunks = (n_groups + p - 1) / p, cost = (chunks * tiles + fill - 1) / fill * (10 * p + 3);
    if (cost < best_cost) {
      best_cost = cost;
      best = p;
    }
  }
  return (uint32_t)best;
}

// Whether a transform of n_cols whole columns over the domain of log_n (10 .. 12) runs on the matrix
// cores; blowup (forward): log_n less the coefficients' log size.  The line lies where the pass has
// made up for the launch that lays out its matrices (6 us), in millions (2^20) of values: 24 in place;
// forward into other columns 32, 36, 48 and 80 (64 onto 2^10) at blowups 1, 2, 4 and 8, since the
// butterflies skip the layers of the zero coefficients and the matrices do not; inverse into other
// columns 36.  Matrix / butterfly time of a call just below and from the line on, for columns of 2^10,
// 2^11 and 2^12:
//   in place inverse      20: 1.05 1.02 0.99   24: 1.01 1.00 0.95   32: 0.97 0.97 0.92
//   in place forward      20: 0.98 1.03 1.00   24: 0.95 0.99 0.96   32: 0.92 0.96 0.94
//   forward, blowup 1     24: 1.01 1.03 1.02   32: 0.97 0.99 0.98   48: 0.95 0.98 0.95
//   forward, blowup 2     32: 1.01 1.02 1.01   36: 0.99 0.94 0.97   48: 0.90 0.93 0.95
//   forward, blowup 4     40: 1.00 1.02 1.01   48: 1.00 0.99 0.99   64: 0.88 0.96 0.94
//   forward, blowup 8     64: 0.92 1.03 1.02   80: 0.90 0.98 0.96  128: 0.86 0.92 0.89
//   inverse               32: 1.06 1.05 1.00   36: 1.00 0.98 0.95  128: 0.92 0.86 0.82
inline bool use_matrices_tile(uint32_t log_n, uint64_t n_cols, bool inverse, uint32_t blowup, bool in_place) {
  constexpr uint32_t FORWARD[4] = {32, 36, 48, 80};
  if (log_n < 10 || log_n > 12 || blowup > 3) return false;
  const uint64_t line = in_place && !blowup ? 24 : inverse ? 36 : blowup == 3 && log_n == 10 ? 64 : FORWARD[blowup];
  return (n_cols << log_n) >= line << 20;
}

// The passes over whole small columns; mats: tile_matrix_bytes of device memory filled by
// tile_matrices, tw / itw: the domain's tree part.
size_t tile_matrix_bytes(uint32_t log_n);
void tile_matrices(bool inverse, uint32_t log_n, const uint32_t* tw, unsigned char* mats);
void interpolate_tiles(const uint32_t* const* src, uint32_t* const* dst, uint32_t n_cols, uint32_t log_n,
                       const uint32_t* itw, unsigned char* mats);
void evaluate_tiles(const uint32_t* const* src, uint32_t* const* dst, uint32_t n_cols, uint32_t src_log, uint32_t log_n,
                    const uint32_t* tw, unsigned char* mats);

// Low-degree extension of columns of log 17 .. 20; mats: lde_matrix_bytes of device memory.
bool use_matrices_lde(uint32_t n, uint32_t log_blowup, uint64_t n_cols);
size_t lde_matrix_bytes(uint32_t n, uint32_t log_blowup);
void lde_matrices(const uint32_t* const* src, uint32_t* const* coeffs, uint32_t* const* lde, uint32_t n_cols, uint32_t n,
                  uint32_t log_blowup, const uint32_t* tw, const uint32_t* itw, unsigned char* mats);

}  // namespace fft
}  // namespace sh
