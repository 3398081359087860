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

// Whole small columns (log 10 .. 12), many at a time; mats: tile_matrix_bytes of device memory
// filled by tile_matrices, tw / itw: the domain's tree part.
bool use_matrices_tile(uint32_t log_n, uint64_t n_cols);
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
