// Host-side interface of the matrix-core FFT passes (fft_matrix.hip).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace sh {
namespace fft {

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
