// Host-side interface of the circle FFT module used by the batched commit plan.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace sh {
namespace fft {

// Pass schedule of one LDE size class, chosen by the autotuner: the number of layers
// in the contiguous passes (12 or 13), whether the strided inverse and forward
// passes are fused into one launch, and whether the passes use the matrix cores
// (fft_matrix.hip; log sizes 17..20, fused).
struct LdeVariant {
  uint8_t kc = 12;
  bool fused = false;
  bool mat = false;
};

// Device memory that lde_same_size needs beside the columns for this shape and variant
// (matrices of the matrix-core passes; 0: none).  Without it the passes run on butterflies: callers
// take it as DevBuf::optional, so no call needs more memory than its columns and tables.
size_t lde_workspace_bytes(uint32_t n, uint32_t log_blowup, uint64_t n_cols, LdeVariant var);

// Interpolate d_src into d_coeffs (may alias) and evaluate on the canonic domain of log
// n + log_blowup into d_lde; device pointer tables of n_cols columns; allocates nothing.
// ws: lde_workspace_bytes of device memory, written by each call; null: the butterfly passes of var.
void lde_same_size(const uint32_t* const* d_src, uint32_t* const* d_coeffs, uint32_t* const* d_lde, uint32_t n_cols,
                   uint32_t n, uint32_t log_blowup, const uint32_t* tw, const uint32_t* itw, uint64_t tree_len,
                   LdeVariant var, void* ws);

// Autotuner results (per log size, blowup and column-count bucket); defaults otherwise.
LdeVariant lde_variant_for(uint32_t n, uint32_t log_blowup, uint64_t n_cols);
void set_lde_variant(uint32_t n, uint32_t log_blowup, uint64_t n_cols, LdeVariant v);

}  // namespace fft
}  // namespace sh
