// Circle FFT passes whose layers from 4 up run on the integer matrix cores.
//
// Four consecutive layers [b, b + 4) map the 16 values whose indexes differ in bits b .. b + 3
// by a 16 x 16 matrix that depends only on the index bits above (h = index >> (b + 4)): the same
// matrix for every column and every value of the low bits.  mfma_m31.hpp applies such a map to
// 32 vectors in four matrix instructions and about 8 VALU instructions per value, a third of
// what four butterfly layers cost, and the passes were bound by exactly those instructions.
// The matrices are laid out by matrix_kernel from the twiddle tree once per call (17 bytes per
// domain point and direction, as much as 4 columns), so the passes here serve batches of many
// columns; see use_matrices_tile and use_matrices_lde for where that starts to pay.
//
// Layers 0..3 stay butterflies: their matrices would differ for every 16 values of a column.
// A thread holds 16 consecutive values there, and its 15 twiddles are seven words: layer 0's
// circle twiddles [y, -y, -x, x] come from the same level-0 words as layer 1's.
#include <algorithm>

#include "fft.hpp"
#include "fft_matrix.hpp"
#include "field.hpp"
#include "gmem.hpp"
#include "mfma_m31.hpp"
#include "runtime.hpp"

namespace sh {
namespace fft {

using mm::Mat;

// ---- matrices ------------------------------------------------------------------
// Stage: `count` matrices over the field of 4 index bits whose top w bits are the layers
// [layer, layer + w) (the lower 4 - w bits pass through), one per value of the index bits above.
struct MatStage {
  const uint32_t* tw;        // the domain's tree part (line level 0)
  uint32_t log_n;            // the domain
  uint32_t inverse;
  uint32_t layer, w, first;  // first: index of the stage's first matrix in the table
  uint32_t scale;            // entries times 2^scale
};
struct MatArgs {
  unsigned char* out;
  uint32_t n_stages;
  MatStage st[8];
};

// A block makes MB matrices, thread (o, m) of it the entry of output o and input m, its four
// digit rotations and their limbs; the chunks are written from LDS.  (2^20 inverse and 2^21
// forward, 53 MB: 45 us with each limb row computing its own entries, 27 us with one matrix per
// block, whose loads and products are one latency after another.)
constexpr uint32_t MB = 4;
__global__ __launch_bounds__(256) void matrix_kernel(MatArgs A, uint32_t total) {
  __shared__ __align__(16) uint32_t out[MB * 1024];
  const uint32_t o = threadIdx.x >> 4, m = threadIdx.x & 15;
  uint32_t e[MB], f[MB][4];
#pragma unroll
  for (uint32_t q = 0; q < MB; q++) {
    const uint32_t mat = min(MB * blockIdx.x + q, total - 1);
    uint32_t k = 0;
    while (k + 1 < A.n_stages && mat >= A.st[k + 1].first) k++;
    const MatStage& S = A.st[k];
    const uint32_t h = mat - S.first, half = 1u << (S.log_n - 1);
#pragma unroll
    for (uint32_t l = 0; l < 4; l++) {
      f[q][l] = 1;
      if (l < 4 - S.w) continue;                       // no layer on this bit
      const uint32_t layer = S.layer + l - (4 - S.w);  // >= 1
      const uint32_t* lvl = S.tw + (half - (half >> (layer - 1)));
      // inverse: (v0 + v1, (v0 - v1) t), t by the input bits above; forward: v0 +- t v1, t by
      // the output bits above
      const uint32_t t = lvl[(h << (3 - l)) | ((S.inverse ? m : o) >> (l + 1))];
      f[q][l] = ((S.inverse ? o : m) >> l) & 1 ? t : 1u;
    }
    const uint32_t none = (1u << (4 - S.w)) - 1;  // bits without a layer pass through
    const uint32_t sign = __popc(o & m & ~none) & 1;
    e[q] = mul(mul(f[q][0], f[q][1]), mul(f[q][2], f[q][3]));
    e[q] = ((o ^ m) & none) ? 0u : mm::rot31(sign ? neg(e[q]) : e[q], S.scale);
  }
  // limb i of the digits j: byte i of each rotation; chunk (o / 8, slot / 4), lane row + 32 g
  const uint32_t slot = m >> 1, lane = ((o & 7) << 2) | ((m & 1) << 5);
#pragma unroll
  for (uint32_t q = 0; q < MB; q++) {
    uint32_t w[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) w[j] = mm::limbs(mm::rot31(e[q], 8 * j));
    uint32_t* const p = out + 1024 * q + 256 * (2 * (o >> 3) + (slot >> 2)) + 4 * lane + (slot & 3);
    // bytes transposed: row limb i holds byte i of w[0..3]
    const uint32_t a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400);
    const uint32_t c = __builtin_amdgcn_perm(w[1], w[0], 0x07030602), d = __builtin_amdgcn_perm(w[3], w[2], 0x07030602);
    p[0] = __builtin_amdgcn_perm(b, a, 0x05040100);
    p[4] = __builtin_amdgcn_perm(b, a, 0x07060302);
    p[8] = __builtin_amdgcn_perm(d, c, 0x05040100);
    p[12] = __builtin_amdgcn_perm(d, c, 0x07060302);
  }
  __syncthreads();
#pragma unroll
  for (uint32_t q = 0; q < MB; q++)
    if (MB * blockIdx.x + q < total)
      reinterpret_cast<uint4*>(A.out + (size_t)(MB * blockIdx.x + q) * mm::MAT_BYTES)[threadIdx.x] =
          reinterpret_cast<const uint4*>(out)[256 * q + threadIdx.x];
}

// ---- butterflies of layers 0..3 on 16 consecutive values -------------------------------
struct Tw16 {
  uint4 a;  // level 0: layer 1's four twiddles, and layer 0's as pairs (x, y)
  uint2 b;  // level 1: layer 2
  uint32_t c;  // level 2: layer 3
};
// g: index of the 16 values within the domain (position >> 4)
__device__ __forceinline__ Tw16 load_tw16(const uint32_t* tw, uint32_t log_n, uint32_t g) {
  const SH_GLOBAL uint32_t* t = as_global(tw);
  const uint32_t half = 1u << (log_n - 1);
  Tw16 r;
  r.a = at(reinterpret_cast<const SH_GLOBAL uint4*>(t), g);
  r.b = at(reinterpret_cast<const SH_GLOBAL uint2*>(t + (half - (half >> 1))), g);
  r.c = at(t + (half - (half >> 2)), g);
  return r;
}
template <bool INV, bool NEG>
__device__ __forceinline__ void butterfly(uint32_t& x0, uint32_t& x1, uint32_t t2) {
  // t2: twice the twiddle, whose sign NEG flips
  if constexpr (INV) {
    const uint32_t a = x0, b = x1;
    x0 = add(a, b);
    x1 = mul_dbl(NEG ? sub(b, a) : sub(a, b), t2);
  } else {
    const uint32_t a = x0, t = mul_dbl(x1, t2);
    x0 = NEG ? sub(a, t) : add(a, t);
    x1 = NEG ? add(a, t) : sub(a, t);
  }
}
template <bool INV>
__device__ __forceinline__ void layers0to3(uint32_t (&v)[16], const Tw16& tw) {
  const uint32_t a[4] = {2 * tw.a.x, 2 * tw.a.y, 2 * tw.a.z, 2 * tw.a.w};
  const uint32_t b[2] = {2 * tw.b.x, 2 * tw.b.y}, c = 2 * tw.c;
  auto layer0 = [&] {
#pragma unroll
    for (int p = 0; p < 2; p++) {  // pair (x, y) = level 0 words 2p, 2p + 1: [y, -y, -x, x]
      butterfly<INV, false>(v[8 * p], v[8 * p + 1], a[2 * p + 1]);
      butterfly<INV, true>(v[8 * p + 2], v[8 * p + 3], a[2 * p + 1]);
      butterfly<INV, true>(v[8 * p + 4], v[8 * p + 5], a[2 * p]);
      butterfly<INV, false>(v[8 * p + 6], v[8 * p + 7], a[2 * p]);
    }
  };
  auto layer1 = [&] {
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int r = 0; r < 2; r++) butterfly<INV, false>(v[4 * k + r], v[4 * k + r + 2], a[k]);
  };
  auto layer2 = [&] {
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
      for (int r = 0; r < 4; r++) butterfly<INV, false>(v[8 * k + r], v[8 * k + r + 4], b[k]);
  };
  auto layer3 = [&] {
#pragma unroll
    for (int r = 0; r < 8; r++) butterfly<INV, false>(v[r], v[r + 8], c);
  };
  if constexpr (INV) {
    layer0();
    layer1();
    layer2();
    layer3();
  } else {
    layer3();
    layer2();
    layer1();
    layer0();
  }
}

// ---- contiguous pass: layers 0 .. K - 1 (K = 10, 11, 12) ---------------------------------
// A block takes 2^13 values at a time: 2^(13 - K) columns of 2^K consecutive values, and walks
// over `per_block` such column groups at one tile, so its matrices and twiddles stay in
// registers and the next group's values are loaded while this one's are transformed.  Position q
// of a group: bits 0 .. K - 1 the index in the column's tile, the rest the column.  Three stages,
// exchanged through LDS (stage B writes back where it reads):
//   A  layers 0..3, thread q >> 4 holds 16 consecutive values; they move between this layout and
//      one where a wave's access covers 1 KiB through an LDS region of the wave's own (16-byte
//      accesses 64 bytes apart straight to memory cost 0.15 ms more on 2^16 columns of 2^12);
//   B  layers 4..7, field bits 4..7; the 32 vectors of a tile are bits 0..3 and column bit K, and
//      the other bits select the tile: bits 8 .. K - 1 choose its matrix;
//   C  layers 8 .. K - 1, field bits K - 4 .. K - 1; vectors bits 1..5, and bit 0 selects the
//      wave's tile, so its two tiles are loaded and stored as 8-byte pairs.
// Two blocks share a CU, so one's exchanges are filled by the other's arithmetic.
struct ContigArgs {
  uint32_t* const* dst;
  const uint32_t* const* src;
  const uint32_t* tw;  // the domain's tree part (line level 0), for layers 0..3
  const unsigned char* mat_b;  // layers 4..7: 2^(log_n - 8) matrices
  const unsigned char* mat_c;  // layers 8..K-1: 2^(log_n - K) matrices
  uint32_t n_cols, log_n;
  uint32_t tiles_log, n_groups, per_block;
};

constexpr int CT = 512;
// LDS word of position q: 16-word rows padded by 4, so the 16-byte accesses of stage A (64 bytes
// apart) spread over the banks
__host__ __device__ constexpr uint32_t lds_pos(uint32_t q) { return q + ((q >> 4) << 2); }
constexpr uint32_t lds_words(uint32_t values) { return values / 16 * 20; }

// NS (forward): source slots of stage C that hold coefficients, 8 / 2^blowup; the rest are zero.
// NT: streaming accesses.
template <bool INV, int K, int NS, bool NT>
__global__ __launch_bounds__(CT) __attribute__((amdgpu_waves_per_eu(4))) void contig_matrix_kernel(ContigArgs A) {
  __shared__ __align__(16) uint32_t s[lds_words(1u << 13)];
  __shared__ __align__(16) uint32_t turn[lds_words(1u << 13)];
  constexpr uint32_t COLS = 1u << (13 - K);
  // neighbours walk the tiles of the same columns
  const uint32_t v = xcd_order();
  const uint32_t tile = v & ((1u << A.tiles_log) - 1);
  uint32_t group = (v >> A.tiles_log) * A.per_block;
  const uint32_t group_end = min(group + A.per_block, A.n_groups);
  const uint32_t base = tile << K;
  const uint32_t t = threadIdx.x, lane = t & 63, n = lane & 31, g = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);

  // stage B: tile o = 2 wave + j of 16: the K - 8 matrix bits and the column bits from K + 1 on;
  // below 16 matrices j is a column bit, so the wave's two tiles share one
  constexpr uint32_t NB = K == 12 ? 2 : 1;
  const uint32_t b_h = (NB * wave) & ((1u << (K - 8)) - 1);
  const uint32_t b_pos = (n & 15) | (g << 4) | (b_h << 8) | ((n >> 4) << K) | ((NB * wave) >> (K - 8) << (K + 2));
  // stage C: field base fb, positions of tile 0 (tile 1: + 1)
  constexpr uint32_t fb = K - 4;
  const uint32_t c_pos = (n << 1) | ((wave & ((1u << (fb - 6)) - 1)) << 6) | (g << fb) | ((wave >> (fb - 6)) << K);
  // stage A: the wave's 1024 values lie in one column (K >= 10)
  const uint32_t a_col = (wave << 10) >> K, a_idx = base + ((wave << 10) & ((1u << K) - 1));
  const uint32_t c_col = wave >> (fb - 6), c_idx = c_pos & ((1u << K) - 1);
  uint4* const sa = reinterpret_cast<uint4*>(s + 20 * t);
  uint4* const own = reinterpret_cast<uint4*>(turn + 20 * t);  // the thread's 16 values
  uint32_t* const row = turn + lds_pos((wave << 10) + 4 * lane);  // 4 values of each of its four 1 KiB rows

  Mat mb[NB];
#pragma unroll
  for (uint32_t j = 0; j < NB; j++) mb[j] = mm::load_mat(as_global(A.mat_b), (tile << (K - 8)) + b_h + j, lane);
  const Mat mc = mm::load_mat(as_global(A.mat_c), tile, lane);
  const Tw16 tw = load_tw16(A.tw, A.log_n, (a_idx >> 4) + lane);

  // (lds_pos adds over the bits from 4 on, so a slot is a constant offset)
  uint32_t* const sb = s + lds_pos(b_pos);
  uint32_t* const sc = s + lds_pos(c_pos);
  constexpr uint32_t B1 = lds_pos(NB == 2 ? 1u << 8 : 1u << (K + 1));
  auto slot_c = [&](uint32_t e) { return reinterpret_cast<uint2*>(sc + lds_pos(e << (fb + 1))); };
  auto stage_b = [&] {
#pragma unroll
    for (uint32_t j = 0; j < 2; j++) {
      uint32_t d[8];
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) d[e] = sb[j * B1 + lds_pos(e << 5)];
      mm::apply<INV ? mm::DIGITS : mm::CANON>(mb[j & (NB - 1)], d, d);
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) sb[j * B1 + lds_pos(e << 5)] = d[e];
    }
  };

  if constexpr (INV) {
    uint4 x[4];
    // (a column past the last is read as the last and not stored)
    auto load = [&](uint32_t grp) {
      const BufCol p(ld_uniform(A.src, min(grp * COLS + a_col, A.n_cols - 1)) + a_idx);
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) x[k] = p.load4<NT>(4 * lane, k << 8);
    };
    load(group);
    for (; group < group_end; group++) {
#pragma unroll
      for (uint32_t k = 0; k < 4; k++) *reinterpret_cast<uint4*>(row + lds_pos(k << 8)) = x[k];
      if (group + 1 < group_end) load(group + 1);
      uint32_t w[16];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint4 y = own[k];
        w[4 * k] = y.x;
        w[4 * k + 1] = y.y;
        w[4 * k + 2] = y.z;
        w[4 * k + 3] = y.w;
      }
      __builtin_amdgcn_wave_barrier();
      layers0to3<true>(w, tw);
#pragma unroll
      for (int k = 0; k < 4; k++)
        sa[k] = make_uint4(mm::digits(w[4 * k]), mm::digits(w[4 * k + 1]), mm::digits(w[4 * k + 2]),
                           mm::digits(w[4 * k + 3]));
      __syncthreads();
      stage_b();
      __syncthreads();
      uint32_t d0[8], d1[8];
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) {
        const uint2 y = *slot_c(e);
        d0[e] = y.x;
        d1[e] = y.y;
      }
      __syncthreads();  // s may be written again
      mm::apply<mm::CANON>(mc, d0, d0);
      mm::apply<mm::CANON>(mc, d1, d1);
      const uint32_t col = group * COLS + c_col;
      if (col < A.n_cols) {
        const BufCol p(ld_uniform(A.dst, col) + base);
#pragma unroll
        for (uint32_t e = 0; e < 8; e++) p.store2<NT>(d0[e], d1[e], c_idx, e << (fb + 1));
      }
    }
  } else {
    uint2 x[NS];
    auto load = [&](uint32_t grp) {
      const BufCol p(ld_uniform(A.src, min(grp * COLS + c_col, A.n_cols - 1)) + base);
#pragma unroll
      for (uint32_t e = 0; e < NS; e++) x[e] = p.load2<NT>(c_idx, e << (fb + 1));
    };
    load(group);
    for (; group < group_end; group++) {
      uint32_t d0[8], d1[8];
#pragma unroll
      for (int e = 0; e < NS; e++) {
        d0[e] = mm::digits(x[e].x);
        d1[e] = mm::digits(x[e].y);
      }
      if (group + 1 < group_end) load(group + 1);
      mm::apply<mm::DIGITS, NS>(mc, d0, d0);
      mm::apply<mm::DIGITS, NS>(mc, d1, d1);
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) *slot_c(e) = make_uint2(d0[e], d1[e]);
      __syncthreads();
      stage_b();
      __syncthreads();
      uint32_t w[16];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint4 y = sa[k];
        w[4 * k] = y.x;
        w[4 * k + 1] = y.y;
        w[4 * k + 2] = y.z;
        w[4 * k + 3] = y.w;
      }
      __syncthreads();  // s may be written again
      layers0to3<false>(w, tw);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < 4; k++) own[k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
      __builtin_amdgcn_wave_barrier();
      const uint32_t col = group * COLS + a_col;
      if (col < A.n_cols) {
        const BufCol p(ld_uniform(A.dst, col) + a_idx);
#pragma unroll
        for (uint32_t k = 0; k < 4; k++)
          p.store4<NT>(*reinterpret_cast<const uint4*>(row + lds_pos(k << 8)), 4 * lane, k << 8);
      }
    }
  }
}

// ---- middle pass of the low-degree extension: layers 12 .. 11 + K (K = 5 .. 8) --------------
// A block takes 2^14 values of one column: 2^T consecutive words (T = 14 - K) at each of the 2^K
// values of index bits 12 .. 11 + K, and walks over `per_block` columns, the next one's values in
// flight.  Tile position q: bits 0 .. T - 1 the word, T .. 13 the layer
// bits.  Two stages, each four field bits; bit 0 selects the wave's tile (8-byte accesses):
//   D  layers 12..15 (q bits T .. T + 3); vectors q bits 1..5, the wave's matrix chosen by the
//      layer bits above;
//   E  the remaining w = K - 4 layers; the field's lower 4 - w bits are q bits from 6 on that no
//      layer touches; vectors q bits 1..5, the wave q bits T .. T + 3.
// Inverse D, E (the interpolation's scale is part of E's matrix), store the coefficients; then
// from the same registers, for each of the evaluation domain's blocks, forward E, D.
// Memory accesses of a wave complete in order, so a matrix loaded from memory after a stage's
// stores would wait for them: a wave keeps its inverse D matrix and its forward D matrix of the
// first block in registers, that of the second block and the three E matrices in LDS (blowup 2;
// further blocks' matrices come from memory).
struct StridedArgs {
  uint32_t* const* coeffs;  // in place
  uint32_t* const* lde;
  const unsigned char *inv_d, *inv_e, *fwd_d, *fwd_e;
  uint32_t n_cols, n, n_blocks;
  uint32_t tiles_log, per_block;
};

constexpr int LT = 1024;
template <int K, bool TWO, bool NT>
__global__ __launch_bounds__(LT) void lde_matrix_kernel(StridedArgs A) {
  constexpr uint32_t T = 14 - K, W = K - 4;
  __shared__ __align__(16) uint32_t s[lds_words(1u << 14)];
  __shared__ __align__(16) mm::v4i mats[(3 + LT / 64) * 256];  // inverse E, forward E 0 and 1, each wave's forward D 1
  const uint32_t v = xcd_order();
  const uint32_t tile = v & ((1u << A.tiles_log) - 1);
  uint32_t col = (v >> A.tiles_log) * A.per_block;
  const uint32_t col_end = min(col + A.per_block, A.n_cols);
  const uint32_t t = threadIdx.x, lane = t & 63, n = lane & 31, g = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // word of the column (from the tile's first) of tile position q
  auto word = [](uint32_t q) { return ((q >> T) << 12) | (q & ((1u << T) - 1)); };
  // stage D: the wave's 4 bits are the W matrix bits, then q bits 6 .. T - 1
  const uint32_t d_h = wave & ((1u << W) - 1);
  const uint32_t d_pos = (n << 1) | ((wave >> W) << 6) | (g << T) | (d_h << (T + 4));
  // stage E: field bit b at q bit 6 + b below 4 - W, at T + 4 + b - (4 - W) from there on; bit 0
  // is the lane's g, bits 1..3 the slot
  auto e_field = [](uint32_t m) {
    const uint32_t low = m & ((1u << (4 - W)) - 1), high = m >> (4 - W);
    return (low << 6) | (high << (T + 4));
  };
  const uint32_t e_pos = (n << 1) | (wave << T) | e_field(g);
  uint32_t* const sd = s + lds_pos(d_pos);
  uint32_t* const se = s + lds_pos(e_pos);
  auto at_d = [&](uint32_t e) { return reinterpret_cast<uint2*>(sd + lds_pos(e << (T + 1))); };
  auto at_e = [&](uint32_t e) { return reinterpret_cast<uint2*>(se + lds_pos(e_field(2 * e))); };
  const uint32_t d_word = word(d_pos), e_word = word(e_pos), tile_word = tile << T;

  uint2 x[8];
  auto load = [&](uint32_t c) {
    const BufCol p(ld_uniform(A.coeffs, c) + tile_word);
#pragma unroll
    for (uint32_t e = 0; e < 8; e++) x[e] = p.load2<NT>(d_word, e << 13);
  };
  load(col);
  if (wave < 3 && wave <= A.n_blocks) {  // uniform
    const Mat m = mm::load_mat(as_global(wave ? A.fwd_e : A.inv_e), wave ? wave - 1 : 0, lane);
#pragma unroll
    for (int k = 0; k < 4; k++) mats[256 * wave + 64 * k + lane] = m.c[k];
  }
  if (A.n_blocks > 1) {
    const Mat m = mm::load_mat(as_global(A.fwd_d), (1u << W) + d_h, lane);
#pragma unroll
    for (int k = 0; k < 4; k++) mats[256 * (3 + wave) + 64 * k + lane] = m.c[k];
  }
  const Mat inv_d = mm::load_mat(as_global(A.inv_d), d_h, lane);
  const Mat fwd_d = mm::load_mat(as_global(A.fwd_d), d_h, lane);
  auto lds_mat = [&](uint32_t i) {
    Mat m;
#pragma unroll
    for (int k = 0; k < 4; k++) m.c[k] = mats[256 * i + 64 * k + lane];
    return m;
  };
  for (; col < col_end; col++) {
    uint32_t d0[8], d1[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      d0[e] = mm::digits(x[e].x);
      d1[e] = mm::digits(x[e].y);
    }
    if (col + 1 < col_end) load(col + 1);
    mm::apply<mm::DIGITS>(inv_d, d0, d0);
    mm::apply<mm::DIGITS>(inv_d, d1, d1);
    __syncthreads();  // the previous column's last stage has read s (at first: mats is written)
#pragma unroll
    for (int e = 0; e < 8; e++) *at_d(e) = make_uint2(d0[e], d1[e]);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint2 y = *at_e(e);
      d0[e] = y.x;
      d1[e] = y.y;
    }
    {
      const Mat m = lds_mat(0);
      mm::apply<mm::CANON>(m, d0, d0);
      mm::apply<mm::CANON>(m, d1, d1);
      const BufCol p(ld_uniform(A.coeffs, col) + tile_word);
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) {
        p.store2<NT>(d0[e], d1[e], e_word, word(e_field(2 * e)));
        d0[e] = mm::digits(d0[e]);
        d1[e] = mm::digits(d1[e]);
      }
    }
    const uint32_t n_blocks = TWO ? 2 : A.n_blocks;
#pragma unroll TWO ? 2 : 1
    for (uint32_t b = 0; b < n_blocks; b++) {
      uint32_t r0[8], r1[8];
      {
        const Mat m = b < 2 ? lds_mat(1 + b) : mm::load_mat(as_global(A.fwd_e), b, lane);
        mm::apply<mm::DIGITS>(m, d0, r0);
        mm::apply<mm::DIGITS>(m, d1, r1);
      }
      if (b) __syncthreads();  // stage D of the previous block has read s
#pragma unroll
      for (int e = 0; e < 8; e++) *at_e(e) = make_uint2(r0[e], r1[e]);
      __syncthreads();
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint2 y = *at_d(e);
        r0[e] = y.x;
        r1[e] = y.y;
      }
      {
        const Mat m = b == 0 ? fwd_d : b == 1 ? lds_mat(3 + wave) : mm::load_mat(as_global(A.fwd_d), (b << W) + d_h, lane);
        mm::apply<mm::CANON>(m, r0, r0);
        mm::apply<mm::CANON>(m, r1, r1);
      }
      const BufCol p(ld_uniform(A.lde, col) + ((size_t)b << A.n) + tile_word);
#pragma unroll
      for (uint32_t e = 0; e < 8; e++) p.store2<NT>(r0[e], r1[e], d_word, e << 13);
    }
  }
}

// ---- host ------------------------------------------------------------------------
// matrices of one direction over a domain of log_n: layers 4..7, 8..(contig - 1), then (strided
// layers k > 0) 12..15 and 16..(11 + k)
struct Tables {
  uint32_t b, c, d, e, total;  // first matrix of each stage
};
static Tables table_layout(uint32_t log_n, uint32_t contig, uint32_t k) {
  Tables t{};
  uint32_t at = 0;
  t.b = at;
  at += 1u << (log_n - 8);
  t.c = at;
  at += 1u << (log_n - contig);
  t.d = at;
  if (k) at += 1u << (log_n - 16);
  t.e = at;
  if (k) at += 1u << (log_n - 12 - k);
  t.total = at;
  return t;
}

// appends the stages of one direction at matrix `first` of the table
static void add_stages(MatArgs& A, bool inverse, const uint32_t* tw, uint32_t log_n, uint32_t contig, uint32_t k,
                       uint32_t first) {
  const Tables t = table_layout(log_n, contig, k);
  const uint32_t inv = inverse ? 1 : 0, scale = inverse ? 31 - log_n : 0;
  A.st[A.n_stages++] = {tw, log_n, inv, 4, 4, first + t.b, 0};
  A.st[A.n_stages++] = {tw, log_n, inv, 8, contig - 8, first + t.c, k ? 0u : scale};
  if (k) {
    A.st[A.n_stages++] = {tw, log_n, inv, 12, 4, first + t.d, 0};
    A.st[A.n_stages++] = {tw, log_n, inv, 16, k - 4, first + t.e, scale};
  }
}
static void build(const MatArgs& A, uint32_t total) {
  timed("fft_matrices", [&] { matrix_kernel<<<ceil_div(total, MB), 256, 0, ctx().cur>>>(A, total); });
}

// Streaming accesses where the columns are far larger than the caches (256 columns of log 20 and
// 21: contiguous passes 0.45 -> 0.43 and 0.99 -> 0.96 ms, middle pass 0.92 -> 0.90 ms); smaller
// batches are read back from the cache by the next pass.
static bool streaming(uint64_t values) { return values >= (1ull << 27); }

template <bool INV, int K, int NS>
static void launch_contig_ns(const ContigArgs& A, uint32_t blocks) {
  if (streaming((uint64_t)A.n_cols << A.log_n))
    contig_matrix_kernel<INV, K, NS, true><<<blocks, CT, 0, ctx().cur>>>(A);
  else
    contig_matrix_kernel<INV, K, NS, false><<<blocks, CT, 0, ctx().cur>>>(A);
}
template <bool INV, int K>
static void launch_contig_k(const ContigArgs& A, uint32_t blocks, uint32_t blowup) {
  if constexpr (!INV) {
    if (blowup == 1) return launch_contig_ns<INV, K, 4>(A, blocks);
    if (blowup == 2) return launch_contig_ns<INV, K, 2>(A, blocks);
    if (blowup == 3) return launch_contig_ns<INV, K, 1>(A, blocks);
  }
  launch_contig_ns<INV, K, 8>(A, blocks);
}

// blowup (forward, log_n = K): the source columns hold 2^(K - blowup) coefficients
template <bool INV>
static void launch_contig(const uint32_t* const* src, uint32_t* const* dst, uint32_t n_cols, uint32_t log_n,
                          uint32_t blowup, uint32_t K, const uint32_t* tw, const unsigned char* mats, uint32_t k) {
  const Tables t = table_layout(log_n, K, k);
  ContigArgs A{};
  A.src = src;
  A.dst = dst;
  A.tw = tw;
  A.mat_b = mats + (size_t)t.b * mm::MAT_BYTES;
  A.mat_c = mats + (size_t)t.c * mm::MAT_BYTES;
  A.n_cols = n_cols;
  A.log_n = log_n;
  A.tiles_log = log_n - K;
  A.n_groups = ceil_div(n_cols, 1u << (13 - K));
  // (interpolation in place of whole columns within the caches: a block's stores go where its next
  // loads would come from, and one group a block is faster, 6144 columns of 2^12 47.3 us against 50.4 in
  // one round, 8192 of 2^12 60.4 / 63.0, 10240 74.4 / 74.9)
  const bool single = INV && src == (const uint32_t* const*)dst && A.tiles_log == 0 && A.n_groups <= 8 * 512;
  A.per_block = single ? 1 : groups_per_block(A.n_groups, 1ull << A.tiles_log, 512);
  const uint32_t blocks = ceil_div(A.n_groups, A.per_block) << A.tiles_log;
  timed(INV ? (log_n == K ? "fft_inv_tile" : "fft_inv_contig") : (log_n == K ? "fft_fwd_tile" : "fft_fwd_contig"), [&] {
    if (K == 12)
      launch_contig_k<INV, 12>(A, blocks, blowup);
    else if (K == 11)
      launch_contig_k<INV, 11>(A, blocks, blowup);
    else
      launch_contig_k<INV, 10>(A, blocks, blowup);
  });
}

size_t tile_matrix_bytes(uint32_t log_n) { return (size_t)table_layout(log_n, log_n, 0).total * mm::MAT_BYTES; }
void tile_matrices(bool inverse, uint32_t log_n, const uint32_t* tw, unsigned char* mats) {
  MatArgs A{};
  A.out = mats;
  add_stages(A, inverse, tw, log_n, log_n, 0, 0);
  build(A, table_layout(log_n, log_n, 0).total);
}
void interpolate_tiles(const uint32_t* const* src, uint32_t* const* dst, uint32_t n_cols, uint32_t log_n,
                       const uint32_t* itw, unsigned char* mats) {
  launch_contig<true>(src, dst, n_cols, log_n, 0, log_n, itw, mats, 0);
}
void evaluate_tiles(const uint32_t* const* src, uint32_t* const* dst, uint32_t n_cols, uint32_t src_log, uint32_t log_n,
                    const uint32_t* tw, unsigned char* mats) {
  launch_contig<false>(src, dst, n_cols, log_n, log_n - src_log, log_n, tw, mats, 0);
}

template <int K>
static void launch_lde(const StridedArgs& S, uint32_t blocks) {
  const bool nt = streaming((uint64_t)S.n_cols << S.n);
  if (S.n_blocks == 2 && nt)
    lde_matrix_kernel<K, true, true><<<blocks, LT, 0, ctx().cur>>>(S);
  else if (S.n_blocks == 2)
    lde_matrix_kernel<K, true, false><<<blocks, LT, 0, ctx().cur>>>(S);
  else if (nt)
    lde_matrix_kernel<K, false, true><<<blocks, LT, 0, ctx().cur>>>(S);
  else
    lde_matrix_kernel<K, false, false><<<blocks, LT, 0, ctx().cur>>>(S);
}

// From 48 million (2^20) values on, where the matrices' launch is made up for.  Time here / on
// butterflies (fused schedule) at 32, 48 and 96 million values, blowup 2 | 4 | 8:
//   log 17   1.05 1.00 0.93 | 1.04 1.00 0.97 | 0.99 0.96 0.95
//   log 18   1.06 0.99 0.92 | 1.01 0.97 0.94 | 0.94 0.92 0.92
//   log 19   0.98 0.94 0.88 | 0.98 0.91 0.90 | 0.92 0.89 0.90
//   log 20   0.96 0.92 0.86 | 0.97 0.91 0.88 | 0.92 0.88 0.86
// and at 48 million and blowup 32 1.00, 0.95, 0.92, 0.91; the autotuner tries it from half of that.
// Log 17 to 20 are the sizes whose middle pass is one launch: stage E needs a fifth strided layer,
// and a ninth would leave its tiles runs of 128 bytes (which cost log 20 1.23 ms instead of 0.98).
bool use_matrices_lde(uint32_t n, uint32_t log_blowup, uint64_t n_cols) {
  return n >= 17 && n <= 20 && log_blowup >= 1 && (n_cols << n) >= (3ull << 24);
}
size_t lde_matrix_bytes(uint32_t n, uint32_t log_blowup) {
  const uint32_t k = n - 12;
  return (size_t)(table_layout(n, 12, k).total + table_layout(n + log_blowup, 12, k).total) * mm::MAT_BYTES;
}
void lde_matrices(const uint32_t* const* src, uint32_t* const* coeffs, uint32_t* const* lde, uint32_t n_cols, uint32_t n,
                  uint32_t log_blowup, const uint32_t* tw, const uint32_t* itw, unsigned char* mats) {
  const uint32_t m = n + log_blowup, k = n - 12;
  const Tables ti = table_layout(n, 12, k), tf = table_layout(m, 12, k);
  unsigned char* const fm = mats + (size_t)ti.total * mm::MAT_BYTES;
  MatArgs M{};
  M.out = mats;
  add_stages(M, true, itw, n, 12, k, 0);
  add_stages(M, false, tw, m, 12, k, ti.total);
  build(M, ti.total + tf.total);
  launch_contig<true>(src, coeffs, n_cols, n, 0, 12, itw, mats, k);
  StridedArgs S{};
  S.coeffs = coeffs;
  S.lde = lde;
  S.inv_d = mats + (size_t)ti.d * mm::MAT_BYTES;
  S.inv_e = mats + (size_t)ti.e * mm::MAT_BYTES;
  S.fwd_d = fm + (size_t)tf.d * mm::MAT_BYTES;
  S.fwd_e = fm + (size_t)tf.e * mm::MAT_BYTES;
  S.n_cols = n_cols;
  S.n = n;
  S.n_blocks = 1u << log_blowup;
  S.tiles_log = k - 2;  // 2^12 words between the layer bits, 2^(14 - k) to a tile
  S.per_block = groups_per_block(n_cols, 1ull << S.tiles_log, 256);
  const uint32_t blocks = ceil_div(n_cols, S.per_block) << S.tiles_log;
  timed("fft_lde_strided", [&] {
    if (k == 8)
      launch_lde<8>(S, blocks);
    else if (k == 7)
      launch_lde<7>(S, blocks);
    else if (k == 6)
      launch_lde<6>(S, blocks);
    else
      launch_lde<5>(S, blocks);
  });
  launch_contig<false>((const uint32_t* const*)lde, lde, n_cols, m, 0, 12, tw, fm, k);
}

}  // namespace fft
}  // namespace sh
