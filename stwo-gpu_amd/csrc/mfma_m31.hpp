// M31 linear maps on the integer matrix cores (v_mfma_i32_32x32x32_i8).
//
// A value x is written in four signed digits of base 2^8, x = sum_j d_j 2^(8j) (mod P), one
// byte each.  A product by a fixed matrix entry e is then linear in the digits:
//   e x = sum_j d_j (e 2^(8j) mod P),
// and with e 2^(8j) mod P itself in four signed digits (limbs i) every limb of the result is
// one integer dot product over (input, digit j).  So a 16 x 16 matrix over M31 is a 64 x 64
// matrix of bytes (rows: output and limb, columns: input and digit), four 32x32x32
// instructions for 32 vectors, and an output is put together from its four limb sums:
// 8 or 9 VALU instructions per value (limb sums to digits, or to a canonical value)
// for whatever the matrix does, where four butterfly layers cost 24.
//
// Register layout of a tile of 32 vectors n of 16 values m (the layout is the same on both
// sides of the instruction, so tiles chain): lane n + 32 g holds m = 2 slot + g, slot 0..7.
// The matrix is the A operand: chunk (T, s) holds output rows 8T .. 8T + 7 and input slots
// 4s .. 4s + 3; lane row + 32 g holds row (output 8T + row / 4, limb row % 4) and, in byte
// 4i + j, digit j of input m = 2 (4s + i) + g.  The accumulator's registers 4q .. 4q + 3 of
// lane n + 32 g are then the four limbs of output m = 8T + 2q + g.
//
// Bounds.  Digits and limbs lie in [-128, 127], so a sum of 64 products lies within 2^20.
#pragma once
#include "field.hpp"
#include "gmem.hpp"

namespace sh {
namespace mm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr uint32_t MAT_BYTES = 4096;  // one 16 x 16 matrix: 4 chunks of 64 lanes x 16 bytes

// x (any value below 2^32 - 2^24, taken mod P) to its four signed digits: x - P fits a signed
// word, whose top byte is signed already; adding 0x80 to the other bytes carries, flipping
// their top bits leaves them signed
__host__ __device__ __forceinline__ uint32_t digits(uint32_t x) { return (x + (0x00808080u - P)) ^ 0x00808080u; }
// limbs of a matrix entry (canonical): centred, then as above; |top limb| <= 64
__host__ __device__ __forceinline__ uint32_t limbs(uint32_t e) {
  const uint32_t c = e > P / 2 ? e - P : e;
  return (c + 0x00808080u) ^ 0x00808080u;
}
// e 2^s mod P for canonical e, 0 <= s < 31
__host__ __device__ __forceinline__ uint32_t rot31(uint32_t e, uint32_t s) {
  return s ? (((e << s) & P) | (e >> (31 - s))) : e;
}

// limb sums to a value below 2^31 + 2^30 + 2^29, exact mod P: the upper two limbs are worth 2^16
// each unit, and of that product the bits from 2^31 on count once more at the bottom.  The sums
// are signed: H makes the upper part nonnegative, and C = -2^16 H (mod P) takes it out again and
// keeps the total between 0 and 2^32.
constexpr uint32_t JOIN_H = (1u << 28) + (1u << 20) + (1u << 14);
constexpr uint32_t JOIN_C = P - (uint32_t)(((uint64_t)JOIN_H << 16) % P);
static_assert(JOIN_C >= (1u << 28) + (1u << 20) && JOIN_C < (1u << 30) + (1u << 28), "join stays within 32 bits");
// What becomes of a joined value: DIGITS its digit word (the operand of the next map), CANON its
// canonical residue.
enum Out { DIGITS, CANON };
// keeps the sum formed so far as it is: left to itself the compiler regroups the sums below so
// that no shift fuses with an addition (10 instructions instead of 8 or 9)
// (constants in scalar registers: a three-operand addition takes no literal)
#if defined(__HIP_DEVICE_COMPILE__)
#define SH_MM_KEEP(x) asm("" : "+v"(x))
#define SH_MM_SCALAR(x) asm("" : "+s"(x))
#else
#define SH_MM_KEEP(x) (void)0
#define SH_MM_SCALAR(x) (void)0
#endif
template <Out OUT>
__host__ __device__ __forceinline__ uint32_t join(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3) {
  uint32_t lo = a0 + (a1 << 8), hi = a2 + (a3 << 8);
  SH_MM_KEEP(lo);
  SH_MM_KEEP(hi);
  hi += JOIN_H;
  uint32_t part = hi & 0x7fffu;
  SH_MM_KEEP(part);
  lo += part << 16;
  SH_MM_KEEP(lo);
  hi >>= 15;
  if constexpr (OUT == DIGITS) {  // digits(lo + hi + C)
    uint32_t c = JOIN_C + (0x00808080u - P);
    SH_MM_SCALAR(c);
    return (lo + hi + c) ^ 0x00808080u;
  } else {
    uint32_t c = JOIN_C;
    SH_MM_SCALAR(c);
    uint32_t x = lo + hi + c;  // <= 2P
    SH_MM_KEEP(x);
    return canon(x);
  }
}

// The limb rows of four entries c[0..3] of a matrix operand: row 4 k + i of the rows from q on
// (16 bytes apart) gets, in its word, limb i of c[k] 2^(8j) for the digits j.
__host__ __device__ __forceinline__ void operand_rows(const uint32_t (&c)[4], uint32_t* q) {
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) {
    uint32_t w[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) w[j] = limbs(rot31(c[k], 8 * j));
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
      uint32_t b = 0;
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) b |= ((w[j] >> (8 * i)) & 0xff) << (8 * j);
      q[4 * (4 * k + i)] = b;
    }
  }
}
// limb sums of many products (each |sum| <= 2^29: up to 2^13 terms of 4 digits) to the canonical
// value: exact in 64 bits, made nonnegative by 2^23 P
__host__ __device__ __forceinline__ uint32_t join64(int a0, int a1, int a2, int a3) {
  const int64_t v = ((((((int64_t)a3 << 8) + a2) << 8) + a1) << 8) + a0;
  const uint64_t u = (uint64_t)(v + ((int64_t)P << 23));  // < 2^55
  return canon((uint32_t)(u & P) + (uint32_t)(u >> 31));
}

struct Mat {
  v4i c[4];  // chunks (T, s) at 2T + s
};
// matrix `index` of a table of matrices (index uniform)
__device__ __forceinline__ Mat load_mat(const SH_GLOBAL unsigned char* table, uint32_t index, uint32_t lane) {
  Mat m;
  const SH_GLOBAL v4i* p = (const SH_GLOBAL v4i*)(table + (size_t)index * MAT_BYTES);
#pragma unroll
  for (int k = 0; k < 4; k++) m.c[k] = p[64 * k + lane];
  return m;
}

// the map applied to a tile: digit words in, values as join<OUT> gives them out (both by slot).
// NS: input slots from NS on are zero.
template <Out OUT, int NS = 8>
__device__ __forceinline__ void apply(const Mat& m, const uint32_t* d, uint32_t* out) {
#if defined(__HIP_DEVICE_COMPILE__)
  v4i b0 = {}, b1 = {};
#pragma unroll
  for (int e = 0; e < 4; e++) {
    if (e < NS) b0[e] = (int)d[e];
    if (4 + e < NS) b1[e] = (int)d[4 + e];
  }
#pragma unroll
  for (int t = 0; t < 2; t++) {
    v16i acc = {};
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(m.c[2 * t], b0, acc, 0, 0, 0);
    if constexpr (NS > 4) acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(m.c[2 * t + 1], b1, acc, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 4; q++)
      out[4 * t + q] = join<OUT>((uint32_t)acc[4 * q], (uint32_t)acc[4 * q + 1], (uint32_t)acc[4 * q + 2],
                            (uint32_t)acc[4 * q + 3]);
    // one accumulator at a time, joined at once (not sunk to the outputs' uses): with several in
    // flight the kernels' registers spill, and the other waves fill the wait
#pragma unroll
    for (int q = 0; q < 4; q++) asm volatile("" : "+v"(out[4 * t + q]));
    __builtin_amdgcn_sched_barrier(0);
  }
#endif
}

}  // namespace mm
}  // namespace sh
