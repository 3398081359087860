// Host build of the matrix-core arithmetic (mfma_m31.hpp): digits, limbs and join, with the limb
// sums formed in plain integers.  Reads "m x[0..15] e[0..15]" rows as words, writes for each row
// the value that the path gives for sum_i e[i] x[i] and the join's unreduced bounds check.
#include <cstdio>
#include <cstdint>
#include "mfma_m31.hpp"
using namespace sh;
int main() {
  uint32_t x[16], e[16];
  while (fread(x, 4, 16, stdin) == 16 && fread(e, 4, 16, stdin) == 16) {
    int64_t a[4] = {0, 0, 0, 0};
    for (int m = 0; m < 16; m++) {
      const uint32_t d = mm::digits(x[m]);
      for (int j = 0; j < 4; j++) {
        const uint32_t w = mm::limbs(mm::rot31(e[m], 8 * j));
        for (int i = 0; i < 4; i++) a[i] += (int64_t)(int8_t)(d >> (8 * j)) * (int8_t)(w >> (8 * i));
      }
    }
    uint32_t out[4] = {0, 0, 0, 1};
    for (int i = 0; i < 4; i++) out[3] &= a[i] >= -(1 << 20) && a[i] <= (1 << 20);
    out[0] = mm::join<mm::CANON>((uint32_t)a[0], (uint32_t)a[1], (uint32_t)a[2], (uint32_t)a[3]);
    out[1] = mm::join<mm::DIGITS>((uint32_t)a[0], (uint32_t)a[1], (uint32_t)a[2], (uint32_t)a[3]);
    out[2] = mm::digits(out[0]);
    fwrite(out, 4, 4, stdout);
  }
  return 0;
}
