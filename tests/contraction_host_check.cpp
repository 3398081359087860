// Host build of the arithmetic of the long contractions on the matrix cores (mfma_m31.hpp).  Reads rows
// of four words:
//   limb sums a0..a3 (signed)  -> join64 of them
//   four entries c[0..3]       -> the 16 operand rows of operand_rows
// and writes for each row the joined value and 16 words.
#include <cstdint>
#include <cstdio>
#include "mfma_m31.hpp"
using namespace sh;
int main() {
  int32_t a[4];
  while (fread(a, 4, 4, stdin) == 4) {
    uint32_t out[17];
    out[0] = mm::join64(a[0], a[1], a[2], a[3]);
    uint32_t rows[64] = {};
    const uint32_t c[4] = {(uint32_t)a[0] % P, (uint32_t)a[1] % P, (uint32_t)a[2] % P, (uint32_t)a[3] % P};
    mm::operand_rows(c, rows);
    for (int i = 0; i < 16; i++) out[1 + i] = rows[4 * i];
    fwrite(out, 4, 17, stdout);
  }
  return 0;
}
