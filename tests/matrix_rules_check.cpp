// The host rules of the matrix-core FFT passes (fft_matrix.hpp) on the command line:
//   split N_GROUPS TILES FILL   groups per block
//   tile LOG_N N_COLS KIND      whether whole small columns take the matrix cores; KIND: log blowup of an
//                               evaluation, 8 an inverse, 16 more for in place
// one query per line of the input, one answer per line of the output.
#include <cstdio>
#include <cstring>
#include "fft_matrix.hpp"
int main() {
  char what[32];
  unsigned long long a, b, c;
  while (scanf("%31s %llu %llu %llu", what, &a, &b, &c) == 4)
    if (!strcmp(what, "split"))
      printf("%u\n", sh::fft::groups_per_block(a, b, (uint32_t)c));
    else if (!strcmp(what, "tile"))
      printf("%d\n", sh::fft::use_matrices_tile((uint32_t)a, b, (c & 8) != 0, (uint32_t)c & 7, (c & 16) != 0) ? 1 : 0);
  return 0;
}
