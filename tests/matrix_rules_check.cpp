// The host rules of the matrix-core FFT passes (fft_matrix.hpp) on the command line:
//   split N_GROUPS TILES FILL   groups per block
// one query per line of the input, one answer per line of the output.
#include <cstdio>
#include <cstring>
#include "fft_matrix.hpp"
int main() {
  char what[32];
  unsigned long long a, b, c;
  while (scanf("%31s %llu %llu %llu", what, &a, &b, &c) == 4)
    if (!strcmp(what, "split")) printf("%u\n", sh::fft::groups_per_block(a, b, (uint32_t)c));
  return 0;
}
