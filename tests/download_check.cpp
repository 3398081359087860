// Host side of the runtime's copies (runtime.hip compiled in, over the stub of the HIP runtime):
// prints for each case whether the copy's stream was waited for after the copy.
#include "hip_stub.hpp"
#include "../stwo-gpu_amd/csrc/runtime.hip"

static bool waited_for(hipStream_t s) {
  for (hipStream_t w : stub::waited)
    if (w == s) return true;
  return false;
}

int main() {
  if (stwo_hip_init(0) != STWO_HIP_OK) return 2;
  sh::Context& x = sh::ctx();
  void *a = nullptr, *b = nullptr;
  static char host[1 << 20];
  if (stwo_hip_malloc(&a, 1 << 20) || stwo_hip_malloc(&b, 1 << 20)) return 2;
  // a copy complete on return, on the library's stream and on another that is current
  for (hipStream_t s : {x.stream, x.aux[0]}) {
    x.cur = s;
    struct {
      void *dst, *src;
      size_t bytes;
    } cases[] = {{host, a, 32}, {host, a, 1 << 20}, {b, a, 4096}, {host, a, 7}};
    for (auto& c : cases) {
      stub::copies.clear();
      stub::waited.clear();
      stub::launched.clear();
      sh::download(c.dst, c.src, c.bytes);
      const bool copied = stub::copies.size() == 1 ? stub::copies[0].stream == s : stub::find("download_kernel") >= 0;
      printf("%d%d ", copied, waited_for(s));
    }
    printf("\n");
  }
  x.cur = x.stream;
  // a synchronous copy of nothing still waits for the library's work
  stub::waited.clear();
  if (stwo_hip_memcpy(host, a, 0)) return 2;
  printf("%d\n", waited_for(x.stream));
  return 0;
}
