// Twiddle trees: PolyOps::precompute_twiddles (stwo_gpu_backend/src/poly.rs:170-192).
//
// Tree layout (cuda/src/poly/twiddles.cu:29-73): for the coset doubled j times
// (j = 0, 1, ...), the x coordinates of its first half in bit-reversed order,
// one level after another, then a trailing 1 (so the tree has coset.size()
// entries).  The inverse tree is the element-wise inverse (poly.rs:180-185).
//
// Here one launch fills every level (the reference launches once per level), and
// the extension entry point caches trees per coset so a prover computes each once.
#include "field.hpp"
#include "runtime.hpp"

namespace sh {
void batch_inverse_m31(const uint32_t* src, uint32_t* dst, uint64_t n);  // batch_inverse.hip

namespace tw {

// Level 0 holds the x of initial + step * brev(i): bit b of i contributes the fixed point
// weight[b] = step * 2^(half_log - 1 - b), so a thread multiplies the weights of its set bits
// and then takes its 4 or 16 values from one product each with as many uniform points.  The level above
// needs no points: brev(2i) over one more bit is brev(i), so entry i of level j + 1 is the
// doubling x -> 2x^2 - 1 of entry 2i of level j, and a block that owns 2^B consecutive values
// (B = 10 or 12) of level 0 owns 2^(B-1) of level 1, ... , one of level B, and, where its index is a
// multiple of 2^z, one of levels B + 1 .. B + z.  Bound by the latency of the products and of the
// doublings (2^22: 103 -> 13.8 us against a full power of the step per entry, which took 2 x 31
// products each; the stores alone take 3 us).
constexpr uint32_t TREE_NT = 256;
// Blocks of 2^12 values (trees from 2^21 on fill their four groups of 2^10), or of 2^10: a quarter of the chain of products and doublings and four times
// the blocks, for trees up to 2^20 (a call with the inverses: 2^14 25.2 us with the small blocks, 28.3
// with the large; 2^20 28.5 / 31.2; 2^21 33.6 / 33.4; 2^22 43.6 / 39.5; a power per entry took 25.4,
// 46, 70 and 120).
constexpr uint32_t TREE_SMALL_MAX = 20;

struct TreeArgs {
  pt initial;
  pt weight[30];  // identity from half_log on
  pt lane16[16];  // sum of the weights of bits 0, 1, 10, 11 selected by the index's bits
};

template <uint32_t BLOCK_LOG>
__global__ __launch_bounds__(TREE_NT) void tree_kernel(uint32_t* __restrict__ out, TreeArgs A, uint32_t log_size) {
  const uint32_t size = 1u << log_size, half_log = log_size - 1, half = size >> 1;  // log_size >= 1
  const uint32_t t = threadIdx.x, blk = blockIdx.x;
  if (blk == 0 && t == 0) out[size - 1] = 1;
  pt q = A.initial;
  for (uint32_t b = BLOCK_LOG; b < half_log; b++)  // uniform
    if ((blk >> (b - BLOCK_LOG)) & 1) q = pmul(q, A.weight[b]);
#pragma unroll
  for (int b = 0; b < 8; b++) {
    if (b + 2 >= (int)half_log) break;  // uniform: a small tree has fewer index bits
    const pt r = pmul(q, A.weight[b + 2]);
    if ((t >> b) & 1) q = r;
  }
  // value c of group k: index i = blk 2^BLOCK_LOG + 2^10 k + 4 t + c (blocks of several groups are for
  // trees that fill them; of a single group that is more than the tree, values past half are not stored)
  constexpr int GROUPS = 1 << (BLOCK_LOG - 10);
  uint32_t x[GROUPS][4];
#pragma unroll
  for (int k = 0; k < GROUPS; k++)
#pragma unroll
    for (int c = 0; c < 4; c++) x[k][c] = pmul(q, A.lane16[4 * k + c]).x;
  auto twice = [](uint32_t v) { return sub(canon(2 * sqr(v)), 1); };
  // level j starts at size - (size >> j); j <= 2: 4, 2, 1 values per thread and group
#pragma unroll
  for (int k = 0; k < GROUPS; k++) {
    const uint32_t i = (blk << BLOCK_LOG) + (k << 10) + 4 * t;
#pragma unroll
    for (int j = 0; j < 3; j++) {
      uint32_t* lvl = out + (size - (size >> j));
#pragma unroll
      for (int c = 0; c < (4 >> j); c++)
        if (i + ((uint32_t)c << j) < half && log_size > (uint32_t)j) lvl[(i >> j) + c] = x[k][c];
#pragma unroll
      for (int c = 0; c < (4 >> (j + 1)); c++) x[k][c] = twice(x[k][2 * c]);
      if (j == 2) x[k][0] = twice(x[k][0]);
    }
  }
#pragma unroll 1
  for (uint32_t j = 3; j < 10; j++) {
    if (j >= log_size) return;  // uniform
    uint32_t* lvl = out + (size - (size >> j));
#pragma unroll
    for (int k = 0; k < GROUPS; k++) {
      const uint32_t i = (blk << BLOCK_LOG) + (k << 10) + 4 * t;
      if ((t & ((1u << (j - 2)) - 1)) == 0 && i < half) lvl[i >> j] = x[k][0];
      x[k][0] = twice(x[k][0]);
    }
  }
  if (t) return;
  // levels 10 .. : the block's values 2^10 k, then its first value alone
#pragma unroll 1
  for (uint32_t j = 10; j < log_size; j++) {
    uint32_t* lvl = out + (size - (size >> j));
#pragma unroll
    for (int k = 0; k < GROUPS; k++) {
      const uint32_t i = (blk << BLOCK_LOG) + (k << 10);
      if ((i & ((1u << j) - 1)) == 0 && i < half) lvl[i >> j] = x[k][0];
      x[k][0] = twice(x[k][0]);
    }
    if (j >= BLOCK_LOG && (blk & ((2u << (j - BLOCK_LOG)) - 1))) return;
  }
}

__global__ void one_kernel(uint32_t* out) { out[0] = 1; }

void compute_tree(uint32_t* out, pt initial, pt step, uint32_t log_size) {
  if (log_size == 0) {  // a coset of one point: the trailing 1 alone
    timed("twiddle_tree", [&] { one_kernel<<<1, 1, 0, ctx().cur>>>(out); });
    return;
  }
  TreeArgs A;
  A.initial = initial;
  const uint32_t half_log = log_size - 1;
  pt w = step;
  for (uint32_t b = 0; b < 30; b++) A.weight[b] = pt{1, 0};
  for (uint32_t b = half_log; b-- > 0; w = pmul(w, w)) A.weight[b] = w;  // weight[half_log - 1] = step
  A.lane16[0] = pt{1, 0};
  const uint32_t bit[4] = {0, 1, 10, 11};
  for (uint32_t b = 0; b < 4; b++)
    for (uint32_t s = 0; s < (1u << b); s++)
      A.lane16[s + (1u << b)] = bit[b] < half_log ? pmul(A.lane16[s], A.weight[bit[b]]) : A.lane16[s];
  const uint32_t block_log = log_size <= TREE_SMALL_MAX ? 10 : 12;
  const uint32_t blocks = half_log > block_log ? 1u << (half_log - block_log) : 1u;
  timed("twiddle_tree", [&] {
    (block_log == 10 ? tree_kernel<10> : tree_kernel<12>)<<<blocks, TREE_NT, 0, ctx().cur>>>(out, A, log_size);
  });
}

}  // namespace tw
}  // namespace sh

using namespace sh;

extern "C" uint32_t* precompute_twiddles(StwoCirclePointM31 initial, StwoCirclePointM31 step, size_t total_size) {
  uint32_t* out = nullptr;
  guarded([&] {
    require(is_pow2(total_size) && total_size >= 1 && total_size <= (1ull << 30),
            "precompute_twiddles: size must be a power of two");
    out = (uint32_t*)ctx().pool.alloc(total_size * 4);
    tw::compute_tree(out, pt{initial.x, initial.y}, pt{step.x, step.y}, log2_exact(total_size));
    sync();
  });
  return out;
}

extern "C" int stwo_hip_twiddles(uint32_t initial_index, uint32_t step_size, uint32_t log_size,
                                 const uint32_t** twiddles, const uint32_t** itwiddles) {
  return guarded([&] {
    require(log_size <= 30, "stwo_hip_twiddles: log size too large");
    TwiddleKey key{initial_index & 0x7fffffffu, step_size & 0x7fffffffu, log_size};
    auto& cache = ctx().twiddles;
    auto it = cache.find(key);
    if (it == cache.end()) {
      uint64_t size = 1ull << log_size;
      TwiddleEntry e;
      e.tw = (uint32_t*)ctx().pool.alloc(size * 4);
      e.itw = (uint32_t*)ctx().pool.alloc(size * 4);
      tw::compute_tree(e.tw, point_at_index(key.initial), point_at_index(key.step), log_size);
      batch_inverse_m31(e.tw, e.itw, size);
      // the cached tree is shared by work on every stream: finish it before handing it out
      hip_check(hipStreamSynchronize(ctx().cur), "hipStreamSynchronize");
      it = cache.emplace(key, e).first;
    }
    *twiddles = it->second.tw;
    *itwiddles = it->second.itw;
  });
}

extern "C" int stwo_hip_release_twiddles(void) {
  return guarded([] {
    sync();
    // proof-server jobs on the slot streams read the cached tables too: wait for every
    // stream, so that no block handed back to the pool here is still being read (new jobs
    // are enqueued under the library lock and fetch the tables again)
    hip_check(hipDeviceSynchronize(), "hipDeviceSynchronize");
    for (auto& kv : ctx().twiddles) {
      ctx().pool.free(kv.second.tw);
      ctx().pool.free(kv.second.itw);
    }
    ctx().twiddles.clear();
    for (auto& kv : ctx().domain_tables) ctx().pool.free(kv.second);
    ctx().domain_tables.clear();
  });
}
