// Column operations: ColumnOps::bit_reverse_column (stwo_gpu_backend/src/column.rs:10-34),
// PolyOps::new_canonical_ordered (poly.rs:23-33) and AccumulationOps::accumulate
// (accumulation.rs:9-19).
//
// bit_reverse: the reference swaps a[i] <-> a[brev(i)] one element per thread
// (cuda/src/bit_reverse.cu:6-16), which scatters every access.  Here an index
// is split into [hi a bits | mid | lo a bits]; brev maps (hi, mid, lo) to
// (brev lo, brev mid, brev hi), so the 2^a x 2^a tile at `mid` and the tile at
// brev(mid) exchange places as a bit-reversed transpose through LDS, with
// 2^a-element contiguous runs on both the read and the write side.
#include "field.hpp"
#include "gmem.hpp"
#include "runtime.hpp"

namespace sh {
namespace cols {

// tile = 2^TA x 2^TA elements for the smaller columns: 64 x 64 for M31 (256-byte runs) below
// 2^14 values, 32 x 32 for QM31 (512-byte runs) below 2^12 values
template <class T>
constexpr int tile_bits() {
  return sizeof(T) == 4 ? 6 : 5;
}

constexpr uint32_t BR_NT = 256;
// 4-byte elements: 64 x 64 tiles, every load of a thread in flight before its LDS stores
template <class T>
__global__ __launch_bounds__(BR_NT) void bitrev_tiled_kernel(T* a, uint32_t log_n) {
  constexpr int TA = tile_bits<T>();
  // LDS rows padded by one element, so the transposed reads hit distinct banks
  constexpr uint32_t W = 1u << TA, RW = W + 1;
  constexpr int PER = (int)(W * W / BR_NT);     // elements per thread and tile
  __shared__ T ta[W * RW];
  __shared__ T tb[W * RW];
  const uint32_t mid_bits = log_n - 2 * TA;
  const uint32_t m = blockIdx.x;
  const uint32_t mr = brev(m, mid_bits);
  if (mr < m) return;  // the pair is handled by block mr
  const bool pair = mr != m;
  auto at = [&](uint32_t hi, uint32_t mid, uint32_t lo) -> size_t {
    return ((size_t)hi << (log_n - TA)) | ((size_t)mid << TA) | lo;
  };
  // every load of the thread is issued before the first LDS store
  T va[PER], vb[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const uint32_t e = threadIdx.x + BR_NT * k, hi = e >> TA, lo = e & (W - 1);
    va[k] = a[at(hi, m, lo)];
    if (pair) vb[k] = a[at(hi, mr, lo)];
  }
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const uint32_t e = threadIdx.x + BR_NT * k, hi = e >> TA, lo = e & (W - 1);
    ta[hi * RW + lo] = va[k];
    if (pair) tb[hi * RW + lo] = vb[k];
  }
  __syncthreads();
  // element (hi, m, lo) goes to (brev lo, mr, brev hi)
#pragma unroll
  for (int k = 0; k < PER; k++) {
    const uint32_t e = threadIdx.x + BR_NT * k, hi2 = e >> TA, lo2 = e & (W - 1);
    const uint32_t src = brev(lo2, TA) * RW + brev(hi2, TA);
    a[at(hi2, mr, lo2)] = ta[src];
    if (pair) a[at(hi2, m, lo2)] = tb[src];
  }
}

// 16-byte elements: 32 x 32 tiles (512-byte runs), unpadded LDS; measured faster with the
// loads interleaved with the LDS stores than with the 4-byte kernel's load-all-first loop
template <class T>
__global__ __launch_bounds__(BR_NT) void bitrev_tiled16_kernel(T* a, uint32_t log_n) {
  constexpr int TA = 5;
  constexpr uint32_t W = 1u << TA;
  __shared__ T ta[W * W];
  __shared__ T tb[W * W];
  const uint32_t mid_bits = log_n - 2 * TA;
  const uint32_t m = blockIdx.x;
  const uint32_t mr = brev(m, mid_bits);
  if (mr < m) return;  // the pair is handled by block mr
  auto at = [&](uint32_t hi, uint32_t mid, uint32_t lo) -> size_t {
    return ((size_t)hi << (log_n - TA)) | ((size_t)mid << TA) | lo;
  };
  for (uint32_t e = threadIdx.x; e < W * W; e += blockDim.x) {
    uint32_t hi = e >> TA, lo = e & (W - 1);
    ta[e] = a[at(hi, m, lo)];
    if (mr != m) tb[e] = a[at(hi, mr, lo)];
  }
  __syncthreads();
  // element (hi, m, lo) goes to (brev lo, mr, brev hi)
  for (uint32_t e = threadIdx.x; e < W * W; e += blockDim.x) {
    uint32_t hi2 = e >> TA, lo2 = e & (W - 1);
    uint32_t src = (brev(lo2, TA) << TA) | brev(hi2, TA);
    a[at(hi2, mr, lo2)] = ta[src];
    if (mr != m) a[at(hi2, m, lo2)] = tb[src];
  }
}

// Tile of block b: neighbouring places of the XCD order alternate between steps of m's lowest and
// of its highest bits, so the tiles that are under way together lie in runs both at m and at the
// mirrored brev(m).
__device__ __forceinline__ uint32_t mirrored_order(uint32_t mid_bits) {
  const uint32_t b = xcd_order();
  uint32_t m = 0;
  for (uint32_t k = 0; k < mid_bits; k++) m |= ((b >> k) & 1u) << ((k & 1) ? mid_bits - 1 - k / 2 : k / 2);
  return m;
}

// 4-byte elements in columns of at least 2^14 (BR_BIG): 128 x 128 tiles (512-byte runs), both tiles of the
// pair in registers and one padded LDS tile for the two transposes.  A wave's 16-byte accesses
// cover two rows.  Bound by the memory system: 2^28 values 591 -> 499 us (4.3 TB/s), where the
// same exchange of tiles without the transposes takes 460 and a pass over the tiles in place 390.
// 8 waves a block leave room for a second one beside it; 16 waves with 8-byte accesses, in the
// order of m, took 585, 64 x 64 tiles 620 or more, 256 x 256 tiles do not leave room for two
// blocks (780 for the exchange alone).
template <bool NT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void bitrev_big_kernel(uint32_t* a,
                                                                                                uint32_t log_n) {
  constexpr uint32_t TA = 7, W = 1u << TA, RW = W + 1;
  constexpr int PER = 8;  // 16-byte accesses per thread and tile
  __shared__ uint32_t t[W * RW];
  const uint32_t m = mirrored_order(log_n - 2 * TA), mr = brev(m, log_n - 2 * TA);
  if (mr < m) return;  // the pair is handled by the block of mr
  const bool pair = mr != m;
  // a wave's access: rows hi, hi + 1 (a half wave each) of the tile, hi = 2 wave + 16 k
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), half = (threadIdx.x >> 5) & 1,
                 l = threadIdx.x & 31;
  const uint32_t off = (half << (log_n - TA)) + 4 * l;
  typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(4)));
  auto row = [&](uint32_t mm, int k) {
    return (SH_GLOBAL u4*)((SH_GLOBAL char*)as_global(a + (((size_t)(2 * wave + 16 * k) << (log_n - TA)) | (mm << TA))) +
                           off * 4u);
  };
  u4 va[PER], vb[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    va[k] = NT ? __builtin_nontemporal_load(row(m, k)) : *row(m, k);
    if (pair) vb[k] = NT ? __builtin_nontemporal_load(row(mr, k)) : *row(mr, k);
  }
  uint32_t* const in = t + (2 * wave + half) * RW + 4 * l;
  // element (hi, m, lo) goes to (brev lo, mr, brev hi): row hi = 16 k + 2 wave + half, column
  // lo = 4 l + j of the result are column and row of the tile, reversed
  const uint32_t* const out = t + brev(l, 5) * RW + (half << 6) + (brev(wave, 3) << 3);
  auto turn = [&](const u4 (&v)[PER], uint32_t to) {
#pragma unroll
    for (int k = 0; k < PER; k++)
#pragma unroll
      for (int j = 0; j < 4; j++) in[16 * RW * k + j] = v[k][j];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int c = (k & 1) << 2 | (k & 2) | k >> 2;
      const u4 x = {out[c], out[64 * RW + c], out[32 * RW + c], out[96 * RW + c]};
      if (NT)
        __builtin_nontemporal_store(x, row(to, k));
      else
        *row(to, k) = x;
    }
  };
  turn(va, mr);
  if (!pair) return;
  __syncthreads();
  turn(vb, m);
}

// 16-byte elements in columns of at least 2^12: 64 x 64 tiles (1 KiB runs), the same way; LDS row
// r starts at element 64 r + r / 8, so the transposed reads of 8 consecutive lanes (rows 8 apart)
// fall in distinct bank groups.  2^26 values 570 -> 469 us (4.6 TB/s).
template <bool NT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void bitrev_big16_kernel(uint4* a,
                                                                                                  uint32_t log_n) {
  constexpr uint32_t TA = 6, W = 1u << TA;
  constexpr int PER = 8;  // elements per thread and tile
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  __shared__ u4 t[W * W + W / 8];
  const uint32_t m = mirrored_order(log_n - 2 * TA), mr = brev(m, log_n - 2 * TA);
  if (mr < m) return;  // the pair is handled by the block of mr
  const bool pair = mr != m;
  // a wave's access: row hi = wave + 8 k of the tile
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  auto row = [&](uint32_t mm, int k) {
    return (SH_GLOBAL u4*)as_global(a + (((size_t)(wave + 8 * k) << (log_n - TA)) | (mm << TA))) + lane;
  };
  auto lds_row = [](uint32_t r) { return r * W + (r >> 3); };
  u4 va[PER], vb[PER];
#pragma unroll
  for (int k = 0; k < PER; k++) {
    va[k] = NT ? __builtin_nontemporal_load(row(m, k)) : *row(m, k);
    if (pair) vb[k] = NT ? __builtin_nontemporal_load(row(mr, k)) : *row(mr, k);
  }
  u4* const in = t + wave * W + lane;
  // element (hi, m, lo) goes to (brev lo, mr, brev hi)
  const u4* const out = t + lds_row(brev(lane, TA)) + (brev(wave, 3) << 3);
  auto turn = [&](const u4 (&v)[PER], uint32_t to) {
#pragma unroll
    for (int k = 0; k < PER; k++) in[8 * W * k + k] = v[k];  // (lds_row(wave + 8 k): wave is below 8)
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const u4 x = out[(k & 1) << 2 | (k & 2) | k >> 2];
      if (NT)
        __builtin_nontemporal_store(x, row(to, k));
      else
        *row(to, k) = x;
    }
  };
  turn(va, mr);
  if (!pair) return;
  __syncthreads();
  turn(vb, m);
}

template <class T>
__global__ void bitrev_simple_kernel(T* a, uint32_t n, uint32_t log_n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t j = brev(i, log_n);
  if (j > i) {
    T t = a[i];
    a[i] = a[j];
    a[j] = t;
  }
}

// log of the 4-byte values from which the accesses are nontemporal (16-byte values: two less), the
// column being larger than the caches.  Nontemporal / plain: 2^27 M31 253 / 280 us, 2^26 135 / 92;
// 2^25 QM31 245 / 262, 2^24 138 / 95.
constexpr uint32_t BR_STREAM = 27;
// log of the 4-byte values from which 128 x 128 tiles fill the chip (256 blocks): below, a block that
// turns a pair of them is the longer chain, and 64 x 64 tiles are faster.  Large / small tiles: 2^16
// 15.7 / 14.2 us, 2^20 16.6 / 15.1, 2^21 17.1 / 16.3, 2^22 18.7 / 19.5, 2^24 34.9 / 39.9; columns off 16
// bytes 2^20 17.2 / 15.5, 2^22 19.4 / 21.8.  In 2^14 and 2^15 values no large tile has a partner: 14.0 / 14.1
// us, off 16 bytes 14.0 / 14.5.
constexpr uint32_t BR_BIG = 22;
template <class T>
void bit_reverse(T* a, uint64_t n) {
  require(is_pow2(n) && n <= (1ull << 31), "bit_reverse: size must be a power of two <= 2^31");
  uint32_t log_n = log2_exact(n);
  constexpr int TA = tile_bits<T>();
  if (log_n >= 2 * TA) {
    timed("bit_reverse", [&] {
      if constexpr (sizeof(T) == 4) {
        if (log_n >= BR_BIG || log_n == 14 || log_n == 15)
          (log_n >= BR_STREAM ? bitrev_big_kernel<true> : bitrev_big_kernel<false>)<<<1u << (log_n - 14), 512, 0,
                                                                                       ctx().cur>>>(a, log_n);
        else
          bitrev_tiled_kernel<T><<<1u << (log_n - 2 * TA), cols::BR_NT, 0, ctx().cur>>>(a, log_n);
      } else if (log_n >= 12)
        (log_n >= BR_STREAM - 2 ? bitrev_big16_kernel<true> : bitrev_big16_kernel<false>)<<<1u << (log_n - 12), 512, 0,
                                                                                         ctx().cur>>>(a, log_n);
      else
        bitrev_tiled16_kernel<T><<<1u << (log_n - 2 * TA), cols::BR_NT, 0, ctx().cur>>>(a, log_n);
    });
  } else if (n > 1) {
    timed("bit_reverse", [&] {
      bitrev_simple_kernel<T><<<ceil_div(n, 256), 256, 0, ctx().cur>>>(a, (uint32_t)n, log_n);
    });
  }
}

// canonic order -> circle-domain order: evens, then odds reversed (cuda/src/poly/twiddles.cu:4-15)
__global__ void sort_values_kernel(const uint32_t* from, uint32_t* dst, uint32_t n) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t half = n >> 1;
  dst[i] = i < half ? from[2 * i] : from[n - 1 - 2 * (i - half)];
}

struct Soa4 {
  uint32_t* c[4];
};
__global__ void accumulate_kernel(uint32_t n, Soa4 l, Soa4 r) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int k = 0; k < 4; k++) l.c[k][i] = add(l.c[k][i], r.c[k][i]);
}

// ---- gathers for Column::at and Merkle decommitment ----
// values[i * n_cols + c] = cols[c][rows[i]]: every queried row of every column in one
// launch (the reference copies a whole column to the host per element, column.rs:49-52).
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint32_t* const* __restrict__ cols, uint32_t n_cols,
                                                          const uint32_t* __restrict__ rows, uint64_t total,
                                                          uint32_t* __restrict__ out) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const uint32_t i = (uint32_t)(t / n_cols), c = (uint32_t)(t % n_cols);
  out[t] = cols[c][rows[i]];
}
struct Hash8 {
  uint32_t s[8];
};
// paths[q * depth + j] = the sibling, at layer depth - j, of the node on leaf q's path
// (j = 0 is the leaf's own sibling): the authentication path of MerkleProver::decommit.
__global__ __launch_bounds__(256) void auth_paths_kernel(const Hash8* const* __restrict__ layers, uint32_t depth,
                                                         const uint32_t* __restrict__ leaves, uint32_t total,
                                                         Hash8* __restrict__ out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const uint32_t q = t / depth, j = t % depth;
  out[t] = layers[depth - j][(leaves[q] >> j) ^ 1u];
}

}  // namespace cols
}  // namespace sh

using namespace sh;

extern "C" int stwo_hip_gather_rows(const uint32_t* const* columns, uint32_t n_cols, uint64_t column_size,
                                    const uint32_t* rows, uint32_t n_rows, uint32_t* values) {
  return guarded([&] {
    if (!n_cols || !n_rows) return;
    require(columns != nullptr && rows != nullptr && values != nullptr, "gather_rows: null argument");
    for (uint32_t i = 0; i < n_rows; i++) require(rows[i] < column_size, "gather_rows: row index out of range");
    const uint64_t total = (uint64_t)n_rows * n_cols;
    require(total <= (1ull << 31), "gather_rows: too many values");
    DevBuf table = upload(columns, n_cols * sizeof(void*));
    DevBuf drows = upload(rows, n_rows * sizeof(uint32_t));
    DevBuf out(total * sizeof(uint32_t));
    timed("gather_rows", [&] {
      cols::gather_rows_kernel<<<ceil_div(total, 256), 256, 0, ctx().cur>>>(table.as<const uint32_t*>(), n_cols,
                                                                            drows.as<uint32_t>(), total,
                                                                            out.as<uint32_t>());
    });
    hip_check(hipMemcpyAsync(values, out.p, total * sizeof(uint32_t), hipMemcpyDeviceToHost, ctx().cur),
              "hipMemcpyAsync D2H");
    sync();
  });
}

extern "C" int stwo_hip_merkle_auth_paths(StwoBlake2sHash* const* layers, uint32_t max_log, const uint32_t* leaves,
                                          uint32_t n_leaves, StwoBlake2sHash* paths) {
  return guarded([&] {
    if (!n_leaves || !max_log) return;
    require(layers != nullptr && leaves != nullptr && paths != nullptr, "merkle_auth_paths: null argument");
    require(max_log <= 31, "merkle_auth_paths: at most 31 layers");
    for (uint32_t q = 0; q < n_leaves; q++)
      require(leaves[q] < (1u << max_log), "merkle_auth_paths: leaf index out of range");
    const uint64_t total = (uint64_t)n_leaves * max_log;
    require(total < (1ull << 31), "merkle_auth_paths: too many hashes");
    DevBuf table = upload(layers, (max_log + 1) * sizeof(void*));
    DevBuf dleaves = upload(leaves, n_leaves * sizeof(uint32_t));
    DevBuf out(total * sizeof(StwoBlake2sHash));
    timed("merkle_auth_paths", [&] {
      cols::auth_paths_kernel<<<ceil_div(total, 256), 256, 0, ctx().cur>>>(
          table.as<const cols::Hash8*>(), max_log, dleaves.as<uint32_t>(), (uint32_t)total, out.as<cols::Hash8>());
    });
    hip_check(hipMemcpyAsync(paths, out.p, total * sizeof(StwoBlake2sHash), hipMemcpyDeviceToHost, ctx().cur),
              "hipMemcpyAsync D2H");
    sync();
  });
}

extern "C" void bit_reverse_base_field(uint32_t* array, size_t size) {
  guarded([&] {
    cols::bit_reverse(array, size);
    sync();
  });
}
extern "C" void bit_reverse_secure_field(uint32_t* array, size_t size) {
  guarded([&] {
    cols::bit_reverse(reinterpret_cast<uint4*>(array), size);
    sync();
  });
}
extern "C" uint32_t* sort_values_and_permute_with_bit_reverse_order(const uint32_t* from, size_t size) {
  uint32_t* dst = nullptr;
  guarded([&] {
    require(is_pow2(size) && size <= (1ull << 31), "sort_values: size must be a power of two");
    dst = (uint32_t*)ctx().pool.alloc(size * 4);
    timed("sort_values", [&] {
      cols::sort_values_kernel<<<ceil_div(size, 256), 256, 0, ctx().cur>>>(from, dst, (uint32_t)size);
    });
    cols::bit_reverse(dst, size);
    sync();
  });
  return dst;
}
extern "C" void accumulate(uint32_t size, uint32_t* const* left_columns, uint32_t* const* right_columns) {
  guarded([&] {
    if (!size) return;
    cols::Soa4 l{{left_columns[0], left_columns[1], left_columns[2], left_columns[3]}};
    cols::Soa4 r{{right_columns[0], right_columns[1], right_columns[2], right_columns[3]}};
    timed("accumulate", [&] {
      cols::accumulate_kernel<<<ceil_div(size, 256), 256, 0, ctx().cur>>>(size, l, r);
    });
    sync();
  });
}
