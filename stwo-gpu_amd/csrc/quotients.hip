// DEEP quotients: QuotientOps::accumulate_quotients (stwo_gpu_backend/src/quotient.rs:17-115).
//
// For row r of the (bit-reversed) evaluation domain, p = domain.at(brev(r)), and
// for each sample batch b (point P_b, samples (column j, value v_j)) in order
// (cuda/src/quotients.cu:111-178):
//   acc = acc * rc^|b| + (sum_j c_j col_j[r] - (a_j p.y + b_j)) * den_b(p)^-1
// with line coefficients a = conj(v) - v, c = conj(P.y) - P.y, b = v c - a P.y,
// each times alpha_j = rc^(j+1) (quotients.cu:49-88), and
//   den_b(p) = (Re P.x - p.x) Im P.y - (Re P.y - p.y) Im P.x   in CM31 (quotients.cu:91-109).
// The line coefficients use the cumulative offset of quotients.cu:147-168 (the
// reference's quotients.cu:74 offset is wrong for batches of different sizes).
//
// MI355X design: the per-batch sums of a_j and b_j and the factor c (shared by
// every sample of a batch, since c depends only on P) are folded on the host, so
// what is left per row is sum_j alpha_j col_j[row] per batch: for up to 4 batches
// a contraction over the columns on the matrix cores (accumulate_mm_kernel; for few samples
// accumulate_cols_kernel), beyond that multiply-accumulates on 64-bit lazy sums, batch by
// batch (accumulate_kernel).
#include <cstring>
#include <map>
#include <vector>

#include "field.hpp"
#include "gmem.hpp"
#include "mfma_m31.hpp"
#include "runtime.hpp"

namespace sh {
namespace quot {

struct Sample {
  uint32_t col;
  uint32_t pad;
  qm31 alpha;  // rc^(j+1)
};
struct Batch {
  uint32_t first, count;
  qm31 c;      // conj(P.y) - P.y
  qm31 a_sum;  // sum_j alpha_j (conj(v_j) - v_j)
  qm31 b_sum;  // sum_j alpha_j (v_j c - (conj(v_j) - v_j) P.y)
  qm31 coeff;  // rc^count
  cm31 prx, pry, pix, piy;
};

__device__ __forceinline__ uint64_t fold64(uint64_t s) { return (s & P) + (s >> 31); }

// Points of CircleDomain(half coset (hi, hs) of log half_log) from two small tables
// instead of a 31-step power per row: lo[j] = G^(hi + hs j) for j < 2^k and
// up[j] = G^(hs j 2^k) for j < 2^(half_log - k), so position i < 2^half_log is
// lo[i mod 2^k] up[i >> k] and position i + 2^half_log its conjugate
// (CircleDomain::index_at, cuda/src/quotients.cu:17-29).
struct DomainTables {
  const pt* lo;
  const pt* up;
  uint32_t k, half_log;
};
constexpr uint32_t DT_LO_BITS = 11;
inline uint32_t dt_k(uint32_t half_log) { return half_log < DT_LO_BITS ? half_log : DT_LO_BITS; }
inline size_t dt_bytes(uint32_t half_log) {
  const uint32_t k = dt_k(half_log);
  return (sizeof(pt) * ((1ull << k) + (1ull << (half_log - k))) + 255) & ~(size_t)255;
}
__global__ void domain_tables_kernel(uint32_t hi, uint32_t hs, uint32_t half_log, uint32_t k, pt* lo, pt* up) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < (1u << k)) lo[t] = point_at_index((uint32_t)((hi + (uint64_t)hs * t) & 0x7fffffffu));
  if (t < (1u << (half_log - k))) up[t] = point_at_index((uint32_t)(((uint64_t)hs * ((uint64_t)t << k)) & 0x7fffffffu));
}
__device__ __forceinline__ pt domain_point(const DomainTables& T, uint32_t i) {
  const uint32_t half = 1u << T.half_log;
  const bool conj = i >= half;
  const uint32_t j = conj ? i - half : i;
  pt q = pmul(T.lo[j & ((1u << T.k) - 1)], T.up[j >> T.k]);
  if (conj) q.y = neg(q.y);
  return q;
}

__global__ __launch_bounds__(256) void accumulate_kernel(DomainTables T, uint32_t log_size,
                                                         const uint32_t* const* __restrict__ cols,
                                                         const Sample* __restrict__ samples,
                                                         const Batch* __restrict__ batches, uint32_t n_batches,
                                                         uint32_t* __restrict__ o0, uint32_t* __restrict__ o1,
                                                         uint32_t* __restrict__ o2, uint32_t* __restrict__ o3) {
  uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= (1u << log_size)) return;
  pt p = domain_point(T, brev(row, log_size));
  qm31 acc = qzero();
  for (uint32_t b = 0; b < n_batches; b++) {
    const Batch B = batches[b];
    uint64_t s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    uint32_t j = 0;
    for (; j + 2 <= B.count; j += 2) {
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const Sample S = samples[B.first + j + u];
        uint64_t v = at(as_global(cols[S.col]), row);
        s0 += S.alpha.x.a * v;
        s1 += S.alpha.x.b * v;
        s2 += S.alpha.y.a * v;
        s3 += S.alpha.y.b * v;
      }
      s0 = fold64(s0);
      s1 = fold64(s1);
      s2 = fold64(s2);
      s3 = fold64(s3);
    }
    if (j < B.count) {
      const Sample S = samples[B.first + j];
      uint64_t v = at(as_global(cols[S.col]), row);
      s0 += S.alpha.x.a * v;
      s1 += S.alpha.x.b * v;
      s2 += S.alpha.y.a * v;
      s3 += S.alpha.y.b * v;
    }
    qm31 sum = {{reduce63(s0), reduce63(s1)}, {reduce63(s2), reduce63(s3)}};
    qm31 num = qsub(qmul(B.c, sum), qadd(qscale(B.a_sum, p.y), B.b_sum));
    cm31 d = csub(cmul(cm31{sub(B.prx.a, p.x), B.prx.b}, B.piy), cmul(cm31{sub(B.pry.a, p.y), B.pry.b}, B.pix));
    acc = qadd(qmul(acc, B.coeff), qmul_cm(num, cinv(d)));
  }
  o0[row] = acc.x.a;
  o1[row] = acc.x.b;
  o2[row] = acc.y.a;
  o3[row] = acc.y.b;
}

__device__ __forceinline__ cm31 batch_denominator(const Batch& B, pt p) {
  return csub(cmul(cm31{sub(B.prx.a, p.x), B.prx.b}, B.piy), cmul(cm31{sub(B.pry.a, p.y), B.pry.b}, B.pix));
}

// the accumulation over the batches at p, from each batch's sum(b): one CM31 inversion for the NB
// denominators (prefix products, Montgomery's trick).  A sum is asked for where it is used, behind the
// inversion (reduced ahead of it the multiply-add kernel takes 91.2 us instead of 88.8, 8 columns
// of 2^20 at four points).
template <int NB, class Sum>
__device__ __forceinline__ qm31 combine(const Batch* __restrict__ batches, Sum sum, pt p) {
  cm31 d[NB], pre[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    d[b] = batch_denominator(batches[b], p);
    pre[b] = b == 0 ? d[0] : cmul(pre[b - 1], d[b]);
  }
  cm31 inv_all = cinv(pre[NB - 1]);
  cm31 dinv[NB];
#pragma unroll
  for (int b = NB - 1; b > 0; b--) {
    dinv[b] = cmul(inv_all, pre[b - 1]);
    inv_all = cmul(inv_all, d[b]);
  }
  dinv[0] = inv_all;
  qm31 r = qzero();
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const Batch& B = batches[b];
    const qm31 num = qsub(qmul(B.c, sum(b)), qadd(qscale(B.a_sum, p.y), B.b_sum));
    r = qadd(qmul(r, B.coeff), qmul_cm(num, dinv[b]));
  }
  return r;
}

// Column-major form for up to 4 batches and few samples (few_samples; or more columns than MM_MAX_SLOTS): each
// sampled column value of a row is loaded once and multiplied into the sums of all NB batches,
// with alpha = 0 for a batch that does not sample the column; loads run one group of QG columns
// ahead of the arithmetic.  A batch's sums are folded after every fourth product taken into
// them: a product of two values below P is at most (P - 1)^2 = 2^62 - 2^33 + 1, and a folded
// sum is below 2^34, so four products on top of it stay below 2^64.
template <int NB>
struct ColSlot {
  const uint32_t* col;  // the column (device pointer)
  uint32_t mask;        // bit b: batch b samples the column (alpha[b] may be nonzero)
  uint32_t pad;
  qm31 alpha[NB];
};

constexpr int QG = 16;  // columns per load group (a multiple of the fold period 4; 8: 6 % slower at 200 x 2^21)

template <int NB>
__global__ __launch_bounds__(256) void accumulate_cols_kernel(DomainTables T, uint32_t log_size,
                                                              const ColSlot<NB>* __restrict__ slots,
                                                              uint32_t n_slots, const Batch* __restrict__ batches,
                                                              uint32_t* __restrict__ o0, uint32_t* __restrict__ o1,
                                                              uint32_t* __restrict__ o2, uint32_t* __restrict__ o3) {
  uint32_t row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= (1u << log_size)) return;
  uint64_t s[NB][4];
#pragma unroll
  for (int b = 0; b < NB; b++) s[b][0] = s[b][1] = s[b][2] = s[b][3] = 0;
  // n_slots is a multiple of QG (zero-alpha slots of column 0 pad it), and QG more such
  // slots follow, so the next group's loads are issued unconditionally: a conditional
  // prefetch makes the compiler wait for every load in flight before the arithmetic
  uint32_t v[QG], vn[QG];
  // products taken into each batch's sums since their last fold (uniform): a batch's sums
  // are folded after its fourth product, not after every fourth column, so batches that
  // sample few of the columns fold rarely
  uint32_t since[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) since[b] = 0;
#pragma unroll
  for (int i = 0; i < QG; i++) v[i] = at(as_global(slots[i].col), row);
  for (uint32_t h = 0; h < n_slots; h += QG) {
#pragma unroll
    for (int i = 0; i < QG; i++) vn[i] = at(as_global(slots[h + QG + i].col), row);
#pragma unroll
    for (int i = 0; i < QG; i++) {
      const ColSlot<NB>& S = slots[h + i];
#pragma unroll
      for (int b = 0; b < NB; b++) {
        if (NB > 1 && !(S.mask & (1u << b))) continue;  // uniform: the slot is the same for every lane
        s[b][0] += (uint64_t)S.alpha[b].x.a * v[i];
        s[b][1] += (uint64_t)S.alpha[b].x.b * v[i];
        s[b][2] += (uint64_t)S.alpha[b].y.a * v[i];
        s[b][3] += (uint64_t)S.alpha[b].y.b * v[i];
        if (++since[b] == 4) {
          since[b] = 0;
          s[b][0] = fold64(s[b][0]);
          s[b][1] = fold64(s[b][1]);
          s[b][2] = fold64(s[b][2]);
          s[b][3] = fold64(s[b][3]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < QG; i++) v[i] = vn[i];
  }
  const pt p = domain_point(T, brev(row, log_size));
  const qm31 acc = combine<NB>(
      batches,
      [&](int b) {
        return qm31{{reduce63(s[b][0]), reduce63(s[b][1])}, {reduce63(s[b][2]), reduce63(s[b][3])}};
      },
      p);
  o0[row] = acc.x.a;
  o1[row] = acc.x.b;
  o2[row] = acc.y.a;
  o3[row] = acc.y.b;
}

// Column-major form for up to 4 batches, on the matrix cores: the sums sum_j alpha_j col_j[row] of
// all batches are one contraction over the columns.  v_mfma_i32_32x32x32_i8 on signed byte digits
// (mfma_m31.hpp) takes a step of 8 columns (4 digits each) of 32 rows times 8 outputs of 4 limbs,
// two batches to an instruction; a column that a batch does not sample has weight 0 there.  Two
// and a half VALU instructions per value instead of four 64-bit multiply-adds per sample and their
// folds leave the kernel bound by the column reads.
//
// The reads need about 64 KB per CU on their way.  Held in registers they cost the occupancy, and
// the compiler waits for all of them at each turn of the loop (360 us at 200 columns of 2^21, 3
// points).  So they go straight to LDS: a wave's 64 rows of DEPTH steps of columns are a ring that
// only this wave reads, after a wait that leaves the newer steps in flight; no registers, no
// barrier.  The operand tiles are the block's, loaded the same way CHUNK steps at a time into the
// half that is not being read (one barrier a chunk; read from L2 by every wave they would be as
// many bytes as the columns).  The LDS reads and their wait are one asm statement: reads through
// the compiler would again wait for every load.  200 columns of 2^21, 3 points: 373 -> 320 us per
// call, the kernel 300 (5.7 TB/s); a ring of 4 steps is no faster; blocks in XCD order 598 us
// instead of 624 at 200 columns of 2^22 (columns not padded apart share an XCD's lines).
constexpr uint32_t KSTEP = 8;            // columns per step
constexpr uint32_t MM_MAX_SLOTS = 8192;  // columns: join64's bound on the limb sums
constexpr uint32_t MM_WAVES = 8;         // per block; 64 rows each
constexpr uint32_t DEPTH = 3;            // steps of columns on their way into a wave's ring
constexpr uint32_t RING = DEPTH * KSTEP * 64, TILE = 256;  // words of a ring, of an operand tile
// Values from which the column reads are nontemporal (more than the caches hold: 200 columns of
// 2^22, 1 point: 597 us instead of 634; below, 64 columns of 2^20: 84 us plain, 90 nontemporal).
constexpr uint64_t MM_STREAM = 1ull << 27;
// Whether a call samples so little that the multiply-adds are the faster form: the matrix form's
// weights are expanded by a launch of their own instead of copied (3 us), and an odd batch fills half
// an operand tile.  The more rows, the sooner that is made up; a batch's multiply-adds also run over
// columns in groups of 16, sampled or not.  Matrix / multiply-add time of a call: one point, 112 samples
// 0.93 .. 1.02 and 128 0.90 .. 1.01.  Two points, 16 columns at both up to 2^16 rows 1.04, 17 columns
// 0.98, 16 of 2^17 1.00.  Three points, 16 columns at each up to 2^16 rows 1.07, 20 1.01, 24 1.00, 40
// columns at one point each 0.98; 11 of 2^19 1.02, 14 1.00; 11 of 2^20 1.00.  Four points, 8 columns at
// each up to 2^16 rows 1.03, 12 0.98, 32 columns at one point each 0.95; 8 of 2^17 0.97.
inline bool few_samples(uint32_t n_batches, uint32_t log_size, uint64_t samples, uint32_t columns) {
  if (samples < 32) return true;
  if (n_batches == 1) return samples < 128;
  if (n_batches == 2) return log_size < 17 && samples < 34;
  if (n_batches == 3) return log_size < 19 ? samples < 64 && columns <= 32 : log_size == 19 && samples < 40;
  return log_size < 17 && samples < 48 && columns <= 16;
}
constexpr uint32_t mm_tiles(uint32_t n_batches) { return (n_batches + 1) / 2; }
constexpr uint32_t padded_slots(uint32_t n_cols) { return (n_cols + KSTEP - 1) / KSTEP * KSTEP; }

// word of the weights of slot, batch: the first of its 16 rows (4 words apart)
__host__ __device__ __forceinline__ uint32_t weight_word(uint32_t slot, uint32_t batch, uint32_t tiles) {
  return ((slot / KSTEP * tiles + batch / 2) * 64 + ((slot >> 2) & 1) * 32 + (batch & 1) * 16) * 4 + (slot & 3);
}

// From a host image (pinned memory) to the kernel's tables: column pointers and
// batches copied, alphas ([slot][batch], n_slots x n_batches) expanded to weights.
__global__ __launch_bounds__(256) void weights_kernel(const uint2* __restrict__ ptrs, const qm31* __restrict__ alphas,
                                                      const uint32_t* __restrict__ batch_words, uint32_t n_slots,
                                                      uint32_t n_batches, uint2* d_ptrs, uint32_t* weights,
                                                      uint32_t* d_batches) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t tiles = mm_tiles(n_batches);
  if (t < n_slots) d_ptrs[t] = ptrs[t];
  if (t < n_batches * (sizeof(Batch) / 4)) d_batches[t] = batch_words[t];
  const uint32_t slot = t / (2 * tiles), b = t % (2 * tiles);
  if (slot >= n_slots) return;
  const qm31 v = b < n_batches ? alphas[slot * n_batches + b] : qzero();
  const uint32_t c[4] = {v.x.a, v.x.b, v.y.a, v.y.b};
  mm::operand_rows(c, weights + weight_word(slot, b, tiles));
}

// js: byte stride between the jobs of a batched launch (blockIdx.z = job): the tables and the
// outputs move by the job's offset (the pointers already are that job's columns)
template <int NB, bool NT>
__global__ __launch_bounds__(MM_WAVES * 64) __attribute__((amdgpu_waves_per_eu(4))) void accumulate_mm_kernel(
    DomainTables T, uint32_t log_size, const uint32_t* const* __restrict__ cols, const uint32_t* __restrict__ weights,
    uint32_t n_steps, const Batch* __restrict__ batches, uint32_t* __restrict__ o0, uint32_t* __restrict__ o1,
    uint32_t* __restrict__ o2, uint32_t* __restrict__ o3, uint64_t js) {
  constexpr int MT = (int)mm_tiles(NB);
  constexpr uint32_t CHUNK = MM_WAVES / MT;  // steps whose operand tiles the block loads together, a tile per wave
  static_assert(CHUNK >= DEPTH, "a chunk's tiles are older than its first step's columns");
  __shared__ __align__(16) uint32_t lds[MM_WAVES * RING + 2 * MM_WAVES * TILE];
  (void)lds;
  const uint64_t jo = job_offset(js);
  cols = jptr(cols, jo);
  batches = jptr(batches, jo);
  uint32_t* const out[4] = {jptr(o0, jo), jptr(o1, jo), jptr(o2, jo), jptr(o3, jo)};
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t n_rows = 1u << log_size, place = (MM_WAVES * xcd_order() + wave) * 64;
  // a wave past the domain's end repeats its first rows, a lane past it the last one
  const uint32_t row0 = place < n_rows ? place : 0, row = min(lane, n_rows - 1 - row0);

  mm::v16i acc[MT][2] = {};  // [tile][rows of the wave's lower or upper 32 lanes]
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) uint32_t lds_word;
  lds_word* const ring = (lds_word*)lds + wave * RING;
  lds_word* const wring = (lds_word*)lds + MM_WAVES * RING;
  constexpr int AUX = NT ? 2 : 0;
  auto fetch = [&](const uint32_t* const (&p)[KSTEP], uint32_t slot) {
#pragma unroll
    for (uint32_t c = 0; c < KSTEP; c++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(BufCol(p[c] + row0).rs, ring + (slot * KSTEP + c) * 64, 4, row * 4, 0,
                                               0, AUX);
  };
  auto pointers = [&](const uint32_t* (&p)[KSTEP], uint32_t step) {
#pragma unroll
    for (uint32_t c = 0; c < KSTEP; c++) p[c] = ld_uniform(cols, KSTEP * step + c);
  };
  const BufCol wbuf(jptr(weights, jo));
  auto fetch_weights = [&](uint32_t chunk) {
    const uint32_t tile = chunk * MM_WAVES + wave;
    if (tile < n_steps * MT)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wbuf.rs, wring + ((chunk & 1) * MM_WAVES + wave) * TILE, 16, lane * 16,
                                               tile * (4 * TILE), 0, 0);
  };
  fetch_weights(0);
  for (uint32_t s = 0; s < DEPTH && s < n_steps; s++) {
    const uint32_t* p[KSTEP];
    pointers(p, s);
    fetch(p, s);
  }
  const uint32_t x_lane = (uint32_t)(size_t)ring + (lane >> 5) * 1024 + (lane & 31) * 4;
  const uint32_t w_lane = (uint32_t)(size_t)wring + lane * 16;
  uint32_t slot = 0;
  for (uint32_t s = 0; s < n_steps; s++) {
    const uint32_t* p[KSTEP];
    pointers(p, min(s + DEPTH, n_steps - 1));
    // the loads come back in order: all but the newest DEPTH - 1 steps are there
    if (s + DEPTH <= n_steps)
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"((DEPTH - 1) * KSTEP) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (s % CHUNK == 0) {
      // every wave's tile of this chunk is there (older than the step just waited for), and nobody
      // reads the other half any more
      __builtin_amdgcn_s_barrier();
      fetch_weights(s / CHUNK + 1);
    }
    typedef uint32_t v2u __attribute__((ext_vector_type(2)));
    v2u x[4];
    mm::v4i w[2];
    const uint32_t xa = x_lane + slot * (KSTEP * 256), xb = xa + 128;
    const uint32_t wa = w_lane + s % (2 * CHUNK) * (MT * 4 * TILE);
    if constexpr (MT == 2) {
      asm volatile(
          "ds_read2st64_b32 %0, %6 offset0:0 offset1:1\n"
          "ds_read2st64_b32 %1, %6 offset0:2 offset1:3\n"
          "ds_read_b128 %4, %8\n"
          "ds_read_b128 %5, %8 offset:1024\n"
          "ds_read2st64_b32 %2, %7 offset0:0 offset1:1\n"
          "ds_read2st64_b32 %3, %7 offset0:2 offset1:3\n"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(w[0]), "=&v"(w[1])
          : "v"(xa), "v"(xb), "v"(wa)
          : "memory");
    } else {
      asm volatile(
          "ds_read2st64_b32 %0, %5 offset0:0 offset1:1\n"
          "ds_read2st64_b32 %1, %5 offset0:2 offset1:3\n"
          "ds_read_b128 %4, %7\n"
          "ds_read2st64_b32 %2, %6 offset0:0 offset1:1\n"
          "ds_read2st64_b32 %3, %6 offset0:2 offset1:3\n"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(w[0])
          : "v"(xa), "v"(xb), "v"(wa)
          : "memory");
    }
    if (s + DEPTH < n_steps) fetch(p, slot);  // into the slot that was just read
    slot = slot + 1 == DEPTH ? 0 : slot + 1;
    mm::v4i lo, hi;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      lo[i] = (int)mm::digits(x[i / 2][i & 1]);
      hi[i] = (int)mm::digits(x[2 + i / 2][i & 1]);
    }
#pragma unroll
    for (int t = 0; t < MT; t++) {
      acc[t][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[t], lo, acc[t][0], 0, 0, 0);
      acc[t][1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[t], hi, acc[t][1], 0, 0, 0);
    }
  }
#endif
  // registers 4q .. 4q + 3 hold the limbs of output 2q + (lane / 32) of either half's rows: the
  // swap gives each lane its own row's outputs 2q and 2q + 1
  qm31 sum[2 * MT];
#pragma unroll
  for (int t = 0; t < MT; t++) {
    uint32_t e[4], o[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const mm::v16i &a = acc[t][0], &b = acc[t][1];
      e[q] = mm::join64(a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]);
      o[q] = mm::join64(b[4 * q], b[4 * q + 1], b[4 * q + 2], b[4 * q + 3]);
#if defined(__HIP_DEVICE_COMPILE__)
      const auto z = __builtin_amdgcn_permlane32_swap(e[q], o[q], false, false);
      e[q] = z[0];
      o[q] = z[1];
#endif
    }
    sum[2 * t] = {{e[0], o[0]}, {e[1], o[1]}};
    sum[2 * t + 1] = {{e[2], o[2]}, {e[3], o[3]}};
  }
  if (lane >= n_rows - row0 || place >= n_rows) return;
  const pt p = domain_point(T, brev(row0 + row, log_size));
  const qm31 r = combine<NB>(batches, [&](int b) { return sum[b]; }, p);
  const uint32_t res[4] = {r.x.a, r.x.b, r.y.a, r.y.b};
#pragma unroll
  for (int k = 0; k < 4; k++) BufCol(out[k] + row0).store(res[k], row, 0);
}

// One batch (every column sampled once at one point) built on the device from a
// point, sample values and random coefficient that live in device memory: lane j
// takes samples j, j + 256, ...; the per-batch sums are reduced in LDS.
constexpr uint32_t SB_NT = 256;
__global__ __launch_bounds__(SB_NT) void single_batch_kernel(const uint32_t* const* __restrict__ cols,
                                                             const qm31* __restrict__ point,
                                                             const qm31* __restrict__ values, uint32_t count,
                                                             const qm31* __restrict__ rc_dev, const uint32_t** ptrs,
                                                             uint32_t* weights, uint32_t n_slots, Batch* bs,
                                                             uint64_t js) {
  __shared__ qm31 sa[SB_NT], sb[SB_NT];
  // batched jobs (blockIdx.z): the slots get the job's own column pointers
  const uint64_t jo = job_offset(js);
  point = jptr(point, jo);
  values = jptr(values, jo);
  rc_dev = jptr(rc_dev, jo);
  ptrs = jptr(ptrs, jo);
  weights = jptr(weights, jo);
  bs = jptr(bs, jo);
  const qm31 px = point[0], py = point[1], rc = *rc_dev;
  const qm31 c = qsub(qm31{py.x, cneg(py.y)}, py);
  qm31 la = qzero(), lb = qzero();
  for (uint32_t j = threadIdx.x; j < n_slots; j += SB_NT) {
    ptrs[j] = jptr(cols[j < count ? j : 0], jo);
    qm31 alpha = qzero();  // slots past the last column weigh nothing
    if (j < count) {
      alpha = qpow(rc, j + 1);
      const qm31 v = values[j];
      const qm31 a = qsub(qm31{v.x, cneg(v.y)}, v);
      const qm31 bb = qsub(qmul(v, c), qmul(a, py));
      la = qadd(la, qmul(alpha, a));
      lb = qadd(lb, qmul(alpha, bb));
    }
    const uint32_t w[4] = {alpha.x.a, alpha.x.b, alpha.y.a, alpha.y.b}, none[4] = {0, 0, 0, 0};
    mm::operand_rows(w, weights + weight_word(j, 0, 1));
    mm::operand_rows(none, weights + weight_word(j, 1, 1));
  }
  sa[threadIdx.x] = la;
  sb[threadIdx.x] = lb;
  __syncthreads();
  for (uint32_t h = SB_NT / 2; h > 0; h >>= 1) {
    if (threadIdx.x < h) {
      sa[threadIdx.x] = qadd(sa[threadIdx.x], sa[threadIdx.x + h]);
      sb[threadIdx.x] = qadd(sb[threadIdx.x], sb[threadIdx.x + h]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) bs[0] = Batch{0, count, c, sa[0], sb[0], qpow(rc, count), px.x, py.x, px.y, py.y};
}

// the quotient of an empty sample set: all four coordinates zero
__global__ __launch_bounds__(256) void zero_kernel(uint32_t n, uint32_t* o0, uint32_t* o1, uint32_t* o2,
                                                   uint32_t* o3) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  o0[i] = 0;
  o1[i] = 0;
  o2[i] = 0;
  o3[i] = 0;
}

}  // namespace quot

// tables of an accumulate_mm launch: pointers | weights | batches
namespace {
struct MmLayout {
  size_t weights, batches, end;
  MmLayout(uint32_t n_slots, uint32_t n_batches) {
    auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
    weights = up(sizeof(void*) * n_slots);
    batches = weights + up((size_t)(n_slots / quot::KSTEP) * quot::mm_tiles(n_batches) * (4 * quot::TILE));
    end = batches + up(sizeof(quot::Batch) * n_batches);
  }
};
template <int NB>
void launch_mm(uint32_t hi, uint32_t hs, uint32_t log_size, const void* tables, uint32_t n_slots, uint32_t* const out[4],
               uint32_t n_jobs, uint64_t js);
}  // namespace
// scratch of accumulate_quotients_single_point_async (the domain tables come from the library's
// per-domain cache)
size_t quotient_single_point_scratch_bytes(uint32_t n_cols, uint32_t max_log) {
  (void)max_log;
  return MmLayout(quot::padded_slots(std::max<uint32_t>(n_cols, 1)), 1).end;
}

// Fill the domain tables of CircleDomain(half coset (hi, hs), log log_size) at `dev`
// (dt_bytes(log_size - 1) bytes) on the current stream.
static quot::DomainTables domain_tables_async(uint32_t hi, uint32_t hs, uint32_t log_size, void* dev) {
  const uint32_t hl = log_size - 1, k = quot::dt_k(hl);
  pt* lo = (pt*)dev;
  pt* up = lo + (1u << k);
  const uint32_t n = std::max(1u << k, 1u << (hl - k));
  timed("quotient_domain_tables", [&] {
    quot::domain_tables_kernel<<<ceil_div(n, 256), 256, 0, ctx().cur>>>(hi, hs, hl, k, lo, up);
  });
  return quot::DomainTables{lo, up, k, hl};
}

// The domain tables of CircleDomain(half coset (hi, hs), log log_size), computed on first
// use and kept in the library context (until stwo_hip_release_twiddles), so repeated
// accumulations over one domain launch no table kernel.
static quot::DomainTables cached_domain_tables(uint32_t hi, uint32_t hs, uint32_t log_size) {
  const uint32_t hl = log_size - 1, k = quot::dt_k(hl);
  const TwiddleKey key{hi, hs, log_size};
  auto& cache = ctx().domain_tables;
  auto it = cache.find(key);
  if (it == cache.end()) {
    void* dev = ctx().pool.alloc(quot::dt_bytes(hl));
    domain_tables_async(hi, hs, log_size, dev);
    // the cached tables are read by work on every stream: finish them before sharing
    hip_check(hipStreamSynchronize(ctx().cur), "hipStreamSynchronize");
    it = cache.emplace(key, dev).first;
  }
  pt* lo = (pt*)it->second;
  return quot::DomainTables{lo, lo + (1u << k), k, hl};
}

// accumulate_quotients for one sample point shared by columns 0 .. n_cols-1 of d_cols, with
// the point (x, y), the sample values and the random coefficient read from device memory.
// n_jobs / js: same-shape jobs of a batched launch, js bytes apart (columns, point, values,
// coefficient, scratch and outputs all move by the job's offset; the domain is shared).
void accumulate_quotients_single_point_async(uint32_t hi, uint32_t hs, uint32_t log_size,
                                             const uint32_t* const* d_cols, uint32_t n_cols, const qm31* d_point,
                                             const qm31* d_values, const qm31* d_rc, void* d_scratch,
                                             uint32_t* const out[4], uint32_t n_jobs, uint64_t js) {
  require(log_size >= 1 && log_size <= 30 && n_cols >= 1, "accumulate_quotients: bad sizes");
  require(n_cols <= quot::MM_MAX_SLOTS, "accumulate_quotients: too many columns for one device-built batch");
  const uint32_t n_slots = quot::padded_slots(n_cols);
  const MmLayout Y(n_slots, 1);
  char* const base = (char*)d_scratch;
  timed("quotient_constants", [&] {
    quot::single_batch_kernel<<<dim3(1, 1, n_jobs), quot::SB_NT, 0, ctx().cur>>>(
        d_cols, d_point, d_values, n_cols, d_rc, (const uint32_t**)base, (uint32_t*)(base + Y.weights), n_slots,
        (quot::Batch*)(base + Y.batches), js);
  });
  launch_mm<1>(hi, hs, log_size, base, n_slots, out, n_jobs, js);
}

namespace {
template <int NB>
void launch_mm(uint32_t hi, uint32_t hs, uint32_t log_size, const void* tables, uint32_t n_slots, uint32_t* const out[4],
               uint32_t n_jobs, uint64_t js) {
  const MmLayout Y(n_slots, NB);
  const char* const base = (const char*)tables;
  const quot::DomainTables T = cached_domain_tables(hi, hs, log_size);
  constexpr uint32_t rows = quot::MM_WAVES * 64;  // per block
  const auto kernel = (uint64_t)n_slots << log_size >= quot::MM_STREAM ? quot::accumulate_mm_kernel<NB, true>
                                                                       : quot::accumulate_mm_kernel<NB, false>;
  timed("accumulate_quotients", [&] {
    kernel<<<dim3(ceil_div(1ull << log_size, rows), 1, n_jobs), quot::MM_WAVES * 64, 0, ctx().cur>>>(
        T, log_size, (const uint32_t* const*)base, (const uint32_t*)(base + Y.weights), n_slots / quot::KSTEP,
        (const quot::Batch*)(base + Y.batches), out[0], out[1], out[2], out[3], js);
  });
}

// column-major launch: per sampled column one slot with the alpha of every batch (0 when
// the batch does not sample it; a column sampled twice in one batch gets the sum)
template <int NB>
void launch_slots(uint32_t hi, uint32_t hs, uint32_t log_size, const uint32_t* const* h_cols,
                    const std::vector<quot::Sample>& ss, const std::vector<quot::Batch>& bs, uint32_t* const out[4]) {
  std::map<uint32_t, quot::ColSlot<NB>> by_col;
  for (uint32_t b = 0; b < (uint32_t)NB; b++)
    for (uint32_t j = 0; j < bs[b].count; j++) {
      const quot::Sample& S = ss[bs[b].first + j];
      auto it = by_col.find(S.col);
      if (it == by_col.end()) {
        quot::ColSlot<NB> z{};
        z.col = h_cols[S.col];
        for (int k = 0; k < NB; k++) z.alpha[k] = qzero();
        it = by_col.emplace(S.col, z).first;
      }
      it->second.alpha[b] = qadd(it->second.alpha[b], S.alpha);
      it->second.mask |= 1u << b;
    }
  std::vector<quot::ColSlot<NB>> slots;
  for (auto& kv : by_col) slots.push_back(kv.second);
  quot::ColSlot<NB> pad{};
  pad.col = slots.empty() ? h_cols[0] : slots[0].col;
  for (int k = 0; k < NB; k++) pad.alpha[k] = qzero();
  while (slots.empty() || slots.size() % quot::QG) slots.push_back(pad);
  const uint32_t n_loop = (uint32_t)slots.size();
  for (int i = 0; i < quot::QG; i++) slots.push_back(pad);  // read by the last group's prefetch
  // one upload: slots, then the batches at a 256-byte boundary
  const size_t slots_bytes = (slots.size() * sizeof(quot::ColSlot<NB>) + 255) & ~(size_t)255;
  std::vector<unsigned char> host(slots_bytes + bs.size() * sizeof(quot::Batch));
  memcpy(host.data(), slots.data(), slots.size() * sizeof(quot::ColSlot<NB>));
  memcpy(host.data() + slots_bytes, bs.data(), bs.size() * sizeof(quot::Batch));
  DevBuf d = upload(host.data(), host.size());
  const quot::ColSlot<NB>* dsl = d.as<quot::ColSlot<NB>>();
  const quot::Batch* dbs = (const quot::Batch*)((const unsigned char*)d.p + slots_bytes);
  const quot::DomainTables T = cached_domain_tables(hi, hs, log_size);
  timed("accumulate_quotients", [&] {
    quot::accumulate_cols_kernel<NB><<<ceil_div(1ull << log_size, 256), 256, 0, ctx().cur>>>(
        T, log_size, dsl, n_loop, dbs, out[0], out[1], out[2], out[3]);
  });
}
// matrix launch: slot_of[c] is the slot of sampled column c, n_used of them
template <int NB>
void launch_matrix(uint32_t hi, uint32_t hs, uint32_t log_size, const uint32_t* const* h_cols,
                   const std::vector<uint32_t>& slot_of, uint32_t n_used, const std::vector<quot::Sample>& ss,
                   const std::vector<quot::Batch>& bs, uint32_t* const out[4]) {
  const uint32_t n_slots = quot::padded_slots(n_used);
  // host image: pointers | alphas | batches
  const size_t o_alpha = sizeof(void*) * n_slots, o_batch = o_alpha + sizeof(qm31) * NB * n_slots;
  const size_t bytes = o_batch + sizeof(quot::Batch) * NB;
  static_assert((sizeof(void*) + sizeof(qm31) * NB) * quot::MM_MAX_SLOTS + sizeof(quot::Batch) * NB <= HOST_BLOCK_MAX,
                "the largest image fits pinned memory");
  HostBlock pinned(bytes);
  unsigned char* const host = pinned.as<unsigned char>();
  memset(host, 0, bytes);
  const uint32_t** ptrs = (const uint32_t**)host;
  qm31* alphas = (qm31*)(host + o_alpha);
  for (uint32_t b = 0; b < (uint32_t)NB; b++)
    for (uint32_t j = 0; j < bs[b].count; j++) {
      const quot::Sample& S = ss[bs[b].first + j];
      const uint32_t slot = slot_of[S.col];
      ptrs[slot] = h_cols[S.col];
      alphas[slot * NB + b] = qadd(alphas[slot * NB + b], S.alpha);
    }
  for (uint32_t i = n_used; i < n_slots; i++) ptrs[i] = ptrs[0];
  memcpy(host + o_batch, bs.data(), sizeof(quot::Batch) * NB);
  const MmLayout Y(n_slots, NB);
  DevBuf d(Y.end);
  char* const base = d.as<char>();
  timed("quotient_constants", [&] {
    const uint32_t threads = std::max<uint32_t>(n_slots * 2 * quot::mm_tiles(NB), NB * sizeof(quot::Batch) / 4);
    quot::weights_kernel<<<ceil_div(threads, 256), 256, 0, ctx().cur>>>(
        (const uint2*)host, (const qm31*)(host + o_alpha), (const uint32_t*)(host + o_batch), n_slots, NB, (uint2*)base,
        (uint32_t*)(base + Y.weights), (uint32_t*)(base + Y.batches));
  });
  launch_mm<NB>(hi, hs, log_size, base, n_slots, out, 1, 0);
}
template <int NB>
void launch_cols_nb(uint32_t hi, uint32_t hs, uint32_t log_size, const uint32_t* const* h_cols, uint32_t n_cols,
                    const std::vector<quot::Sample>& ss, const std::vector<quot::Batch>& bs, uint32_t* const out[4]) {
  constexpr uint32_t NONE = ~0u;
  std::vector<uint32_t> slot_of;
  uint32_t n_used = 0;
  if (ss.size() >= 32) slot_of.resize(n_cols, NONE);  // (fewer samples need no slots to decide)
  for (const quot::Sample& S : ss)
    if (!slot_of.empty() && slot_of[S.col] == NONE) slot_of[S.col] = n_used++;
  if (n_used > quot::MM_MAX_SLOTS || quot::few_samples(NB, log_size, ss.size(), n_used))
    launch_slots<NB>(hi, hs, log_size, h_cols, ss, bs, out);
  else
    launch_matrix<NB>(hi, hs, log_size, h_cols, slot_of, n_used, ss, bs, out);
}
void launch_cols(uint32_t hi, uint32_t hs, uint32_t log_size, const uint32_t* const* h_cols, uint32_t n_cols,
                 const std::vector<quot::Sample>& ss, const std::vector<quot::Batch>& bs, uint32_t n_batches,
                 uint32_t* const out[4]) {
  switch (n_batches) {
    case 1: launch_cols_nb<1>(hi, hs, log_size, h_cols, n_cols, ss, bs, out); break;
    case 2: launch_cols_nb<2>(hi, hs, log_size, h_cols, n_cols, ss, bs, out); break;
    case 3: launch_cols_nb<3>(hi, hs, log_size, h_cols, n_cols, ss, bs, out); break;
    default: launch_cols_nb<4>(hi, hs, log_size, h_cols, n_cols, ss, bs, out);
  }
}
}  // namespace

// points: n_batches x StwoCirclePointQM31 (host); indexes/values flattened in batch order (host).
// h_cols: the n_cols column pointers in host memory; d_cols: the same table in device memory,
// or null (uploaded here when the batch-major kernel needs it).
void accumulate_quotients_async(uint32_t hi, uint32_t hs, uint32_t domain_size, const uint32_t* const* d_cols,
                                const uint32_t* const* h_cols, uint32_t n_cols,
                                qm31 rc, uint32_t n_batches, const StwoCirclePointQM31* points,
                                const uint32_t* sizes, const uint32_t* col_idx, const StwoQM31* values,
                                uint32_t* const out[4]) {
  // column offsets are formed in 32 bits (gmem.hpp): at most 2^30 rows
  require(is_pow2(domain_size) && domain_size >= 2 && domain_size <= (1u << 30),
          "accumulate_quotients: domain size must be a power of two in 2 .. 2^30");
  uint32_t log_size = log2_exact(domain_size);
  uint64_t n_samples = 0;
  for (uint32_t b = 0; b < n_batches; b++) n_samples += sizes[b];
  if (n_samples == 0) {
    // every numerator is zero, so is the accumulation: no column is read
    timed("quotients_zero", [&] {
      quot::zero_kernel<<<ceil_div(domain_size, 256), 256, 0, ctx().cur>>>(domain_size, out[0], out[1], out[2],
                                                                             out[3]);
    });
    return;
  }
  require(n_cols >= 1 && h_cols != nullptr, "accumulate_quotients: samples name columns but none are given");
  std::vector<quot::Batch> bs(n_batches);
  std::vector<quot::Sample> ss;
  uint32_t off = 0;
  for (uint32_t b = 0; b < n_batches; b++) {
    qm31 px = from_w(qm31w{points[b].x.a, points[b].x.b, points[b].x.c, points[b].x.d});
    qm31 py = from_w(qm31w{points[b].y.a, points[b].y.b, points[b].y.c, points[b].y.d});
    qm31 c = qsub(qm31{py.x, cneg(py.y)}, py);
    quot::Batch& B = bs[b];
    B.first = (uint32_t)ss.size();
    B.count = sizes[b];
    B.c = c;
    B.a_sum = qzero();
    B.b_sum = qzero();
    B.coeff = qpow(rc, sizes[b]);
    B.prx = px.x;
    B.pix = px.y;
    B.pry = py.x;
    B.piy = py.y;
    qm31 alpha = qone();
    for (uint32_t j = 0; j < sizes[b]; j++) {
      const StwoQM31& w = values[off + j];
      qm31 v = {{w.a, w.b}, {w.c, w.d}};
      alpha = qmul(alpha, rc);
      qm31 a = qsub(qm31{v.x, cneg(v.y)}, v);
      qm31 bb = qsub(qmul(v, c), qmul(a, py));
      B.a_sum = qadd(B.a_sum, qmul(alpha, a));
      B.b_sum = qadd(B.b_sum, qmul(alpha, bb));
      ss.push_back(quot::Sample{col_idx[off + j], 0, alpha});
    }
    off += sizes[b];
  }
  if (n_batches >= 1 && n_batches <= 4) {
    launch_cols(hi, hs, log_size, h_cols, n_cols, ss, bs, n_batches, out);
    return;
  }
  if (ss.empty()) ss.push_back(quot::Sample{0, 0, qzero()});
  if (bs.empty()) bs.push_back(quot::Batch{});
  // one upload: samples, batches and (when the caller has no device table) the columns
  const size_t ss_bytes = (ss.size() * sizeof(quot::Sample) + 255) & ~(size_t)255;
  const size_t bs_bytes = (bs.size() * sizeof(quot::Batch) + 255) & ~(size_t)255;
  const size_t cols_bytes = d_cols ? 0 : (size_t)n_cols * sizeof(void*);
  std::vector<unsigned char> host(ss_bytes + bs_bytes + cols_bytes);
  memcpy(host.data(), ss.data(), ss.size() * sizeof(quot::Sample));
  memcpy(host.data() + ss_bytes, bs.data(), bs.size() * sizeof(quot::Batch));
  if (cols_bytes) memcpy(host.data() + ss_bytes + bs_bytes, h_cols, cols_bytes);
  DevBuf d = upload(host.data(), host.size());
  const unsigned char* base = (const unsigned char*)d.p;
  if (!d_cols) d_cols = (const uint32_t* const*)(base + ss_bytes + bs_bytes);
  const quot::DomainTables T = cached_domain_tables(hi, hs, log_size);
  timed("accumulate_quotients", [&] {
    quot::accumulate_kernel<<<ceil_div(domain_size, 256), 256, 0, ctx().cur>>>(
        T, log_size, d_cols, (const quot::Sample*)base, (const quot::Batch*)(base + ss_bytes), n_batches, out[0],
        out[1], out[2], out[3]);
  });
}

}  // namespace sh

using namespace sh;

extern "C" int stwo_hip_accumulate_quotients_async(uint32_t half_coset_initial_index, uint32_t half_coset_step_size,
                                                   uint32_t domain_size, const uint32_t* const* columns,
                                                   uint32_t n_columns, StwoQM31 random_coeff, uint32_t n_batches,
                                                   const StwoCirclePointQM31* points, const uint32_t* batch_sizes,
                                                   const uint32_t* column_indexes, const StwoQM31* values,
                                                   uint32_t* const* out) {
  return guarded([&] {
    uint64_t total = 0;
    for (uint32_t b = 0; b < n_batches; b++) total += batch_sizes[b];
    for (uint64_t i = 0; i < total; i++)
      require(column_indexes[i] < n_columns, "accumulate_quotients: column index out of range");
    uint32_t* o[4] = {out[0], out[1], out[2], out[3]};
    accumulate_quotients_async(half_coset_initial_index, half_coset_step_size, domain_size, nullptr, columns,
                               n_columns, qm31{{random_coeff.a, random_coeff.b},
                                                                 {random_coeff.c, random_coeff.d}},
                               n_batches, points, batch_sizes, column_indexes, values, o);
  });
}

extern "C" void accumulate_quotients(uint32_t half_coset_initial_index, uint32_t half_coset_step_size,
                                     uint32_t domain_size, uint32_t* const* columns, size_t number_of_columns,
                                     StwoQM31 random_coeff, const uint32_t* sample_points,
                                     const uint32_t* sample_column_indexes, uint32_t sample_column_indexes_size,
                                     const StwoQM31* sample_column_values,
                                     const uint32_t* sample_column_and_values_sizes, uint32_t sample_size,
                                     uint32_t* result_column_0, uint32_t* result_column_1, uint32_t* result_column_2,
                                     uint32_t* result_column_3, uint32_t flattened_line_coeffs_size) {
  (void)flattened_line_coeffs_size;
  guarded([&] {
    uint64_t total = 0;
    for (uint32_t b = 0; b < sample_size; b++) total += sample_column_and_values_sizes[b];
    require(total == sample_column_indexes_size, "accumulate_quotients: batch sizes do not sum to the index count");
    for (uint64_t i = 0; i < total; i++)
      require(sample_column_indexes[i] < number_of_columns, "accumulate_quotients: column index out of range");
    uint32_t* out[4] = {result_column_0, result_column_1, result_column_2, result_column_3};
    // `columns` is a device table (copy_device_pointer_vec_from_host_to_device); keep a host copy
    std::vector<const uint32_t*> host_cols(std::max<size_t>(number_of_columns, 1));
    if (number_of_columns) {
      hip_check(hipMemcpyAsync(host_cols.data(), columns, number_of_columns * sizeof(void*), hipMemcpyDeviceToHost,
                               ctx().cur),
                "hipMemcpyAsync D2H");
      sync();
    }
    accumulate_quotients_async(half_coset_initial_index, half_coset_step_size, domain_size,
                               (const uint32_t* const*)columns, host_cols.data(), (uint32_t)number_of_columns,
                               qm31{{random_coeff.a, random_coeff.b},
                                                                     {random_coeff.c, random_coeff.d}},
                               sample_size, (const StwoCirclePointQM31*)sample_points, sample_column_and_values_sizes,
                               sample_column_indexes, sample_column_values, out);
    sync();
  });
}
