// PolyOps::eval_at_point (stwo_gpu_backend/src/poly.rs:84-94).
//
// For coefficients c[0 .. 2^L) and a QM31 point (x, y), the factors are
// f = [pi^(L-2)(x), ..., pi(x), x, y] with pi(x) = 2x^2 - 1
// (cuda/src/poly/eval_at_point.cu:99-110), and the value is the fold
//   fold(c, f) = fold(lo half, f[1:]) + fold(hi half, f[1:]) * f[0],
// i.e. bit b of a coefficient index selects factor f[L-1-b].
//
// Two launches: blocks reduce 2^11 coefficients each in LDS (bits 0..10), then
// one block reduces the block results (remaining bits).  The reference's shared
// memory aliasing (eval_at_point.cu:17-18) has no counterpart here: separate
// arrays, and every level reads into registers before a barrier and writes after.
#include <cstring>
#include <utility>
#include <vector>

#include "field.hpp"
#include "gmem.hpp"
#include "mfma_m31.hpp"
#include "runtime.hpp"

namespace sh {
namespace eap {

constexpr int CB = 11;  // coefficients per first-pass block = 2^CB
constexpr int NT = 256;

struct Factors {
  qm31 f[31];
};

// Reduce `cnt` level values in s (cnt power of two) with factors f[fi], f[fi-1], ...
__device__ void tree_reduce(qm31* s, uint32_t cnt, const Factors& F, int fi) {
  while (cnt > 1) {
    uint32_t half = cnt >> 1;
    qm31 r[4];
    uint32_t k = 0;
    for (uint32_t i = threadIdx.x; i < half; i += NT, k++) r[k & 3] = qadd(s[2 * i], qmul(s[2 * i + 1], F.f[fi]));
    __syncthreads();
    k = 0;
    for (uint32_t i = threadIdx.x; i < half; i += NT, k++) s[i] = r[k & 3];
    __syncthreads();
    cnt = half;
    fi--;
  }
}

// First pass: block b folds coefficients [b 2^cb, (b+1) 2^cb) with f[L-1], ..., f[L-cb].
__global__ __launch_bounds__(NT) void first_pass(const uint32_t* __restrict__ c, uint32_t L, uint32_t cb, Factors F,
                                                 qm31* partial) {
  __shared__ qm31 s[1 << (CB - 1)];
  const uint32_t pairs = 1u << (cb - 1);
  const size_t base = (size_t)blockIdx.x << cb;
  const qm31 fy = F.f[L - 1];
  for (uint32_t i = threadIdx.x; i < pairs; i += NT) {
    uint32_t c0 = c[base + 2 * i], c1 = c[base + 2 * i + 1];
    qm31 v = qscale(fy, c1);
    v.x.a = add(v.x.a, c0);
    s[i] = v;
  }
  __syncthreads();
  tree_reduce(s, pairs, F, (int)L - 2);
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// Later passes: block b folds partials [b 2^g, (b+1) 2^g) with f[fi], f[fi-1], ...
__global__ __launch_bounds__(NT) void reduce_pass(const qm31* in, uint32_t g, Factors F, int fi, qm31* out) {
  __shared__ qm31 s[1 << (CB - 1)];
  const uint32_t cnt = 1u << g;
  for (uint32_t i = threadIdx.x; i < cnt; i += NT) s[i] = in[((size_t)blockIdx.x << g) + i];
  __syncthreads();
  tree_reduce(s, cnt, F, fi);
  if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

// ---- many columns of one size at points held in device memory ----
// js (here and below): byte stride between the jobs of a batched launch (blockIdx.z = job)
// factors of one point: f[L-1] = y, f[L-2] = x, f[L-3] = pi(x), ...
__host__ __device__ inline void point_factors(qm31 x, qm31 y, uint32_t L, Factors& F) {
  F.f[L - 1] = y;
  for (uint32_t i = 2; i <= L; i++) {
    F.f[L - i] = x;
    x = qsub(qadd(qsqr(x), qsqr(x)), qone());
  }
}
__global__ void factors_kernel(const qm31* __restrict__ point, uint32_t L, Factors* F, uint64_t js) {
  const uint64_t jo = job_offset(js);
  point = jptr(point, jo);
  point_factors(point[0], point[1], L, *jptr(F, jo));
}

// a whole column of at most 2^CB coefficients per block (blockIdx.y)
__global__ __launch_bounds__(NT) void fold_cols(const uint32_t* const* __restrict__ cols, uint32_t L,
                                                const Factors* __restrict__ F, qm31* out, uint64_t js) {
  __shared__ qm31 s[1 << (CB - 1)];
  const uint64_t jo = job_offset(js);
  F = jptr(F, jo);
  out = jptr(out, jo);
  const uint32_t* c = jptr(cols[blockIdx.y], jo);
  const uint32_t pairs = 1u << (L - 1);
  const qm31 fy = F->f[L - 1];
  for (uint32_t i = threadIdx.x; i < pairs; i += NT) {
    uint32_t c0 = c[2 * i], c1 = c[2 * i + 1];
    qm31 v = qscale(fy, c1);
    v.x.a = add(v.x.a, c0);
    s[i] = v;
  }
  __syncthreads();
  tree_reduce(s, pairs, *F, (int)L - 2);
  if (threadIdx.x == 0) out[blockIdx.y] = s[0];
}

// ---- columns of log >= 12 as a product with a basis on the matrix cores ------------------
// The value at a point is sum_i c_i B_i with B_i the product of the factors selected by the bits
// of i.  Split i = 128 k + l and k = R h + r: B_i = Lo[l] Mid[r] Hi[h].  A wave takes one range h
// of one column and forms sum_r Mid[r] c[128 (R h + r) + l] for its 128 values of l at up to two
// points: the contraction over r by v_mfma_i32_32x32x32_i8 on signed byte digits (mfma_m31.hpp:
// rows point, coordinate, limb; 8 values of r with 4 digits each per instruction; the 32 columns
// of the tile are l / 4, and l mod 4 selects one of four accumulators, so each coefficient load
// is 16 bytes per lane and 512 contiguous bytes per half wave).  What is left is one QM31 product
// with Lo per l, the sum over the wave and one product with Hi.
//
// Every coefficient is read once for both points and costs two VALU instructions (its digits),
// so the kernel is bound by the reads (multiply-adds of M31 x QM31 on the VALU took 12 per
// coefficient and point).  256 columns of 2^18 at two points: 2 x 55 -> 51 us, 5.2 TB/s; the whole
// call 204 -> 91 us with one launch per step for both points, the factors made on the host and
// the values written to host memory by the last kernel.
constexpr uint32_t MIN_GEMV_LOG = 12, LO_BITS = 7, PTS = 2;

// R (a power of two) ranges of r, H of h; blocks of four ranges
struct Shape {
  uint32_t r_log, h;  // R = 2^r_log, H ranges
};
// Enough blocks to fill the chip, a block being four ranges of a column, within 16 <= R <= 256
// (8 at log 12, where that is one block per column): fewer, longer ranges amortise the wave's
// sum.  From log 23 on R is at least 32 (64 for one column), which keeps Hi and the partial sums
// within eval_at_point_columns_scratch_bytes.
static Shape gemv_shape(uint32_t n_cols, uint32_t L, uint32_t n_jobs) {
  const uint32_t k_log = L - LO_BITS;  // >= 5
  const uint32_t min_r = L <= 22 ? 4 : n_cols == 1 ? 6 : 5;
  uint32_t hb_log = 0;  // blocks per column
  while (((uint64_t)n_cols * n_jobs << hb_log) < 2048 && k_log - 2 - hb_log > min_r) hb_log++;
  while (k_log - 2 - hb_log > 8) hb_log++;
  const uint32_t r_log = k_log - 2 - hb_log;
  return {r_log, 1u << (k_log - r_log)};
}

// One launch for all tables of a pair of points: Mid's limbs as matrix operands, Lo, Hi.
__global__ __launch_bounds__(256) void basis_tables_kernel(const Factors* __restrict__ F, uint32_t n_points, uint32_t L,
                                                           uint32_t r_log, uint32_t n_hi, uint32_t* mid, qm31* lo,
                                                           qm31* hi, uint64_t js) {
  uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t jo = job_offset(js);
  F = jptr(F, jo) + blockIdx.y;
  const uint32_t p = blockIdx.y;  // PTS of them; a missing second point has zero weights
  const uint32_t n_lo = 1u << LO_BITS, n_mid = 1u << r_log;
  // product of the factors of index bits [first, first + n) selected by v's bits
  auto product = [&](uint32_t v, uint32_t first, uint32_t n) {
    qm31 r = qone();
    for (uint32_t b = 0; b < n; b++)
      if ((v >> b) & 1) r = qmul(r, F->f[L - 1 - first - b]);
    return r;
  };
  if (t < n_mid) {
    const qm31 v = p < n_points ? product(t, LO_BITS, r_log) : qzero();
    const uint32_t c[4] = {v.x.a, v.x.b, v.y.a, v.y.b};
    // matrix operand of 8 values of r: lane row + 32 (bit 2 of r), word r mod 4
    uint32_t* const q = jptr(mid, jo) + 4 * (64 * (t >> 3) + 32 * ((t >> 2) & 1)) + (t & 3);
    mm::operand_rows(c, q + 16 * 4 * p);
    return;
  }
  t -= n_mid;
  if (p >= n_points) return;
  if (t < n_lo)
    jptr(lo, jo)[p * n_lo + t] = product(t, 0, LO_BITS);
  else if (t - n_lo < n_hi)
    jptr(hi, jo)[p * n_hi + t - n_lo] = product(t - n_lo, LO_BITS + r_log, L - LO_BITS - r_log);
}

template <int W>
__device__ __forceinline__ qm31 lanes_sum(qm31 v) {  // over groups of W lanes
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1) {
    v.x.a = add(v.x.a, (uint32_t)__shfl_xor((int)v.x.a, o));
    v.x.b = add(v.x.b, (uint32_t)__shfl_xor((int)v.x.b, o));
    v.y.a = add(v.y.a, (uint32_t)__shfl_xor((int)v.y.a, o));
    v.y.b = add(v.y.b, (uint32_t)__shfl_xor((int)v.y.b, o));
  }
  return v;
}
__device__ __forceinline__ qm31 wave_sum(qm31 v) { return lanes_sum<64>(v); }

// block (b, column): ranges 4b .. 4b + 3, one per wave.  out[(p n_cols + column) out_stride + b]
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void gemv_kernel(const uint32_t* const* __restrict__ cols, uint32_t n_cols,
                                                   uint32_t r_log, uint32_t n_hi, uint32_t n_points,
                                                   const uint32_t* __restrict__ mid, const qm31* __restrict__ lo,
                                                   const qm31* __restrict__ hi, qm31* __restrict__ out, uint64_t js) {
  __shared__ qm31 wsum[4][PTS];
  const uint64_t jo = job_offset(js);
  const uint32_t lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t h = 4 * blockIdx.x + wave;  // < n_hi, a multiple of 4
  const uint32_t steps = 1u << (r_log - 3);
  const uint32_t* col = jptr(ld_uniform(cols, blockIdx.y), jo);
  // coefficients 128 (R h + 8 s + 4 g + i) + 4 n ..: lane offset, uniform step
  const BufCol c(col + ((size_t)h << (r_log + LO_BITS)));
  const SH_GLOBAL mm::v4i* w = (const SH_GLOBAL mm::v4i*)as_global(jptr(mid, jo)) + lane;
  const uint32_t off = (g << (LO_BITS + 2)) + 4 * n;
  uint4 x[4], y[4];
  mm::v4i a, an;
  auto load = [&](uint32_t s, uint4 (&v)[4], mm::v4i& m) {
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) v[i] = c.load4(off, (s << (LO_BITS + 3)) + (i << LO_BITS));
    m = w[64 * s];
  };
  mm::v16i acc[4] = {};
  load(0, x, a);
  for (uint32_t s = 0; s < steps; s++) {
    load(min(s + 1, steps - 1), y, an);  // unconditional: the arithmetic waits for the older loads only
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      auto word = [&](const uint4& v) { return (int)mm::digits(j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w); };
      acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, mm::v4i{word(x[0]), word(x[1]), word(x[2]), word(x[3])}, acc[j],
                                                     0, 0, 0);
    }
#endif
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = y[i];
    a = an;
  }
  // lane (g, n) holds coordinates g and 2 + g of both points for l = 4n + j; after the exchange
  // with lane (1 - g, n) it holds point g's four
  const qm31* const lop = jptr(lo, jo) + (g < n_points ? g << LO_BITS : 0);
  qm31 sum = qzero();
#pragma unroll
  for (int j = 0; j < 4; j++) {
    uint32_t v[4];
#pragma unroll
    for (int q = 0; q < 4; q++)
      v[q] = mm::join64(acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]);
    const uint32_t z0 = (uint32_t)__shfl_xor((int)(g ? v[0] : v[2]), 32);
    const uint32_t z1 = (uint32_t)__shfl_xor((int)(g ? v[1] : v[3]), 32);
    const qm31 val = g ? qm31{{z0, v[2]}, {z1, v[3]}} : qm31{{v[0], z0}, {v[1], z1}};
    sum = qadd(sum, qmul(val, lop[4 * n + j]));
  }
  sum = lanes_sum<32>(sum);
  if (n == 0 && g < n_points) wsum[wave][g] = qmul(sum, jptr(hi, jo)[g * n_hi + h]);
  __syncthreads();
  if (threadIdx.x < n_points) {
    const uint32_t p = threadIdx.x;
    jptr(out, jo)[((size_t)p * n_cols + blockIdx.y) * gridDim.x + blockIdx.x] =
        qadd(qadd(wsum[0][p], wsum[1][p]), qadd(wsum[2][p], wsum[3][p]));
  }
}

// out[c] = sum of the n_hi partials of column c (one block per column)
__global__ __launch_bounds__(256) void sum_partials_kernel(const qm31* __restrict__ partial, uint32_t n_hi,
                                                           qm31* __restrict__ out, uint64_t js) {
  __shared__ qm31 ws[4];
  const uint64_t jo = job_offset(js);
  partial = jptr(partial, jo);
  out = jptr(out, jo);
  const uint32_t c = blockIdx.x, t = threadIdx.x;
  qm31 r = qzero();
  for (uint32_t h = t; h < n_hi; h += 256) r = qadd(r, partial[(size_t)c * n_hi + h]);
  r = wave_sum(r);
  if ((t & 63) == 0) ws[t >> 6] = r;
  __syncthreads();
  if (t == 0) out[c] = qadd(qadd(ws[0], ws[1]), qadd(ws[2], ws[3]));
}

}  // namespace eap

// Columns of log >= 12: factors of two points | Lo | Mid operands | Hi | partial sums.  The bound
// is that of a shape with 4096-value tables and one partial sum per 4096 coefficients, whose
// callers' limits it sets; gemv_layout stays within it.
size_t eval_at_point_columns_scratch_bytes(uint32_t n_cols, uint32_t L) {
  if (L >= eap::MIN_GEMV_LOG) return 512 + sizeof(qm31) * (4096 + (1ull << (L - 12)) * (1 + (size_t)n_cols));
  return 512 + 2 * sizeof(qm31) * (size_t)n_cols;  // (the factors take 496; callers' limits are set by this)
}

namespace {
struct GemvLayout {
  eap::Shape shape;
  size_t lo, mid, hi, partial, end;
  GemvLayout(uint32_t n_cols, uint32_t L, uint32_t n_jobs) : shape(eap::gemv_shape(n_cols, L, n_jobs)) {
    const size_t hb = shape.h / 4;
    lo = eap::PTS * sizeof(eap::Factors);
    mid = lo + eap::PTS * (sizeof(qm31) << eap::LO_BITS);
    hi = mid + ((size_t)eap::PTS * 64 << shape.r_log);
    partial = hi + eap::PTS * sizeof(qm31) * shape.h;
    end = partial + (hb > 1 ? eap::PTS * sizeof(qm31) * hb * n_cols : 0);
    require(end <= eval_at_point_columns_scratch_bytes(n_cols, L), "eval_at_point_columns: scratch layout");
  }
};
}  // namespace

// Small columns (log < 12) at one point.
static void eval_at_point_small_columns_async(const uint32_t* const* d_cols, uint32_t n_cols, uint32_t L,
                                              const qm31* d_point, qm31* d_out, void* d_scratch, uint32_t n_jobs,
                                              uint64_t js) {
  static_assert(eap::MIN_GEMV_LOG == eap::CB + 1, "a small column is one block");
  eap::Factors* F = (eap::Factors*)d_scratch;
  timed("eval_at_point", [&] {
    eap::factors_kernel<<<dim3(1, 1, n_jobs), 1, 0, ctx().cur>>>(d_point, L, F, js);
    eap::fold_cols<<<dim3(1, n_cols, n_jobs), eap::NT, 0, ctx().cur>>>(d_cols, L, F, d_out, js);
  });
}

// d_out[k n_cols + c] = value at point k, d_points[2k], d_points[2k + 1] = (x, y), of the polynomial
// with coefficients d_cols[c] (2^L each); two points at a time.  factors (host, one per point) saves
// computing the points' factors on the device; d_points is not read then.
// n_jobs / js: same-shape jobs of a batched launch, js bytes apart (points, output, scratch and
// columns all move by the job's offset).
void eval_at_points_columns_async(const uint32_t* const* d_cols, uint32_t n_cols, uint32_t L, uint32_t n_points,
                                  const qm31* d_points, const eap::Factors* d_factors, qm31* d_out, void* d_scratch,
                                  uint32_t n_jobs, uint64_t js) {
  // coefficient offsets are formed in 32 bits (gmem.hpp): at most 2^30 coefficients
  require(L >= 1 && L <= 30 && n_cols >= 1 && n_cols <= 65535, "eval_at_point_columns: bad sizes");
  if (L >= eap::MIN_GEMV_LOG) {
    const GemvLayout Y(n_cols, L, n_jobs);
    char* const base = (char*)d_scratch;
    eap::Factors* F = (eap::Factors*)base;
    qm31 *lo = (qm31*)(base + Y.lo), *hi = (qm31*)(base + Y.hi), *partial = (qm31*)(base + Y.partial);
    uint32_t* mid = (uint32_t*)(base + Y.mid);
    const uint32_t hb = Y.shape.h / 4;
    const uint32_t n_table = (1u << Y.shape.r_log) + (1u << eap::LO_BITS) + Y.shape.h;
    for (uint32_t k = 0; k < n_points; k += eap::PTS) {
      const uint32_t np = std::min(eap::PTS, n_points - k);
      qm31* const out = d_out + (size_t)k * n_cols;
      timed("eval_at_point", [&] {
        if (!d_factors)
          for (uint32_t p = 0; p < np; p++)
            eap::factors_kernel<<<dim3(1, 1, n_jobs), 1, 0, ctx().cur>>>(d_points + 2 * (k + p), L, F + p, js);
        eap::basis_tables_kernel<<<dim3(ceil_div(n_table, 256), eap::PTS, n_jobs), 256, 0, ctx().cur>>>(
            d_factors ? d_factors + k : F, np, L, Y.shape.r_log, Y.shape.h, mid, lo, hi, js);
        eap::gemv_kernel<<<dim3(hb, n_cols, n_jobs), 256, 0, ctx().cur>>>(
            d_cols, n_cols, Y.shape.r_log, Y.shape.h, np, mid, lo, hi, hb > 1 ? partial : out, js);
        if (hb > 1)
          eap::sum_partials_kernel<<<dim3(n_cols * np, 1, n_jobs), 256, 0, ctx().cur>>>(partial, hb, out, js);
      });
    }
    return;
  }
  for (uint32_t k = 0; k < n_points; k++)
    eval_at_point_small_columns_async(d_cols, n_cols, L, d_points + 2 * k, d_out + (size_t)k * n_cols, d_scratch, n_jobs,
                                      js);
}

qm31 eval_at_point_sync(const uint32_t* coeffs, uint64_t n, qm31 px, qm31 py) {
  require(is_pow2(n) && n <= (1ull << 30), "eval_at_point: size must be a power of two <= 2^30");
  uint32_t L = log2_exact(n);
  if (L == 0) {
    uint32_t c0;
    hip_check(hipMemcpyAsync(&c0, coeffs, 4, hipMemcpyDeviceToHost, ctx().stream), "hipMemcpy");
    sync();
    return qm31{{c0, 0}, {0, 0}};
  }
  eap::Factors F{};
  F.f[L - 1] = py;
  qm31 x = px;
  for (uint32_t i = 2; i <= L; i++) {
    F.f[L - i] = x;
    x = qsub(qadd(qsqr(x), qsqr(x)), qone());
  }
  uint32_t cb = std::min<uint32_t>(L, eap::CB);
  uint32_t blocks = 1u << (L - cb);
  DevBuf pa(sizeof(qm31) * blocks), pb(sizeof(qm31) * blocks);
  timed("eval_at_point", [&] {
    eap::first_pass<<<blocks, eap::NT, 0, ctx().cur>>>(coeffs, L, cb, F, pa.as<qm31>());
  });
  int fi = (int)(L - cb) - 1;
  while (blocks > 1) {
    uint32_t lb = log2_exact(blocks);
    uint32_t g = std::min<uint32_t>(lb, eap::CB - 1);
    uint32_t nb = blocks >> g;
    timed("eval_at_point", [&] {
      eap::reduce_pass<<<nb, eap::NT, 0, ctx().cur>>>(pa.as<qm31>(), g, F, fi, pb.as<qm31>());
    });
    std::swap(pa.p, pb.p);
    fi -= (int)g;
    blocks = nb;
  }
  qm31 r;
  hip_check(hipMemcpyAsync(&r, pa.p, sizeof(qm31), hipMemcpyDeviceToHost, ctx().stream), "hipMemcpy");
  sync();
  return r;
}

}  // namespace sh

using namespace sh;

extern "C" StwoQM31 eval_at_point(const uint32_t* coeffs, uint32_t coeffs_size, StwoQM31 point_x, StwoQM31 point_y) {
  StwoQM31 out{0, 0, 0, 0};
  guarded([&] {
    qm31 r = eval_at_point_sync(coeffs, coeffs_size, qm31{{point_x.a, point_x.b}, {point_x.c, point_x.d}},
                                qm31{{point_y.a, point_y.b}, {point_y.c, point_y.d}});
    out = StwoQM31{r.x.a, r.x.b, r.y.a, r.y.b};
  });
  return out;
}

extern "C" int stwo_hip_eval_at_points_columns(const uint32_t* const* columns, uint32_t n_cols, uint32_t log_size,
                                               const StwoCirclePointQM31* points, uint32_t n_points,
                                               StwoQM31* values) {
  return guarded([&] {
    require(columns != nullptr && values != nullptr && points != nullptr && n_cols >= 1 && n_points >= 1 &&
                log_size >= 1 && log_size <= 30,
            "eval_at_points_columns: bad arguments");
    // one upload: the points' factors (columns of log >= 12) or the points, then the pointer table
    const bool gemv = log_size >= eap::MIN_GEMV_LOG;
    const size_t p_bytes = (size_t)n_points * (gemv ? sizeof(eap::Factors) : 2 * sizeof(qm31));
    std::vector<unsigned char> host(p_bytes + (size_t)n_cols * sizeof(void*));
    for (uint32_t k = 0; k < n_points; k++) {
      const StwoCirclePointQM31& q = points[k];
      const qm31 x = {{q.x.a, q.x.b}, {q.x.c, q.x.d}}, y = {{q.y.a, q.y.b}, {q.y.c, q.y.d}};
      if (gemv) {
        eap::Factors F{};
        eap::point_factors(x, y, log_size, F);
        memcpy(host.data() + k * sizeof(F), &F, sizeof(F));
      } else {
        memcpy(host.data() + 2 * k * sizeof(qm31), &x, sizeof(qm31));
        memcpy(host.data() + (2 * k + 1) * sizeof(qm31), &y, sizeof(qm31));
      }
    }
    memcpy(host.data() + p_bytes, columns, (size_t)n_cols * sizeof(void*));
    // input and scratch in one block; the last kernel writes the values to host memory (more than
    // HOST_BLOCK_MAX bytes of them to the device first, which keeps the pinned buffers small)
    const size_t in_bytes = (host.size() + 255) & ~(size_t)255;
    const size_t out_bytes = sizeof(qm31) * n_cols * (size_t)n_points;
    const size_t scratch_bytes = (eval_at_point_columns_scratch_bytes(n_cols, log_size) + 255) & ~(size_t)255;
    const bool to_host = out_bytes <= HOST_BLOCK_MAX;
    DevBuf dev(in_bytes + scratch_bytes + (to_host ? 0 : out_bytes));
    unsigned char* const base = dev.as<unsigned char>();
    upload_to(base, host.data(), host.size());
    const uint32_t* const* table = (const uint32_t* const*)(base + p_bytes);
    auto enqueue = [&](qm31* out) {
      eval_at_points_columns_async(table, n_cols, log_size, n_points, dev.as<qm31>(),
                                   gemv ? dev.as<eap::Factors>() : nullptr, out, base + in_bytes, 1, 0);
    };
    if (to_host) {
      HostBlock out(out_bytes);
      enqueue(out.as<qm31>());
      sync();
      memcpy(values, out.as<void>(), out_bytes);
    } else {
      qm31* const out = (qm31*)(base + in_bytes + scratch_bytes);
      enqueue(out);
      hip_check(hipMemcpyAsync(values, out, out_bytes, hipMemcpyDeviceToHost, ctx().cur), "hipMemcpyAsync D2H");
      sync();
    }
  });
}

// ---- the batched evaluation with no device allocation ----------------------------------
// For callers that cannot allocate (code under graph capture, serving loops, harnesses that
// forbid hipMalloc): the pointer table, the points, the values and the partial sums live in
// this fixed array instead of pooled buffers.  Each device holds its own copy until the
// process ends.  Every call on a device shares that copy, so calls that overlap on one device
// race; nothing in it has to start at zero (every partial is written before it is read).
namespace {
constexpr size_t NOALLOC_BYTES = 32u << 20;
__device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];
constexpr int MAX_DEVICES = 64;
void* g_scratch[MAX_DEVICES];  // device address of `scratch` per device, under the library lock

// The device address of this device's `scratch` (the array's name is only a host-side
// stand-in); looked up on the first call on each device, with that device current.
void* noalloc_scratch() {
  const int dev = ctx().device;
  require(dev >= 0 && dev < MAX_DEVICES, "eval_at_points_columns_noalloc: device index out of range");
  if (!g_scratch[dev]) {
    void* p = nullptr;
    hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    require(p != nullptr, "eval_at_points_columns_noalloc: no device address for the scratch array");
    g_scratch[dev] = p;
  }
  return g_scratch[dev];
}
size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }
}  // namespace

extern "C" int stwo_hip_eval_at_points_columns_noalloc(const uint32_t* const* columns, uint32_t n_cols,
                                                       uint32_t log_size, const StwoCirclePointQM31* points,
                                                       uint32_t n_points, StwoQM31* values) {
  return guarded([&] {
    require(columns != nullptr && values != nullptr && points != nullptr && n_cols >= 1 && n_points >= 1 &&
                log_size >= 1 && log_size <= 30 && n_cols <= 65535,
            "eval_at_points_columns_noalloc: bad arguments");
    const size_t t_bytes = align256((size_t)n_cols * sizeof(void*));
    const size_t p_bytes = align256(2 * sizeof(qm31) * (size_t)n_points);
    const size_t o_bytes = align256(sizeof(qm31) * (size_t)n_cols * n_points);
    const size_t need = t_bytes + p_bytes + o_bytes + eval_at_point_columns_scratch_bytes(n_cols, log_size);
    if (need > NOALLOC_BYTES)
      fail(STWO_HIP_ERR_ARG,
           "eval_at_points_columns_noalloc: %u columns of log %u at %u points need %zu scratch bytes; the "
           "fixed scratch holds %zu",
           n_cols, log_size, n_points, need, NOALLOC_BYTES);
    char* base = (char*)noalloc_scratch();
    const uint32_t** table = (const uint32_t**)base;
    qm31* dpt = (qm31*)(base + t_bytes);
    qm31* out = (qm31*)(base + t_bytes + p_bytes);
    void* work = base + t_bytes + p_bytes + o_bytes;
    // points in the kernels' (x, y) layout; QM31 words are (a, b, c, d) in both
    static_assert(sizeof(StwoCirclePointQM31) == 2 * sizeof(qm31), "point layout");
    hipStream_t s = ctx().cur;
    hip_check(hipMemcpyAsync(table, columns, (size_t)n_cols * sizeof(void*), hipMemcpyHostToDevice, s),
              "hipMemcpyAsync H2D");
    hip_check(hipMemcpyAsync(dpt, points, 2 * sizeof(qm31) * (size_t)n_points, hipMemcpyHostToDevice, s),
              "hipMemcpyAsync H2D");
    eval_at_points_columns_async(table, n_cols, log_size, n_points, dpt, nullptr, out, work, 1, 0);
    hip_check(hipMemcpyAsync(values, out, sizeof(qm31) * n_cols * (size_t)n_points, hipMemcpyDeviceToHost, s),
              "hipMemcpyAsync D2H");
    sync();
  });
}

extern "C" int stwo_hip_eval_at_point_columns(const uint32_t* const* columns, uint32_t n_cols, uint32_t log_size,
                                              StwoQM31 point_x, StwoQM31 point_y, StwoQM31* values) {
  const StwoCirclePointQM31 p{point_x, point_y};
  return stwo_hip_eval_at_points_columns(columns, n_cols, log_size, &p, 1, values);
}
