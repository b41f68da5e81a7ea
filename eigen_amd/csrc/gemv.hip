// gemv.hip -- matrix-vector products (C with one column or one row).
//
// Eigen sends a product whose result is a vector to its GEMV kernels
// instead of GEBP (GeneralMatrixMatrix.h:480-490 ->
// Eigen/src/Core/products/GeneralMatrixVector.h:71-289, the column-major
// "y += alpha*A*x" and row-major "y += alpha*A^T*x" kernels).  Such a
// product reads every element of the matrix once and does two flops per
// element, so it is bound by HBM bandwidth; MFMA tiles would waste all but
// one column.  Two streaming kernels:
//
//   gemv_n_kernel  op(A)(i,k) = A[i + k*lda] (rows contiguous): each thread
//                  owns 16 contiguous bytes of rows and walks k, the vector
//                  element of each k being wave-uniform (scalar loads);
//   gemv_t_kernel  op(A)(i,k) = A[k + i*lda] (k contiguous): each wave walks
//                  one row (or four short ones), lanes reading 16-byte chunks
//                  along k against x in LDS, then reduces across the wave;
//   gemv_t_short_kernel  the same for rows of at most one chunk per lane,
//                  eight to a wave.
//
// Both split K over a second grid dimension when the rows alone cannot fill
// the chip; partial sums go to the workspace and are added in a fixed order
// (deterministic), by a reduction kernel or, for Aᵀx where the caller has
// tickets to give, by the last workgroup of each row block.  Operands are read through
// raw buffer resources: reads past the end of the matrix return zero and
// rows past m only feed outputs that are never stored.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace eh {

template <typename T>
struct GemvParams {
  const T* A;
  const T* x;
  T* y;
  T* W;            // split-K partials (splits x m) or nullptr
  int64_t lda, incx, incy;
  int m, k, k_per_split;
  uint32_t bytesA;  // extent of A from its base pointer (< 2^32, checked on the host)
  T alpha, beta;
  unsigned* tickets;  // with W: one zero word per row block, or nullptr (gemv_reduce_kernel follows)
};

// DEV: partial sums carry the device scope, for another workgroup of this
// launch, on any XCD, that may add them up.  Past the L2 they cost
// more, so sums for the next launch do without (FP32 Ax 4096^2 17.1 -> 16.1 us).
template <bool DEV, typename T>
__device__ inline void gemv_store(const GemvParams<T>& p, int i, T acc, int z) {
  if (p.W) {
    T* dst = &p.W[(int64_t)z * p.m + i];
    if constexpr (DEV)
      __hip_atomic_store(dst, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
      *dst = acc;
  } else {
    T* dst = p.y + (int64_t)i * p.incy;
    *dst = (p.beta == T(0)) ? p.alpha * acc : fma_t(p.alpha, acc, p.beta * *dst);
  }
}

// y from the partial sums of row i, in split order; loads issued sixteen at a
// time so that a long split list costs splits/16 memory latencies, not splits.
template <bool DEV, typename T>
__device__ inline void gemv_add_splits(const GemvParams<T>& p, int i, int splits) {
  T s = T(0);
  for (int z = 0; z < splits; z += 16) {
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      const T* src = &p.W[(int64_t)min(z + u, splits - 1) * p.m + i];
      v[u] = DEV ? __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : *src;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) s = z + u < splits ? s + v[u] : s;
  }
  T* dst = p.y + (int64_t)i * p.incy;
  *dst = (p.beta == T(0)) ? p.alpha * s : fma_t(p.alpha, s, p.beta * *dst);
}

// After a workgroup's partial sums: the last one of the row block to get here
// adds the block's rows [i0, i1) up, in place of a second launch.  Aᵀx only: Ax
// has few row blocks and many splits, and one workgroup adding them took longer
// than a launch (FP64 300 x 12000: 20.7 against 18.1 us).
template <typename T>
__device__ inline void gemv_finish(const GemvParams<T>& p, int i0, int i1) {
  if (!p.tickets) return;
  __shared__ int last;
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's partial sums have reached memory
  __syncthreads();
  if (threadIdx.x == 0) {
    last = atomicAdd(&p.tickets[blockIdx.x], 1u) == gridDim.y - 1;
    if (last) __hip_atomic_store(&p.tickets[blockIdx.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;
  for (int i = i0 + threadIdx.x; i < i1; i += blockDim.x) gemv_add_splits<true>(p, i, gridDim.y);
}

// A's loads, with the non-temporal hint (NT) when the matrix will not be found
// in the 256 MB last-level cache by the next call anyway: it then reads 10%
// faster (16384^2 FP64 A^T x 369 -> 331 us, Ax 361 -> 328; FP32 A^T x 204 ->
// 181).  Below 256 MB a matrix may stay there between calls and be read faster
// without the hint: A^T x of 192 MB 37.6 -> 34.2 us when it does not, 31.0 ->
// 33.9 when it does, Ax 39.5 -> 37.6 and 31.7 -> 35.7.  So A^T x takes the hint
// from half that cache on, which survives only if little else is used, Ax from
// all of it; small matrices lose either way (Ax 500 x 4000 11.8 -> 17.3).
template <bool NT>
__device__ inline u32x4 matrix_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return NT ? buf_load16_stream(r, voff, soff) : buf_load16(r, voff, soff);
}
// Short columns of Ax share lines with their neighbours, which the hint drops
// between the two reads: FP64 250 x 400,000 155 us without, 173 with it, 500 x
// 200,000 143 and 126; FP32 100 x 1,000,000 339 and 359, 500 x 200,000 101 and 96.
bool gemv_streams(bool trans, int m, uint32_t bytes) {
  return bytes >= (trans ? 128u : 256u) << 20 && (trans || m >= 384);
}

// k unroll of gemv_n_kernel (loads in flight per thread): 16 for FP64
// (16384^2: 370 -> 362 us), 8 for FP32 (16 measured 2% slower).
__host__ __device__ constexpr int gemv_n_unroll(int es) { return es == 8 ? 16 : 8; }

// 256 threads x EPT rows; k range of split blockIdx.y, unrolled by U.
template <typename T, bool NT>
__global__ void __launch_bounds__(256) gemv_n_kernel(GemvParams<T> p) {
  constexpr int EPT = 16 / sizeof(T);
  constexpr int U = gemv_n_unroll((int)sizeof(T));
  const int i0 = (blockIdx.x * 256 + threadIdx.x) * EPT;
  const int z = blockIdx.y;
  const int kb = z * p.k_per_split, ke = min(p.k, kb + p.k_per_split);
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, p.bytesA);
  const uint32_t vo = (uint32_t)i0 * sizeof(T);
  T acc[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) acc[e] = T(0);
  int kk = kb;
  for (; kk + U <= ke; kk += U) {
    u32x4 v[U];
    T xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = matrix_load<NT>(rA, vo, (uint32_t)((uint64_t)(kk + u) * p.lda * sizeof(T)));
      xv[u] = p.x[(int64_t)(kk + u) * p.incx];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const T* a = reinterpret_cast<const T*>(&v[u]);
#pragma unroll
      for (int e = 0; e < EPT; ++e) acc[e] = fma_t(a[e], xv[u], acc[e]);
    }
  }
  for (; kk < ke; ++kk) {
    const u32x4 v = matrix_load<NT>(rA, vo, (uint32_t)((uint64_t)kk * p.lda * sizeof(T)));
    const T xv = p.x[(int64_t)kk * p.incx];
    const T* a = reinterpret_cast<const T*>(&v);
#pragma unroll
    for (int e = 0; e < EPT; ++e) acc[e] = fma_t(a[e], xv, acc[e]);
  }
#pragma unroll
  for (int e = 0; e < EPT; ++e)
    if (i0 + e < p.m) gemv_store<false>(p, i0 + e, acc[e], z);
}

// Sum over the 64 lanes of a wave (butterfly, every lane ends with the sum).
template <typename T>
__device__ inline T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Eight waves; the workgroup's rows [blockIdx.x * rows, + rows) over the k range
// of split blockIdx.y, whose part of x lies in LDS.  A wave walks RB rows at a
// time, each a contiguous stream of 1 KB loads, RB*U of them in flight: of one
// row when the range is long, of four when it is short.  HBM bound.  Against
// eight rows of 1 KB per wave with x read from L1, K split only by doubling:
// FP64 6000 x 4001 43 -> 38 us (5.1 TB/s, matrix not in cache), 2000 x 2500 38
// -> 12, 16384 x 256 25 -> 12, 5000 x 10000 86 -> 75; with the non-temporal hint
// (matrix_load) 34, 68 and, 16384^2, 351 -> 331 (6.5 TB/s); FP32 16384^2 178 ->
// 181.
constexpr int kGemvTWaves = 8;
constexpr int kGemvTBytes = 32768;  // of x in LDS: four workgroups per CU, whole batches of U chunks
// PARTS: the split is longer than one LDS part; the parts follow one another,
// the sums of the workgroup's rows so far in LDS (16M FP64 elements by one row:
// 79 us, 172 with one split per part, whose 1954 sums one thread added).
template <typename T, int RB, int U, bool NT, bool PARTS>
__global__ void __launch_bounds__(64 * kGemvTWaves, 8) gemv_t_kernel(GemvParams<T> p, int rows) {
  constexpr int EPT = 16 / sizeof(T);
  constexpr int CH = 64 * EPT;  // elements of one load of a wave
  constexpr int PART = kGemvTBytes / sizeof(T);
  __shared__ __attribute__((aligned(16))) T xs[PART];
  __shared__ T sums[PARTS ? 2 * kGemvTWaves * RB : 1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int z = blockIdx.y;
  const int kz = z * p.k_per_split, ke = min(p.k, kz + p.k_per_split);
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, p.bytesA);
  const int i0 = blockIdx.x * rows, i1 = min(p.m, i0 + rows);
  int kb = kz;
  do {
    const int len = PARTS ? min(ke - kb, PART) : ke - kb;
    const int chunks = (len + CH - 1) / CH;
    if (PARTS && kb != kz) __syncthreads();  // xs is free again
    for (int i = threadIdx.x; i < (chunks + U - 1) / U * U * CH; i += 64 * kGemvTWaves)
      xs[i] = i < len ? p.x[(int64_t)(kb + i) * p.incx] : T(0);
    __syncthreads();
    auto load = [&](int r, int c, u32x4(&v)[RB][U]) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const uint32_t vo = (uint32_t)(((uint64_t)min(r + b, p.m - 1) * p.lda + lane * EPT) * sizeof(T));
#pragma unroll
        for (int u = 0; u < U; ++u)
          v[b][u] = matrix_load<NT>(rA, vo, (uint32_t)((uint64_t)(kb + min(c + u, chunks - 1) * CH) * sizeof(T)));
      }
    };
    T acc[RB][EPT] = {};
    // every wave starts its rows at another batch of the range: rows a power of
    // two apart would otherwise all be read at one memory channel's addresses
    const int batches = (chunks + U - 1) / U;
    const int c0 = (int)((blockIdx.x * kGemvTWaves + wave) % batches) * U;
    int r = i0 + wave * RB, c = c0;
    while (r < i1) {
      u32x4 v[RB][U];
      load(r, c, v);
      const int cn = c + U >= chunks ? 0 : c + U;
      const bool row_ends = cn == c0;
      const int rn = row_ends ? r + kGemvTWaves * RB : r;
      if ((c + U) * CH > len) {
        // elements past the range (the next row's data, the next split's, a
        // repeated chunk) meet x = 0 only if they are finite; select them away
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < EPT; ++e) {
              T* a = reinterpret_cast<T*>(&v[b][u]);
              a[e] = (c + u) * CH + lane * EPT + e < len ? a[e] : T(0);
            }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const u32x4 xv = *reinterpret_cast<const u32x4*>(&xs[(c + u) * CH + lane * EPT]);
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
          for (int e = 0; e < EPT; ++e)
            acc[b][e] = fma_t(reinterpret_cast<const T*>(&v[b][u])[e], reinterpret_cast<const T*>(&xv)[e], acc[b][e]);
      }
      if (row_ends) {
#pragma unroll
        for (int b = 0; b < RB; ++b) {
          T s = acc[b][0];
#pragma unroll
          for (int e = 1; e < EPT; ++e) s += acc[b][e];
          s = wave_sum(s);
          if (lane == 0 && r + b < i1) {
            if (PARTS && kb != kz) s += sums[r + b - i0];  // the wave's own: its rows are the same in every part
            if (PARTS && kb + len < ke)
              sums[r + b - i0] = s;
            else
              gemv_store<true>(p, r + b, s, z);
          }
#pragma unroll
          for (int e = 0; e < EPT; ++e) acc[b][e] = T(0);
        }
      }
      r = rn;
      c = cn;
    }
    kb += len;
  } while (PARTS && kb < ke);
  gemv_finish(p, i0, i1);
}

// Rows that end within one load of a wave (k <= 64 * EPT): a wave takes eight
// rows at once, x in registers, all eight loads in flight, and nothing is
// staged or split.  Bound by HBM at full rows and by the sums across the wave at
// short ones; gemv_t_kernel spends its two loads per row and the copy of x to
// LDS on rows that need neither: FP32 500,000 rows of 100 35.4 us (5.6 TB/s)
// against 80.8, 1,000,000 of 8 63 against 85, FP64 500,000 of 100 71 against 94.
// Rows that fill the chip two to a wave or not at all run so, since the sums of
// eight end later: FP32 1000 x 64 3.9 -> 2.4 us, 16,000 x 128 4.4 -> 3.5 (64,000:
// 7.4 -> 8.9), FP64 1000 x 64 4.0 -> 2.4, 64,000 x 128 14.3 -> 11.3.
constexpr int kGemvShortRows = 8;
template <typename T, int RW>
__global__ void __launch_bounds__(256) gemv_t_short_kernel(GemvParams<T> p) {
  constexpr int EPT = 16 / sizeof(T);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = (blockIdx.x * 4 + wave) * RW, kl = lane * EPT;
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, p.bytesA);
  u32x4 v[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) v[r] = buf_load16(rA, (uint32_t)(((uint64_t)(r0 + r) * p.lda + kl) * sizeof(T)), 0);
  T xv[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) xv[e] = kl + e < p.k ? p.x[(int64_t)(kl + e) * p.incx] : T(0);
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    const T* a = reinterpret_cast<const T*>(&v[r]);
    T acc = T(0);
    // elements past k (the next row's) meet x = 0 only if they are finite
#pragma unroll
    for (int e = 0; e < EPT; ++e) acc = fma_t(kl + e < p.k ? a[e] : T(0), xv[e], acc);
    const T s = wave_sum(acc);
    if (lane == 0 && r0 + r < p.m) gemv_store<false>(p, r0 + r, s, 0);
  }
}

template <typename T>
__global__ void __launch_bounds__(256) gemv_reduce_kernel(GemvParams<T> p, int splits) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < p.m; i += gridDim.x * 256) gemv_add_splits<false>(p, i, splits);
}

// Grid of a matrix-vector product: row blocks, and splits of K.
//
// Aᵀx: splits whose part of x fits in LDS (past kGemvTSplits of them, several
// parts to a split: one thread adds a row's partial sums, sixteen loads at a
// time), in whole batches of loads; among them, and one or two rows (or groups of rows) per wave, the plan whose rounds
// of resident workgroups (four per CU) stream the fewest bytes, x's part
// counted as one row and a workgroup's start as 16 KB.  More rows per workgroup
// leave the last round uneven (16384^2 FP64: 361, 363, 368 us with 16, 32, 64).
constexpr int kGemvTSplits = 256;
static GemvPlan gemv_t_plan(int m, int k, int es) {
  constexpr int kGroups = 1024;
  const int chunk = 64 * 16 / es;
  GemvPlan best{};
  if (k <= chunk) {  // gemv_t_short_kernel
    best.batch = kGemvShortRows;
    best.rows = 4 * (m <= (es == 8 ? 65536 : 16384) ? 2 : kGemvShortRows);
    best.blocks = (int)(((int64_t)m + best.rows - 1) / best.rows);
    best.splits = 1;
    best.per = k;
    return best;
  }
  double best_cost = 0;
  const int smin = (int)std::min<int64_t>(kGemvTSplits, ((int64_t)k * es + kGemvTBytes - 1) / kGemvTBytes);
  for (int s = smin; s == smin || (s < smin + 16 && s <= kGemvTSplits && (int64_t)k * es >= (int64_t)s * 4096); ++s) {
    int64_t per = ((int64_t)k + s - 1) / s;
    GemvPlan g{};
    g.batch = per >= 6 * chunk ? 1 : 4;
    const int whole = 8 * chunk / g.batch;  // whole batches: 8 KB of a row, or 2 KB
    per = (per + whole - 1) / whole * whole;
    g.per = (int)per;
    g.splits = (int)(((int64_t)k + per - 1) / per);
    const int step = kGemvTWaves * g.batch;
    for (g.rows = step; g.rows <= 2 * step; g.rows += step) {
      g.blocks = (m + g.rows - 1) / g.rows;
      const int64_t rounds = ((int64_t)g.blocks * g.splits + kGroups - 1) / kGroups;
      const double cost = (double)rounds * ((g.rows + 1.0) * (double)per * es + 16384.0);
      if (best.blocks == 0 || cost < best_cost) {
        best = g;
        best_cost = cost;
      }
    }
  }
  return best;
}

// Ax: about 256 workgroups' worth of streaming, one long-running workgroup per
// CU: each then streams long runs of its columns, where 2048 shorter workgroups
// measured 10-20% slower.  Below 128 columns no split, whose second launch takes
// longer than the columns (64^2: 10.3 us, 7.5 without).  Splits of 32 columns while they are few (FP64 12000 x
// 300: 15.1 -> 11.1 us, 1000^2 11.5 -> 10.3), of 64 after that: adding up many
// takes longer than they save (FP32 300 x 12000: 14.4 against 16.3 us).
GemvPlan gemv_plan(bool trans, int m, int k, int es) {
  if (trans) return gemv_t_plan(m, k, es);
  const int ept = 16 / es, chunk = gemv_n_unroll(es);
  GemvPlan g{};
  g.blocks = (m + 256 * ept - 1) / (256 * ept);
  int s = 1;
  while ((int64_t)g.blocks * s < 256 && k / (2 * s) >= (k >= 128 && s <= 16 ? 32 : 64) && s < 256) s *= 2;
  int64_t per = ((int64_t)k + s - 1) / s;
  per = (per + chunk - 1) / chunk * chunk;
  g.per = (int)per;
  g.splits = (int)(((int64_t)k + per - 1) / per);
  if (g.splits < 1) g.splits = 1;
  return g;
}

size_t gemv_workspace_bytes(const GemvPlan& g, int m, int es) {
  return g.splits > 1 ? (size_t)g.splits * m * es : 0;
}

template <typename T>
hipError_t launch_gemv(const GemvPlan& g, bool trans, int m, int k, T alpha, const T* A, int64_t lda,
                       uint32_t bytesA, const T* x, int64_t incx, T beta, T* y, int64_t incy, void* workspace,
                       unsigned* tickets, hipStream_t s) {
  GemvParams<T> p{};
  p.A = A;
  p.x = x;
  p.y = y;
  p.lda = lda;
  p.incx = incx;
  p.incy = incy;
  p.m = m;
  p.k = k;
  p.bytesA = bytesA;
  p.alpha = alpha;
  p.beta = beta;
  p.k_per_split = g.per;
  p.W = g.splits > 1 ? static_cast<T*>(workspace) : nullptr;
  p.tickets = trans && g.splits > 1 ? tickets : nullptr;
  dim3 grid((unsigned)g.blocks, (unsigned)g.splits);
  const bool nt = gemv_streams(trans, m, bytesA);
  const bool short_rows = trans && g.batch == kGemvShortRows;
  const dim3 threads(trans && !short_rows ? 64 * kGemvTWaves : 256);
  if (short_rows) {
    auto k = g.rows == 4 * kGemvShortRows ? gemv_t_short_kernel<T, kGemvShortRows> : gemv_t_short_kernel<T, 2>;
    hipLaunchKernelGGL(k, grid, threads, 0, s, p);
  } else if (trans) {
    const bool parts = (int64_t)g.per * (int)sizeof(T) > kGemvTBytes;
    auto k = parts          ? (nt ? gemv_t_kernel<T, 1, 8, true, true> : gemv_t_kernel<T, 1, 8, false, true>)
             : g.batch == 1 ? (nt ? gemv_t_kernel<T, 1, 8, true, false> : gemv_t_kernel<T, 1, 8, false, false>)
                            : (nt ? gemv_t_kernel<T, 4, 2, true, false> : gemv_t_kernel<T, 4, 2, false, false>);
    hipLaunchKernelGGL(k, grid, threads, 0, s, p, g.rows);
  } else {
    auto k = nt ? gemv_n_kernel<T, true> : gemv_n_kernel<T, false>;
    hipLaunchKernelGGL(k, grid, threads, 0, s, p);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || g.splits == 1 || p.tickets) return e;
  int64_t rb = (m + 255) / 256;
  if (rb > 65536) rb = 65536;
  hipLaunchKernelGGL(gemv_reduce_kernel<T>, dim3((unsigned)rb), dim3(256), 0, s, p, g.splits);
  return hipGetLastError();
}

template hipError_t launch_gemv<float>(const GemvPlan&, bool, int, int, float, const float*, int64_t, uint32_t,
                                       const float*, int64_t, float, float*, int64_t, void*, unsigned*, hipStream_t);
template hipError_t launch_gemv<double>(const GemvPlan&, bool, int, int, double, const double*, int64_t, uint32_t,
                                        const double*, int64_t, double, double*, int64_t, void*, unsigned*,
                                        hipStream_t);

}  // namespace eh
