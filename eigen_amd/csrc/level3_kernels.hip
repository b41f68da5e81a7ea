// level3_kernels.hip -- device kernels of the level-3 routines built on the product.
//
// Eigen runs TRMM, TRSM, SYMM and the rank updates on the same pack + GEBP
// engine as GEMM (Eigen/src/Core/products/TriangularMatrixMatrix.h,
// TriangularSolverMatrix.h, SelfadjointMatrixMatrix.h,
// GeneralMatrixMatrixTriangular.h).  Here the bulk of their flops goes to the
// MFMA product kernels through a blocking on the host; the kernels below do the
// rest:
//
//   tri_dense_kernel   the dense form of a matrix stored in one triangle:
//                      symmetric (mirror the stored triangle) or triangular
//                      (zeros outside it, optional unit diagonal).  64x64
//                      tiles; the mirrored half goes through LDS so that both
//                      the reads and the writes are coalesced.  HBM-bound.
//   trtri64_kernel     the inverses of all 64 x 64 diagonal blocks of a real
//                      triangular matrix in one launch (trtri_kernel: the 32 x
//                      32 blocks of a complex one);
//   trsm_panel_kernel  the solve of up to 512 rows of a real system for 16
//                      columns per workgroup, on those inverses.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace eh {

// T is a real type or cplx<R>; herm (complex only): the mirror is conjugated
// and the diagonal's imaginary part is dropped (BLAS ?hemm reads only the
// real part of a Hermitian diagonal); conj: every element is conjugated.
template <typename T>
__global__ void __launch_bounds__(256) tri_dense_kernel(const T* A, int64_t lda, int n, T* D, int64_t ldd, int lower,
                                                        int sym, int unit, int herm, int conj) {
  __shared__ T mir[64][65];
  const int bi = blockIdx.x * 64, bj = blockIdx.y * 64;  // D rows bi.., columns bj..
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  // (i, j) is stored when i >= j (lower) or i <= j (upper)
  auto stored = [&](int i, int j) { return lower ? i >= j : i <= j; };
  // does the tile hold elements outside the stored triangle?
  const bool mixed = lower ? bi < bj + 63 : bj < bi + 63;
  if (sym && mixed) {
    // mir[c][r] = A(bj + c, bi + r) = the mirror of D(bi + r, bj + c); lanes
    // walk rows of A (coalesced), only stored elements are read
    const int ar = bj + tx;
    for (int r = ty; r < 64; r += 4) {
      const int ac = bi + r;
      mir[tx][r] = (ar < n && ac < n && stored(ar, ac)) ? conj_if(A[ar + (int64_t)ac * lda], herm) : T(0);
    }
    __syncthreads();
  }
  const int i = bi + tx;
  if (i >= n) return;
  for (int r = ty; r < 64; r += 4) {
    const int j = bj + r;
    if (j >= n) break;
    T v;
    if (unit && i == j)
      v = T(1);
    else if (herm && i == j)
      v = real_part(A[i + (int64_t)j * lda]);
    else if (stored(i, j))
      v = A[i + (int64_t)j * lda];
    else
      v = sym ? mir[r][tx] : T(0);
    D[i + (int64_t)j * ldd] = conj_if(v, conj);
  }
}

template <typename T>
hipError_t launch_tri_dense(const T* A, int64_t lda, int n, T* D, int64_t ldd, bool lower, bool sym, bool unit,
                            hipStream_t s, bool herm, bool conj) {
  if (n <= 0) return hipSuccess;
  const unsigned nb = (unsigned)((n + 63) / 64);
  hipLaunchKernelGGL(tri_dense_kernel<T>, dim3(nb, nb), dim3(256), 0, s, A, lda, n, D, ldd, (int)lower, (int)sym,
                     (int)unit, (int)herm, (int)conj);
  return hipGetLastError();
}

// Inverses of the 64 x 64 diagonal blocks of a real triangular matrix, one
// workgroup of four waves per block: block b is M_b(i, k) = mt ? A[k + i*lda]
// : A[i + k*lda] at A + b*64 (1 + lda), of order nb = min(64, order - 64 b),
// lower or upper, unit diagonal or not; its inverse goes to W + b*64*64
// (ld 64, stored like M: column-major, or row-major when mt and not columns;
// zeros outside the triangle).  Entries of M_b outside
// its triangle and past nb are zero in LDS and the diagonal past nb is one.
// An upper block is inverted as the lower one its reversed rows and columns
// form.
//
// A block is a serial chain of 64 substitution steps, so latency bounds it.
// Only its four 16 x 16 diagonal blocks are inverted by substitution, one wave
// each, multiplying by the reciprocal of the diagonal as
// TriangularSolverMatrix.h:67 does; the rest follows from
//   inv([M11 0; M21 M22]) = [I1 0; -I2 (M21 I1), I2]
// on the matrix cores, twice (16 -> 32 -> 64).  One thread per column of the
// whole block (64 steps, 2048 unrolled multiply-adds) took 46.8 us for the 16
// FP64 blocks of order 1000; this takes
// 11.3 us.
template <typename T>
__global__ void __launch_bounds__(256) trtri64_kernel(TrtriParams<T> p) {
  using F = Mfma16<T>;
  constexpr int NB = 64;
  __shared__ T M[NB][NB + 1], V[NB][NB + 1], P[NB][33];
  __shared__ T dinv[NB];
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = min(NB, p.order - b * NB);
  const T* A = p.A + (int64_t)b * NB * (1 + p.lda);
  const bool rev = !p.lower;
#pragma unroll
  for (int q = 0; q < NB * NB / 256; ++q) {  // lanes walk the contiguous index of A
    const int c = lane, o = w + 4 * q;
    const int i = p.mt ? o : c, k = p.mt ? c : o;
    const bool in = i < nb && k < nb && (p.lower ? k < i : k > i);
    const T x = in ? A[c + (int64_t)o * p.lda] : T(0);
    M[rev ? NB - 1 - i : i][rev ? NB - 1 - k : k] = x;
    V[o][c] = T(0);
  }
  if (tid < NB) dinv[rev ? NB - 1 - tid : tid] = (tid >= nb || p.unit) ? T(1) : recip(A[tid + (int64_t)tid * p.lda]);
  __syncthreads();
  {  // 16 x 16 diagonal blocks: lane v < 16 of wave w solves for column v of block w
    const int o = 16 * w, v = lane & 15;
    T x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = i == v ? T(1) : T(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      x[i] *= dinv[o + i];
#pragma unroll
      for (int r = i + 1; r < 16; ++r) x[r] = fma_t(-M[o + r][o + i], x[i], x[r]);
    }
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i) V[o + i][o + v] = x[i];
    }
  }
  __syncthreads();
  const int li = lane & 15, lg = lane >> 4;
  // 16 x 16 block of X*Y over K terms, X and Y given by element functions
  auto product = [&](int K, auto x, auto y) {
    typename F::acc_t acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = T(0);
#pragma unroll
    for (int k = 0; k < K; k += 4) acc = F::mma(x(li, k + lg), y(k + lg, li), acc);
    return acc;
  };
  // 16 -> 32: waves 0 and 1 take the two pairs of blocks
  const int o = 32 * (w & 1);
  if (w < 2) {
    const auto t = product(16, [&](int i, int k) { return M[o + 16 + i][o + k]; }, [&](int k, int j) { return V[o + k][o + j]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) P[o + F::row(r, lane)][li] = t[r];
  }
  __syncthreads();
  if (w < 2) {
    const auto t = product(16, [&](int i, int k) { return V[o + 16 + i][o + 16 + k]; }, [&](int k, int j) { return P[o + k][j]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) V[o + 16 + F::row(r, lane)][o + li] = -t[r];
  }
  __syncthreads();
  // 32 -> 64: the 32 x 32 off-diagonal block, one 16 x 16 quarter per wave
  const int ti = 16 * (w & 1), tj = 16 * (w >> 1);
  {
    const auto t = product(32, [&](int i, int k) { return M[32 + ti + i][k]; }, [&](int k, int j) { return V[k][tj + j]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) P[ti + F::row(r, lane)][tj + li] = t[r];
  }
  __syncthreads();
  {
    const auto t = product(32, [&](int i, int k) { return V[32 + ti + i][32 + k]; }, [&](int k, int j) { return P[k][tj + j]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) V[32 + ti + F::row(r, lane)][tj + li] = -t[r];
  }
  __syncthreads();
  T* W = p.W + (int64_t)b * NB * NB;
#pragma unroll
  for (int q = 0; q < NB * NB / 256; ++q) {
    const int i = lane, k = w + 4 * q;
    // row-major: row i of the inverse is contiguous in W, else column k
    const bool rows = p.mt && !p.columns;
    const int r = rows ? k : i, c = rows ? i : k;
    W[i + k * NB] = rev ? V[NB - 1 - r][NB - 1 - c] : V[r][c];
  }
}

// Solve of one panel of a real triangular system in place: E X = alpha*B with
// E of order sz (lower or upper, E(i, k) = ta ? A[k + i*lda] : A[i + k*lda])
// and B's element (r, c) at B[r*rs + c*cs].  Columns are independent, so a
// workgroup takes 16 of them and holds them in LDS for the whole solve; E
// streams from the caches once per workgroup.  Per 64-row block b (in solve
// order)
//   Y = B_b - sum_{j solved} E(b, j) X_j,   X_b = inv(E_bb) Y
// as 16-row strips of 16x16x4 MFMAs.
//
// What bounds it: the chain of blocks, two dependent 64-deep products and
// three barriers each, and the matrix cores of the ceil(ncols / 16) CUs in
// use.  Sixteen waves, four per strip (and SIMD): the waves of group 0 run the
// chain -- E(b, b-1) X_(b-1), then the inverse -- while groups 1 to 3 share
// the products with the blocks solved earlier, one block ahead of the chain,
// so its latencies are filled with their MFMAs.  E does not depend on the
// solve: every wave loads its next 64-deep slab (16 values per lane) before it
// multiplies the current one, and the barriers wait for LDS only.
// A 512-row FP64 panel with 600 columns takes 38.5 us (15.4 us of MFMA issue on
// 38 CUs); with one group of waves and three slabs ahead in registers it took
// 52 us.
//
// With few right-hand sides every load of E is the first one anywhere, and a
// step waits for memory twice.  Up to eight workgroups leave most CUs idle, so
// the launch then holds readers as well: kPanelReaders workgroups on each of the
// workers' XCDs (workgroup x runs on XCD x % 8; elsewhere they only fill the
// shared last-level cache) read the blocks, in the order of the solve, into that
// L2 and compute nothing.  FP64, 16 right-hand sides: 42 -> 38 us a panel, order
// 12288 1450 -> 1365 us.
constexpr int kPanelReaders = 8;
inline int panel_readers_from(int workers, int nblk) { return workers <= 8 && nblk > 2 ? 8 * (1 + kPanelReaders) : workers; }

template <typename T, bool TA>
__device__ inline void panel_read(const TrsmPanelParams<T>& p, int nblk) {
  constexpr int NB = kTrsmLeaf, EPC = 16 / sizeof(T), V = NB / EPC * NB / 1024;  // loads of a thread per block
  constexpr int MOST = (8 * 7 / 2 + kPanelReaders - 1) / kPanelReaders;        // blocks of a reader
  const int me = blockIdx.x / 8 - 1;
  auto blk = [&](int s) { return p.lower ? s : nblk - 1 - s; };
  u32x4 sum = {};
  u32x4 v[MOST + 1][V];
  auto read = [&](const T* base, int64_t ld, int64_t bytes, u32x4(&t)[V]) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(base, (uint32_t)max((int64_t)0, min(bytes, (int64_t)0xFFFFFFF0)));
#pragma unroll
    for (int x = 0; x < V; ++x) {
      const int i = threadIdx.x + 1024 * x;
      t[x] = buf_load16(rs, (uint32_t)((i / (NB / EPC) * ld + i % (NB / EPC) * EPC) * sizeof(T)), 0);
    }
  };
  int s = 1, j = me;
#pragma unroll
  for (int q = 0; q < MOST; ++q, j += kPanelReaders) {
    while (j >= s) j -= s++;  // pair (s, j), j < s, number me + q*kPanelReaders
    const int r0 = blk(min(s, nblk - 1)) * NB, c0 = blk(min(j, nblk - 1)) * NB;
    const int64_t first = TA ? c0 + r0 * p.lda : r0 + c0 * p.lda, last = (p.sz - 1) * (p.lda + 1);
    read(p.A + first, p.lda, s < nblk ? (last - first + 1) * (int64_t)sizeof(T) : 0, v[q]);
  }
  read(p.inv + (int64_t)blk(min(me, nblk - 1)) * NB * NB, NB, NB * NB * sizeof(T), v[MOST]);
#pragma unroll
  for (int q = 0; q <= MOST; ++q)
#pragma unroll
    for (int x = 0; x < V; ++x) sum ^= v[q][x];
  if (p.sz < 0) p.B[0] = (T)(sum.x ^ sum.y ^ sum.z ^ sum.w);  // never: keeps the loads
}

template <typename T, bool TA>
__global__ void __launch_bounds__(1024) trsm_panel_kernel(TrsmPanelParams<T> p) {
  using F = Mfma16<T>;
  constexpr int NB = kTrsmLeaf, NC = 16, XS = NC + 1, NT = 1024, NH = 3;  // NH: helper groups
  constexpr int EPC = 16 / sizeof(T);  // consecutive k of one lane
  __shared__ T Xs[kTrsmPanel * XS];    // row r of the panel at Xs[r*XS]
  __shared__ T Y[NB * XS];
  __shared__ T R[NH][NB * XS];         // partial sums of the helper groups
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int strip = w & 3, group = w >> 2;
  const int li = lane & 15, lg = lane >> 4;
  const int c0 = blockIdx.x * NC;
  const int nblk = (p.sz + NB - 1) / NB;
  const int workers = (p.ncols + NC - 1) / NC;
  if ((int)blockIdx.x >= workers) {
    if (blockIdx.x >= 8 && (int)blockIdx.x % 8 < workers) panel_read<T, TA>(p, nblk);
    return;
  }
  T* B = p.B + c0 * p.cs;
  const int nc = min(NC, p.ncols - c0);
  auto blk = [&](int s) { return p.lower ? s : nblk - 1 - s; };  // block solved at step s

  // slab of E or of an inverse: lane's values v[q*EPC + e] = X(16 strip + li, k)
  // with k = 4*EPC*q + EPC*lg + e, q < 16 / EPC
  struct Slab {
    T v[16];
  };
  // The slab of E(blk(s), blk(j)), or of the inverse of block blk(s) when j <
  // 0, through a buffer resource based at the slab, so that a load costs one
  // scalar add.  Reads past the panel's last element return zero.
  const uint32_t vo_e = (uint32_t)((TA ? (int64_t)li * p.lda + EPC * lg : (int64_t)EPC * lg * p.lda + li) * sizeof(T));
  const uint32_t vo_i = (uint32_t)((TA ? li * NB + EPC * lg : EPC * lg * NB + li) * sizeof(T));
  auto load = [&](int s, int j) {
    Slab t;
    const bool inv = j < 0;
    const int64_t ld = inv ? NB : p.lda;
    const int i0 = (inv ? 0 : blk(s) * NB) + 16 * strip, k0 = inv ? 0 : blk(j) * NB, end = inv ? NB : p.sz;
    const int64_t first = TA ? k0 + i0 * ld : i0 + k0 * ld, last = (end - 1) * (ld + 1);
    const T* base = (inv ? p.inv + (int64_t)blk(s) * NB * NB : p.A) + first;
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(base, (uint32_t)max((int64_t)0, min((last - first + 1) * (int64_t)sizeof(T), (int64_t)0xFFFFFFF0)));
    const uint32_t vo = inv ? vo_i : vo_e;
    if constexpr (TA) {
#pragma unroll
      for (int q = 0; q < 16 / EPC; ++q)
        *reinterpret_cast<u32x4*>(&t.v[q * EPC]) = buf_load16(rs, vo, 4 * EPC * q * sizeof(T));
    } else {
#pragma unroll
      for (int q = 0; q < 16; ++q)
        t.v[q] = buf_load(rs, vo, (uint32_t)((4 * EPC * (q / EPC) + q % EPC) * ld * sizeof(T)), (T*)nullptr);
    }
    return t;
  };
  // acc + slab * x, x the 64 rows of LDS at `x`; k0: the slab's first column
  // of the panel (-NB: an inverse).  k-contiguous rows run on into the next
  // row past the panel's last column (the ragged last block of an upper
  // panel): zeros from there on.
  struct Acc {
    typename F::acc_t a, b;
  };
  auto multiply = [&](const Slab& t, const T* x, int k0, Acc& acc) {
    const int live = p.sz - max(k0, 0) - EPC * lg;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int k = 4 * EPC * (q / EPC) + q % EPC;
      const T a = !TA || k0 < 0 || k < live ? t.v[q] : T(0);
      const T y = x[(k + EPC * lg) * XS + li];
      if (q & 1)
        acc.b = F::mma(a, y, acc.b);
      else
        acc.a = F::mma(a, y, acc.a);
    }
  };
  auto clear = [&](Acc& acc) {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc.a[r] = acc.b[r] = T(0);
  };

  // panel -> LDS, threads along the contiguous index of B; zeros past sz and nc
  const bool rows_fast = p.rs == 1;
  const int rows = nblk * NB, total = rows * NC;
  auto fill = [&]() {
    for (int q = tid; q < total; q += NT) {
      const int r = rows_fast ? q % rows : q / NC, c = rows_fast ? q / rows : q % NC;
      Xs[r * XS + c] = r < p.sz && c < nc ? p.alpha * B[r * p.rs + c * p.cs] : T(0);
    }
  };
  // Both branches run the same barriers: one after the fill, three per step.
  if (group == 0) {
    __builtin_amdgcn_s_setprio(3);  // the chain's MFMAs go before the helpers'
    Slab inv = load(0, -1), sub = load(min(1, nblk - 1), 0);
    fill();
    lds_barrier();
    Acc acc;
    for (int s = 0; s < nblk; ++s) {
      const int b = blk(s), nx = min(s + 1, nblk - 1);
      clear(acc);
      if (s > 0) multiply(sub, Xs + blk(s - 1) * NB * XS, blk(s - 1) * NB, acc);
      if (s > 0) sub = load(nx, s);
      lds_barrier();  // the helpers' sums are in R
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * strip + F::row(r, lane), o = row * XS + li;
        T v = Xs[b * NB * XS + o] - (acc.a[r] + acc.b[r]);
        if (s > 1) v -= (R[0][o] + R[1][o]) + R[2][o];
        Y[o] = b * NB + row < p.sz ? v : T(0);
      }
      lds_barrier();  // Y
      clear(acc);
      multiply(inv, Y, -NB, acc);
      inv = load(nx, -1);
#pragma unroll
      for (int r = 0; r < 4; ++r) Xs[(b * NB + 16 * strip + F::row(r, lane)) * XS + li] = acc.a[r] + acc.b[r];
      lds_barrier();  // X of block b
    }
  } else {
    // E(s, j) for j = group - 1, group + 2, ... < s - 1, s = 2 ...
    int ns = group + 1, nj = group - 1;  // the next slab to load
    auto load_next = [&]() {
      const Slab t = load(min(ns, nblk - 1), min(nj, nblk - 1));
      nj += NH;
      if (nj >= ns - 1) {
        ++ns;
        nj = group - 1;
      }
      return t;
    };
    Slab next = load_next();
    fill();
    lds_barrier();
    Acc acc;
    clear(acc);
    int j = group - 1;  // the next product of the step ahead
    auto product = [&]() {
      const Slab cur = next;
      next = load_next();
      multiply(cur, Xs + blk(j) * NB * XS, blk(j) * NB, acc);
      j += NH;
    };
    for (int s = 0; s < nblk; ++s) {
      while (j < s - 1) product();
      if (s > 1) {
#pragma unroll
        for (int r = 0; r < 4; ++r) R[group - 1][(16 * strip + F::row(r, lane)) * XS + li] = acc.a[r] + acc.b[r];
      }
      lds_barrier();  // R
      lds_barrier();  // Y
      clear(acc);
      j = group - 1;
      if (j < s && s + 1 < nblk) product();  // blocks before s are solved
      lds_barrier();  // X of block blk(s)
    }
  }
  for (int q = tid; q < total; q += NT) {
    const int r = rows_fast ? q % rows : q / NC, c = rows_fast ? q / rows : q % NC;
    if (r < p.sz && c < nc) B[r * p.rs + c * p.cs] = Xs[r * XS + c];
  }
}

template <typename T>
hipError_t launch_trsm_panel(const TrsmPanelParams<T>& p, hipStream_t s) {
  if (p.sz <= 0 || p.ncols <= 0) return hipSuccess;
  if (p.sz > kTrsmPanel) return hipErrorInvalidValue;
  const dim3 grid((unsigned)panel_readers_from((p.ncols + 15) / 16, (p.sz + kTrsmLeaf - 1) / kTrsmLeaf));
  if (p.ta)
    hipLaunchKernelGGL((trsm_panel_kernel<T, true>), grid, dim3(1024), 0, s, p);
  else
    hipLaunchKernelGGL((trsm_panel_kernel<T, false>), grid, dim3(1024), 0, s, p);
  return hipGetLastError();
}
template hipError_t launch_trsm_panel<float>(const TrsmPanelParams<float>&, hipStream_t);
template hipError_t launch_trsm_panel<double>(const TrsmPanelParams<double>&, hipStream_t);

// The panels' off-diagonal 64 x 64 blocks of a triangle with contiguous rows,
// turned through LDS; workgroup (q, p) takes the q-th pair of blocks of panel p.
// The panel kernel reads contiguous rows 64 bytes at a time, of sixteen rows at
// once: FP64 rows a multiple of 128 bytes apart then all want the same halves of
// their lines, and a panel of 512 takes 54 us instead of 36 (44 at other leading
// dimensions).  One pass over the panels, each read by every workgroup of 16
// right-hand sides, costs 3 us for one panel and about 1 for each further:
// order 8192, 16 right-hand sides, transposed: 1153 -> 870 us.
template <typename T>
__global__ void __launch_bounds__(256) turn_panels_kernel(const T* A, int64_t lda, int order, int lower, T* D, int ldd) {
  constexpr int NB = kTrsmLeaf;
  __shared__ T tile[NB][NB + 1];
  int bi = 1, bj = blockIdx.x;  // bi > bj
  while (bj >= bi) bj -= bi++;
  if (!lower) {
    const int t = bi;
    bi = bj;
    bj = t;
  }
  const int64_t d = (int64_t)blockIdx.y * kTrsmPanel;
  const int i0 = bi * NB, k0 = bj * NB, sz = (int)min((int64_t)kTrsmPanel, order - d);
  if (max(i0, k0) >= sz) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  A += d * (1 + lda);
  D += d * ldd;
#pragma unroll
  for (int q = 0; q < NB / 4; ++q) {
    const int i = w + 4 * q;
    tile[i][lane] = i0 + i < sz && k0 + lane < sz ? A[k0 + lane + (int64_t)(i0 + i) * lda] : T(0);
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NB / 4; ++q) {
    const int k = w + 4 * q;
    D[i0 + lane + (int64_t)(k0 + k) * ldd] = tile[lane][k];
  }
}
template <typename T>
hipError_t launch_turn_panels(const T* A, int64_t lda, int order, bool lower, T* D, int ldd, hipStream_t s) {
  if (order <= kTrsmLeaf) return hipSuccess;
  const int blocks = (std::min(order, kTrsmPanel) + kTrsmLeaf - 1) / kTrsmLeaf;
  const dim3 grid((unsigned)(blocks * (blocks - 1) / 2), (unsigned)((order + kTrsmPanel - 1) / kTrsmPanel));
  hipLaunchKernelGGL(turn_panels_kernel<T>, grid, dim3(256), 0, s, A, lda, order, (int)lower, D, ldd);
  return hipGetLastError();
}
template hipError_t launch_turn_panels<double>(const double*, int64_t, int, bool, double*, int, hipStream_t);

// D (m x n, ld m) = B, lanes along the columns' rows.
// Eight columns per workgroup and pass, all their loads before the first store
// (FP32 TRMM 1500 x 1100: 51.3 -> 48.5 us, 1000 x 100: 27.0 -> 24.5, against one
// element per thread and pass).
template <typename T>
__global__ void __launch_bounds__(256) copy_block_kernel(const T* B, int64_t ldb, int m, int n, T* D) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= m) return;
  for (int c0 = blockIdx.y * 8; c0 < n; c0 += gridDim.y * 8) {
    T v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) v[c] = B[r + (int64_t)min(c0 + c, n - 1) * ldb];
#pragma unroll
    for (int c = 0; c < 8; ++c)
      if (c0 + c < n) D[r + (int64_t)(c0 + c) * m] = v[c];
  }
}
template <typename T>
hipError_t launch_copy_block(const T* B, int64_t ldb, int m, int n, T* D, hipStream_t s) {
  if (m <= 0 || n <= 0) return hipSuccess;
  const dim3 grid((unsigned)((m + 255) / 256), (unsigned)std::min<int64_t>(((int64_t)n + 7) / 8, 65535));
  hipLaunchKernelGGL(copy_block_kernel<T>, grid, dim3(256), 0, s, B, ldb, m, n, D);
  return hipGetLastError();
}
template hipError_t launch_copy_block<float>(const float*, int64_t, int, int, float*, hipStream_t);
template hipError_t launch_copy_block<double>(const double*, int64_t, int, int, double*, hipStream_t);

// The same for complex types, blocks of order NB, one workgroup per
// block: block b is M_b(i, k) = mt ? A[k + i*lda] : A[i + k*lda] at A + b*NB
// (1 + lda), of order nb = min(NB, order - b*NB), lower or upper, unit
// diagonal or not.  Thread v solves M_b x = e_v by substitution, multiplying
// by the reciprocal of the diagonal as TriangularSolverMatrix.h:67 does, and
// writes column v of inv(M_b) to W + b*NB*NB (NB x NB, column-major, zero
// outside the triangle and past nb).  Entries of M_b outside its triangle
// and past nb are zero in LDS and the reciprocal diagonal past nb is one, so
// the unrolled substitution needs no guards.  Each dot product runs as two
// interleaved partial sums (half the dependent chain).  p.conj conjugates M,
// for an inverse of A^H's blocks.
template <typename T, int NB>
__global__ void __launch_bounds__(NB) trtri_kernel(TrtriParams<T> p) {
  __shared__ T M[NB][NB];
  __shared__ T dinv[NB];
  const int b = blockIdx.x;
  const int nb = min(NB, p.order - b * NB);
  const T* A = p.A + (int64_t)b * NB * (1 + p.lda);
  for (int idx = threadIdx.x; idx < NB * NB; idx += NB) {
    const int i = idx % NB, k = idx / NB;
    const bool in = i < nb && k < nb && (p.lower ? k < i : k > i);
    M[i][k] = in ? conj_if(p.mt ? A[k + (int64_t)i * p.lda] : A[i + (int64_t)k * p.lda], p.conj != 0) : T(0);
  }
  if (threadIdx.x < NB) {
    const int i = threadIdx.x;
    dinv[i] = (i >= nb || p.unit) ? T(1) : recip(conj_if(A[i + (int64_t)i * p.lda], p.conj != 0));
  }
  __syncthreads();
  const int v = threadIdx.x;
  T x[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) x[i] = (i == v && i < nb) ? T(1) : T(0);
  if (p.lower) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      T s0 = x[i], s1 = T(0);
#pragma unroll
      for (int k = 0; k + 1 < i; k += 2) {
        s0 = fma_t(-M[i][k], x[k], s0);
        s1 = fma_t(-M[i][k + 1], x[k + 1], s1);
      }
      if (i & 1) s0 = fma_t(-M[i][i - 1], x[i - 1], s0);
      x[i] = (s0 + s1) * dinv[i];
    }
  } else {
#pragma unroll
    for (int i = NB - 1; i >= 0; --i) {
      T s0 = x[i], s1 = T(0);
#pragma unroll
      for (int k = i + 1; k + 1 < NB; k += 2) {
        s0 = fma_t(-M[i][k], x[k], s0);
        s1 = fma_t(-M[i][k + 1], x[k + 1], s1);
      }
      if ((NB - 1 - i) & 1) s0 = fma_t(-M[i][NB - 1], x[NB - 1], s0);
      x[i] = (s0 + s1) * dinv[i];
    }
  }
  T* w = p.W + (int64_t)b * NB * NB + (int64_t)v * NB;
#pragma unroll
  for (int i = 0; i < NB; ++i) w[i] = x[i];
}

// Complex rank updates: on the lower (upper) triangle of the n x n result,
//   C(i, j) = alpha*W(i, j) + alpha2*f(W(j, i)) + beta*C(i, j)
// with f = conj when herm (the W^H term of HER2K) else identity (W^T of
// SYR2K), the alpha2 term only when use2, C not read when beta == 0, and
// (herm) the diagonal's imaginary part set to zero as ?herk / ?her2k do.
// W == nullptr: the W terms are zero (C = beta*C on the triangle).  64 x 64
// tiles, tiles off the triangle return at once; the transposed term goes
// through LDS so both its reads and the writes of C are coalesced.
template <typename R>
__global__ void __launch_bounds__(256) tri_combine_kernel(const cplx<R>* W, int64_t ldw, int n, cplx<R>* C,
                                                          int64_t ldc, int lower, cplx<R> alpha, cplx<R> alpha2,
                                                          int use2, cplx<R> beta, int herm) {
  __shared__ cplx<R> tr[64][65];
  const int bi = blockIdx.x * 64, bj = blockIdx.y * 64;  // C rows bi.., columns bj..
  if (lower ? bi + 63 < bj : bj + 63 < bi) return;      // the whole tile is off the triangle
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  if (W && use2) {
    // tr[c][r] = W(bj + c, bi + r): lanes walk rows of W (coalesced)
    const int wr = bj + tx;
    for (int r = ty; r < 64; r += 4) {
      const int wc = bi + r;
      tr[tx][r] = (wr < n && wc < n) ? W[wr + (int64_t)wc * ldw] : cplx<R>(0);
    }
    __syncthreads();
  }
  const int i = bi + tx;
  if (i >= n) return;
  const bool read_c = !(beta == cplx<R>(0));
  for (int r = ty; r < 64; r += 4) {
    const int j = bj + r;
    if (j >= n) break;
    if (lower ? i < j : i > j) continue;
    cplx<R> v(0);
    if (W) {
      v = alpha * W[i + (int64_t)j * ldw];
      if (use2) v = v + alpha2 * conj_if(tr[r][tx], herm != 0);
    }
    if (read_c) v = v + beta * C[i + (int64_t)j * ldc];
    if (herm && i == j) v.im = R(0);
    C[i + (int64_t)j * ldc] = v;
  }
}

template <typename R>
hipError_t launch_tri_combine(const cplx<R>* W, int64_t ldw, int n, cplx<R>* C, int64_t ldc, bool lower,
                              cplx<R> alpha, cplx<R> alpha2, bool use2, cplx<R> beta, bool herm, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const unsigned nb = (unsigned)((n + 63) / 64);
  hipLaunchKernelGGL(tri_combine_kernel<R>, dim3(nb, nb), dim3(256), 0, s, W, ldw, n, C, ldc, (int)lower, alpha, alpha2,
                     (int)use2, beta, (int)herm);
  return hipGetLastError();
}
template hipError_t launch_tri_combine<float>(const cplx<float>*, int64_t, int, cplx<float>*, int64_t, bool,
                                              cplx<float>, cplx<float>, bool, cplx<float>, bool, hipStream_t);
template hipError_t launch_tri_combine<double>(const cplx<double>*, int64_t, int, cplx<double>*, int64_t, bool,
                                               cplx<double>, cplx<double>, bool, cplx<double>, bool, hipStream_t);

template <typename T>
struct TrtriLaunch {  // real types
  static constexpr int NB = kTrsmLeaf, NT = 256;
  static constexpr auto kernel = trtri64_kernel<T>;
};
template <typename R>
struct TrtriLaunch<cplx<R>> {
  static constexpr int NB = kTrsmLeafComplex, NT = kTrsmLeafComplex;
  static constexpr auto kernel = trtri_kernel<cplx<R>, kTrsmLeafComplex>;
};

template <typename T>
hipError_t launch_trtri(const TrtriParams<T>& p, hipStream_t s) {
  if (p.order <= 0) return hipSuccess;
  using L = TrtriLaunch<T>;
  hipLaunchKernelGGL(L::kernel, dim3((unsigned)((p.order + L::NB - 1) / L::NB)), dim3(L::NT), 0, s, p);
  return hipGetLastError();
}

#define EH_L3_INST(T)                                                                                       \
  template hipError_t launch_tri_dense<T>(const T*, int64_t, int, T*, int64_t, bool, bool, bool, hipStream_t, \
                                          bool, bool);                                                      \
  template hipError_t launch_trtri<T>(const TrtriParams<T>&, hipStream_t);
EH_L3_INST(float)
EH_L3_INST(double)
EH_L3_INST(cplx<float>)
EH_L3_INST(cplx<double>)
#undef EH_L3_INST

}  // namespace eh
