// gemm_small.hip -- plain FP32 / FP64 products of small matrices.
//
// A product with a few dozen to a few hundred rows, columns and k is over in
// the time of a few memory latencies, and gemm_mfma_kernel's 64x64 tiles give
// it a handful of workgroups that walk their k slices one latency after
// another.  Here a workgroup computes 32x32 of C and its eight waves share the
// k range: every wave loads its operands straight into MFMA registers (four
// steps in flight, no LDS staging), and the eight partial tiles meet in LDS,
// summed in wave order.  Latency bound; calls of 64x64 tiles (with split K)
// against this kernel, host and launch included: FP32 96x80x112 10.3 -> 8.1 us,
// FP64 308x281x136 13.3 -> 8.2, 512^3 17.7 -> 9.4.
#include "common.hpp"
#include "kernels.hpp"

namespace eh {

constexpr int kSmallWaves = 8;

template <typename T, bool TA, bool TB>
__global__ void __launch_bounds__(64 * kSmallWaves) gemm_small_kernel(GemmParams<T> p) {
  using F = Mfma<T>;
  constexpr int B = kSmallTile, RM = B / F::MI;
  constexpr int EPC = 16 / sizeof(T);
  constexpr int KD = F::KG * EPC;  // k of one step: EPC MFMAs deep
  constexpr int U = 4;             // steps in flight
  constexpr uint32_t SZ = sizeof(T);
  constexpr uint32_t kOutside = 0x80000000u;  // past any operand (the host keeps them below 2 GB): reads zero
  __shared__ T part[kSmallWaves][B][B + 1];

  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane % F::MI, lg = lane / F::MI;
  const int ntm = (p.M + B - 1) / B;
  const int m0 = blockIdx.x % ntm * B, n0 = blockIdx.x / ntm * B;
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, p.bytesA), rB = make_rsrc(p.B, p.bytesB);

  // lane's first element of row block i at step 0; element e of a
  // rows-contiguous operand is e columns further
  uint32_t voA[RM], voB[RM];
#pragma unroll
  for (int i = 0; i < RM; ++i) {
    const int64_t ra = m0 + i * F::MI + li, rb = n0 + i * F::NI + li, k = lg * EPC;
    voA[i] = (uint32_t)((TA ? ra * p.lda + k : ra + k * p.lda) * SZ);
    voB[i] = (uint32_t)((TB ? rb + k * p.ldb : rb * p.ldb + k) * SZ);
  }
  auto load = [&](__amdgpu_buffer_rsrc_t rs, bool kcont, uint32_t vo, int s, int64_t ld, T(&t)[EPC]) {
    if (kcont) {
      const u32x4 v = buf_load16(rs, vo, (uint32_t)(s * KD) * SZ);
#pragma unroll
      for (int e = 0; e < EPC; ++e) t[e] = reinterpret_cast<const T*>(&v)[e];
    } else {
#pragma unroll
      for (int e = 0; e < EPC; ++e) t[e] = buf_load(rs, vo, (uint32_t)((uint64_t)(s * KD + e) * ld * SZ), (T*)nullptr);
    }
  };

  typename F::acc_t acc[RM][RM] = {};
  const int steps = (p.K + KD - 1) / KD, per = (steps + kSmallWaves - 1) / kSmallWaves;
  const int end = min(steps, (wid + 1) * per);
  for (int s = wid * per; s < end; s += U) {
    T a[U][RM][EPC], b[U][RM][EPC];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < RM; ++i) {
        const bool in = s + u < end;
        load(rA, TA, in ? voA[i] : kOutside, in ? s + u : 0, p.lda, a[u][i]);
        load(rB, !TB, in ? voB[i] : kOutside, in ? s + u : 0, p.ldb, b[u][i]);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < EPC; ++e) {
        // past K a k-contiguous operand holds the next row
        const bool in = (s + u) * KD + lg * EPC + e < p.K;
#pragma unroll
        for (int i = 0; i < RM; ++i) {
          if (TA) a[u][i][e] = in ? a[u][i][e] : T(0);
          if (!TB) b[u][i][e] = in ? b[u][i][e] : T(0);
        }
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RM; ++j) F::mma(a[u][i][e], b[u][j][e], acc[i][j]);
      }
  }
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RM; ++j)
#pragma unroll
      for (int r = 0; r < F::ACC; ++r)
        part[wid][j * F::NI + F::col(lane)][i * F::MI + F::row(r, lane)] = acc[i][j][r];
  __syncthreads();
#pragma unroll
  for (int x = 0; x < B * B / (64 * kSmallWaves); ++x) {
    const int r = threadIdx.x % B, c = threadIdx.x / B + x * (64 * kSmallWaves / B);
    T sum = T(0);
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) sum += part[w][c][r];
    if (m0 + r < p.M && n0 + c < p.N) {
      T* dst = p.C + m0 + r + (int64_t)(n0 + c) * p.ldc;
      *dst = p.beta == T(0) ? p.alpha * sum : fma_t(p.alpha, sum, p.beta * *dst);
    }
  }
}

template <typename T>
hipError_t launch_gemm_small(const GemmParams<T>& p, bool ta, bool tb, hipStream_t s) {
  const int64_t tiles = (int64_t)((p.M + kSmallTile - 1) / kSmallTile) * ((p.N + kSmallTile - 1) / kSmallTile);
  const dim3 grid((unsigned)tiles), threads(64 * kSmallWaves);
  if (!ta && !tb)
    hipLaunchKernelGGL((gemm_small_kernel<T, false, false>), grid, threads, 0, s, p);
  else if (ta && !tb)
    hipLaunchKernelGGL((gemm_small_kernel<T, true, false>), grid, threads, 0, s, p);
  else if (!ta)
    hipLaunchKernelGGL((gemm_small_kernel<T, false, true>), grid, threads, 0, s, p);
  else
    hipLaunchKernelGGL((gemm_small_kernel<T, true, true>), grid, threads, 0, s, p);
  return hipGetLastError();
}
template hipError_t launch_gemm_small<float>(const GemmParams<float>&, bool, bool, hipStream_t);
template hipError_t launch_gemm_small<double>(const GemmParams<double>&, bool, bool, hipStream_t);

}  // namespace eh
