// gemm_mfma.hpp -- kernel templates of the plain FP32 / FP64 MFMA products.
//
// One workgroup computes a BM x BN tile of C = alpha*op(A)*op(B) + beta*C
// over a K range (the whole K, or one split of it).  This is the device form
// of Eigen's GEBP (Eigen/src/Core/products/GeneralBlockPanelKernel.h):
//   * gemm_pack_lhs / gemm_pack_rhs (:1893-2478) become the global->LDS
//     staging of one BK-deep slice of op(A) and op(B), double buffered, with
//     every LDS row holding 128 contiguous bytes of k for one row of op(A) /
//     one column of op(B) (an XOR-swizzled, bank-conflict-free packed layout);
//   * the register-blocked micro-kernel (gebp_micro_panel_impl, :1352-1456)
//     becomes a WGM x WGN grid of waves (2x2, or 4x2 / 2x4 for two waves per
//     SIMD), each issuing RM x RN MFMA micro-tiles;
//   * the store `C += alpha*acc` (:1446-1455) becomes a fused alpha/beta
//     epilogue (beta == 0 never reads C, matching blas/level3_impl.h:82-87).
// Transposed operands only change which global index is contiguous; the LDS
// layout is the same for all four op combinations.
#pragma once
#include "common.hpp"
#include "kernels.hpp"

namespace eh {

// A triangular update (tri != 0) of a square result with square tiles
// launches only the tiles on or beside the triangle (tri_tile_coords);
// otherwise the full grid runs and tiles off the triangle return at once.
template <int BM, int BN, typename T>
__host__ __device__ inline bool tri_compact(const GemmParams<T>& p) {
  return p.tri != 0 && BM == BN && p.M == p.N;
}
template <int BM, int BN, typename T>
inline int64_t grid_tiles(const GemmParams<T>& p) {
  const int64_t ntm = (p.M + BM - 1) / BM, ntn = (p.N + BN - 1) / BN;
  return tri_compact<BM, BN>(p) ? ntm * (ntm + 1) / 2 : ntm * ntn;
}

// LDS bytes of one tile_product: two stages of (BM + BN) rows of 128 bytes.
template <int BM, int BN>
constexpr int tile_smem_bytes() {
  return 2 * (BM + BN) * 128;
}

// One BM x BN tile of op(A)*op(B) at (m0, n0) over k in [kbeg, kend): the body
// of a product workgroup.  At the end epi(acc) takes the wave's accumulators.
// smem holds tile_smem_bytes<BM, BN>(); the caller synchronises before reusing
// it.
// MODE: operand forms read in place of a repacked copy.
//   kComplexA      A holds interleaved (re, im) pairs (lda in pairs): each
//                  pair is staged as the 2x2 real block of alpha * op(A)
//                  (conjugated when p.conj), so M and K are twice op(A)'s.
//   kTriA, kTriB   op(A) (op(B)) is triangular, lower or upper by p.lower:
//                  elements off the triangle are staged as zeros whatever the
//                  memory holds, the diagonal as ones when p.unit.
// FOLD: every 128 of k the accumulators are added to a second set and start
// again from zero, so that a sum over one long run of k rounds no worse than
// one cut into splits or blocks (FP32 TRMM 1500 x 1100: relative error 2.1e-7
// against 3.6e-7 in one chain and 2.5e-7 over 256-row leaves).
template <typename T, int BM, int BN, int WGM, int WGN, bool TA, bool TB, int RS, int MODE, bool FOLD, typename Epi>
__device__ __forceinline__ void gemm_tile(GemmParams<T> p, int m0, int n0, int kbeg, int kend,
                                          unsigned char* __restrict__ smem, Epi epi) {
  using F = Mfma<T>;
  constexpr int NT = 64 * WGM * WGN;
  constexpr int ROWB = 128;                // bytes of k per LDS row
  constexpr int BK = ROWB / sizeof(T);     // 32 (f32) or 16 (f64)
  constexpr int EPC = 16 / sizeof(T);      // elements per 16-byte chunk
  constexpr int CH = ROWB / 16;            // chunks per row = 8
  constexpr int WTM = BM / WGM, WTN = BN / WGN;
  constexpr int RM = WTM / F::MI, RN = WTN / F::NI;
  constexpr int KPL = BK / F::KG;          // k values one lane feeds per slice
  constexpr int CPL = KPL / EPC;           // chunks one lane reads per row
  // chunks a thread loads per slice (a complex chunk makes two LDS chunks)
  constexpr int A_CH = BM * CH / NT / (MODE == kComplexA ? 2 : 1), B_CH = BN * CH / NT;
  constexpr int AR = MODE == kComplexA ? BM / 2 : BM;  // rows of op(A) in the tile
  static_assert(RM >= 1 && RN >= 1, "wave tile smaller than one MFMA block");
  static_assert(BM * CH % NT == 0 && BN * CH % NT == 0, "tile not divisible by threads");
  static_assert(CPL * EPC == KPL, "lane k range must be whole chunks");
  static_assert(RS == 1 || RS == 2, "one or two register stages");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int wm = wid % WGM, wn = wid / WGM;
  const int nkt = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;

  constexpr uint32_t SZ = sizeof(T);
  // A rows-contiguous operand (k is its column index) gets a buffer range
  // that ends at column kend, so every element with k >= kend reads zero;
  // k-contiguous operands are masked in registers instead.
  const uint32_t bytesA = TA ? p.bytesA : (uint32_t)min((uint64_t)p.bytesA, (uint64_t)kend * p.lda * SZ);
  const uint32_t bytesB = !TB ? p.bytesB : (uint32_t)min((uint64_t)p.bytesB, (uint64_t)kend * p.ldb * SZ);
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(p.A, bytesA);
  const __amdgpu_buffer_rsrc_t rB = make_rsrc(p.B, bytesB);

  // Loop-invariant per-lane byte offsets of every staged chunk; the k advance
  // goes into the wave-uniform soffset.  Rows / columns past M / N read zeros
  // or in-range values that only reach outputs that are never stored.
  uint32_t voA[A_CH], voB[B_CH];
#pragma unroll
  for (int j = 0; j < A_CH; ++j) {
    const int q = tid + NT * j;
    if constexpr (TA) {  // op(A)(i,k) = A[k + i*lda]: k contiguous
      const int r = q / CH, c = q % CH;
      if constexpr (MODE == kComplexA)
        voA[j] = (uint32_t)(((uint64_t)(m0 / 2 + r) * p.lda * 2 + c * EPC) * SZ);
      else
        voA[j] = (uint32_t)(((uint64_t)(m0 + r) * p.lda + c * EPC) * SZ);
    } else {  // op(A)(i,k) = A[i + k*lda]: rows contiguous
      if constexpr (MODE == kComplexA)  // with the chunk's first k: a wave's lanes may hold two chunks
        voA[j] = (uint32_t)((m0 + 2 * (q % AR) + (uint64_t)(q / AR * EPC) * p.lda) * SZ);
      else
        voA[j] = (uint32_t)((m0 + q % AR) * SZ);
    }
  }
#pragma unroll
  for (int j = 0; j < B_CH; ++j) {
    const int q = tid + NT * j;
    if constexpr (!TB) {  // op(B)(k,j) = B[k + j*ldb]: k contiguous
      const int r = q / CH, c = q % CH;
      voB[j] = (uint32_t)(((uint64_t)(n0 + r) * p.ldb + c * EPC) * SZ);
    } else {  // op(B)(k,j) = B[j + k*ldb]
      voB[j] = (uint32_t)((n0 + q % BN) * SZ);
    }
  }

  // One BK slice of both operands in registers.  No load depends on data or
  // on the slice index, so the code between loads and their use has no
  // branches and each wait covers exactly the loads it needs.
  struct Stage {
    u32x4 a[A_CH], b[B_CH];
  };
  // k-contiguous chunk: one 16-byte load (buffer loads need 4-byte alignment
  // only); rows-contiguous chunk: EPC loads, one per k, coalesced across the
  // wave.
  auto load_mncont = [&](__amdgpu_buffer_rsrc_t rs, uint32_t vo, int k0, int cu, int64_t ld) -> u32x4 {
    T t[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e)
      t[e] = buf_load(rs, vo, (uint32_t)((uint64_t)(k0 + cu * EPC + e) * ld * SZ), (T*)nullptr);
    return *reinterpret_cast<u32x4*>(t);
  };
  // the same for complex pairs: the pair of one k (FP64) or of two (FP32)
  auto load_pairs = [&](uint32_t vo, int k0) -> u32x4 {
    const uint32_t so = (uint32_t)((uint64_t)k0 * p.lda * SZ);
    if constexpr (SZ == 8) {
      return buf_load16(rA, vo, so);
    } else {
      typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 lo = __builtin_amdgcn_raw_buffer_load_b64(rA, (int)vo, (int)so, 0);
      const u32x2 hi = __builtin_amdgcn_raw_buffer_load_b64(rA, (int)(vo + (uint32_t)p.lda * 8), (int)so, 0);
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };
  // slice s (clamped to the last one: a prefetch past the end re-reads it)
  auto load = [&](Stage& st, int s) {
    const int k0 = kbeg + min(s, nkt - 1) * BK;
#pragma unroll
    for (int j = 0; j < A_CH; ++j) {
      const int q = tid + NT * j;
      if constexpr (TA)
        st.a[j] = buf_load16(rA, voA[j], (uint32_t)k0 * SZ);
      else if constexpr (MODE == kComplexA)
        st.a[j] = load_pairs(voA[j], k0);
      else
        st.a[j] = load_mncont(rA, voA[j], k0, __builtin_amdgcn_readfirstlane(q / AR), p.lda);
    }
#pragma unroll
    for (int j = 0; j < B_CH; ++j) {
      const int q = tid + NT * j;
      if constexpr (!TB)
        st.b[j] = buf_load16(rB, voB[j], (uint32_t)k0 * SZ);
      else
        st.b[j] = load_mncont(rB, voB[j], k0, __builtin_amdgcn_readfirstlane(q / BN), p.ldb);
    }
  };
  // k-contiguous chunk c of the slice at k0: zero the elements at k >= kend
  // (selects, no branch; a no-op except on the last slice)
  auto mask_kcont = [&](u32x4& v, int k0, int c) {
    T* t = reinterpret_cast<T*>(&v);
#pragma unroll
    for (int e = 0; e < EPC; ++e) t[e] = (k0 + c * EPC + e < kend) ? t[e] : T(0);
  };
  // chunk of line i (row of op(A), column of op(B)) at k..: elements off the
  // triangle become zeros; keep k <= i or k >= i
  auto mask_tri = [&](u32x4& v, int i, int k, bool keep_below) {
    T* t = reinterpret_cast<T*>(&v);
#pragma unroll
    for (int e = 0; e < EPC; ++e) {
      const int d = keep_below ? i - k - e : k + e - i;
      t[e] = d < 0 ? T(0) : t[e];
      t[e] = (d == 0) & (p.unit != 0) ? T(1) : t[e];
    }
  };
  // ---- registers -> LDS buffer -------------------------------------------
  auto store = [&](Stage& st, int s, int buf) {
    const int k0 = kbeg + min(s, nkt - 1) * BK;
    unsigned char* As = smem + buf * (BM + BN) * ROWB;
    unsigned char* Bs = As + BM * ROWB;
#pragma unroll
    for (int j = 0; j < A_CH; ++j) {
      const int q = tid + NT * j;
      const int r = TA ? q / CH : q % AR, c = TA ? q % CH : q / AR;
      if constexpr (TA) mask_kcont(st.a[j], k0, c);
      if constexpr (MODE == kTriA) mask_tri(st.a[j], m0 + r, k0 + c * EPC, p.lower);
      if constexpr (MODE == kComplexA) {
        // alpha * op(A)(i, k) = (x, y): row 2i holds (x, -y), row 2i + 1 (y, x)
        const T* t = reinterpret_cast<const T*>(&st.a[j]);
        u32x4 lo, hi;
        T *rl = reinterpret_cast<T*>(&lo), *rh = reinterpret_cast<T*>(&hi);
#pragma unroll
        for (int e = 0; e < EPC; e += 2) {
          const T im = p.conj ? -t[e + 1] : t[e + 1];
          const T x = p.alpha * t[e] - p.alpha_im * im, y = p.alpha * im + p.alpha_im * t[e];
          rl[e] = x;
          rl[e + 1] = -y;
          rh[e] = y;
          rh[e + 1] = x;
        }
        *reinterpret_cast<u32x4*>(As + (2 * r) * ROWB + swz8(2 * r, c) * 16) = lo;
        *reinterpret_cast<u32x4*>(As + (2 * r + 1) * ROWB + swz8(2 * r + 1, c) * 16) = hi;
      } else {
        *reinterpret_cast<u32x4*>(As + r * ROWB + swz8(r, c) * 16) = st.a[j];
      }
    }
#pragma unroll
    for (int j = 0; j < B_CH; ++j) {
      const int q = tid + NT * j;
      const int r = TB ? q % BN : q / CH, c = TB ? q / BN : q % CH;
      if constexpr (!TB) mask_kcont(st.b[j], k0, c);
      if constexpr (MODE == kTriB) mask_tri(st.b[j], n0 + r, k0 + c * EPC, !p.lower);
      *reinterpret_cast<u32x4*>(Bs + r * ROWB + swz8(r, c) * 16) = st.b[j];
    }
  };

  typename F::acc_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int r = 0; r < F::ACC; ++r) acc[i][j][r] = T(0);

  const int li = lane % F::MI;  // row of the MFMA operand this lane feeds
  const int lg = lane / F::MI;  // k group of this lane

  // ---- MFMAs over the slice in LDS buffer `buf` ---------------------------
  auto compute = [&](int buf) {
    const unsigned char* As = smem + buf * (BM + BN) * ROWB;
    const unsigned char* Bs = As + BM * ROWB;
#pragma unroll
    for (int cc = 0; cc < CPL; ++cc) {
      const int c = lg * CPL + cc;
      T a[RM][EPC], b[RN][EPC];
#pragma unroll
      for (int i = 0; i < RM; ++i) {
        const int r = wm * WTM + i * F::MI + li;
        u32x4 v = *reinterpret_cast<const u32x4*>(As + r * ROWB + swz8(r, c) * 16);
        const T* t = reinterpret_cast<const T*>(&v);
#pragma unroll
        for (int e = 0; e < EPC; ++e) a[i][e] = t[e];
      }
#pragma unroll
      for (int j = 0; j < RN; ++j) {
        const int r = wn * WTN + j * F::NI + li;
        u32x4 v = *reinterpret_cast<const u32x4*>(Bs + r * ROWB + swz8(r, c) * 16);
        const T* t = reinterpret_cast<const T*>(&v);
#pragma unroll
        for (int e = 0; e < EPC; ++e) b[j][e] = t[e];
      }
#pragma unroll
      for (int e = 0; e < EPC; ++e)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j) F::mma(a[i][e], b[j][e], acc[i][j]);
    }
  };

  typename F::acc_t total[FOLD ? RM : 1][FOLD ? RN : 1] = {};
  auto fold = [&]() {
    if constexpr (FOLD) {
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = typename F::acc_t{};
        }
    }
  };
  constexpr int FS = 128 / BK;  // slices between folds

  if (nkt > 0) {
    if constexpr (RS == 2) {
      // Two register stages: the loads of slice s + 2 are issued while slice
      // s is multiplied, so every slice has two slices of MFMA time to arrive.
      Stage r0, r1;
      load(r0, 0);
      store(r0, 0, 0);
      load(r1, 1);
      load(r0, 2);
      __syncthreads();
      // at the top of each pair: LDS buffer 0 holds slice kt, r1 slice
      // kt + 1, r0 slice kt + 2
      int kt = 0;
      for (; kt + 2 <= nkt; kt += 2) {
        compute(0);
        store(r1, kt + 1, 1);
        __syncthreads();
        load(r1, kt + 3);
        compute(1);
        store(r0, kt + 2, 0);
        __syncthreads();
        load(r0, kt + 4);
        if (FOLD && kt % FS == FS - 2) fold();
      }
      if (kt < nkt) compute(0);  // odd slice count: the last slice is in buffer 0
    } else {
      Stage r0;
      load(r0, 0);
      store(r0, 0, 0);
      __syncthreads();
      for (int kt = 0; kt < nkt; ++kt) {
        load(r0, kt + 1);
        compute(kt & 1);
        store(r0, kt + 1, (kt + 1) & 1);
        __syncthreads();
      }
    }
  }

  if constexpr (FOLD) {
    static_assert(RS == 2, "folding runs in the two-stage loop");
    fold();
    epi(total, lane, wm, wn);
  } else {
    epi(acc, lane, wm, wn);
  }
}

// The store of a tile: C = alpha*acc + beta*C, or (partial) acc to split z of
// the partial buffer p.W.
template <typename T, int BM, int BN, int WGM, int WGN, typename Acc>
__device__ __forceinline__ void tile_store(const GemmParams<T>& p, T alpha, int m0, int n0, int z, bool partial,
                                           const Acc& acc, int lane, int wm, int wn) {
  using F = Mfma<T>;
  constexpr int WTM = BM / WGM, WTN = BN / WGN;
#pragma unroll
  for (int i = 0; i < WTM / F::MI; ++i)
#pragma unroll
    for (int j = 0; j < WTN / F::NI; ++j) {
      const int col = n0 + wn * WTN + j * F::NI + F::col(lane);
      if (col >= p.N) continue;
#pragma unroll
      for (int r = 0; r < F::ACC; ++r) {
        const int row = m0 + wm * WTM + i * F::MI + F::row(r, lane);
        if (row >= p.M || (p.tri == 1 && row < col) || (p.tri == 2 && row > col)) continue;
        if (partial) {
          p.W[(int64_t)z * p.M * p.N + row + (int64_t)col * p.M] = acc[i][j][r];
        } else {
          T* dst = p.C + row + (int64_t)col * p.ldc;
          T v = acc[i][j][r];
          *dst = (p.beta == T(0)) ? alpha * v : fma_t(alpha, v, p.beta * *dst);
        }
      }
    }
}

template <typename T, int BM, int BN, int WGM, int WGN, bool TA, bool TB, int RS>
__global__ void __launch_bounds__(64 * WGM * WGN) gemm_mfma_kernel(GemmParams<T> p) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[tile_smem_bytes<BM, BN>()];
  const int ntm = (p.M + BM - 1) / BM, ntn = (p.N + BN - 1) / BN;
  int tm, tn;
  if (tri_compact<BM, BN>(p)) {
    // the grid holds only the tiles that meet the triangle (lower: tn <= tm)
    int r, c;
    tri_tile_coords(xcd_remap(blockIdx.x, gridDim.x), ntm, 8, r, c);
    tm = p.tri == 1 ? r : c;
    tn = p.tri == 1 ? c : r;
  } else {
    tile_coords(xcd_remap(blockIdx.x, gridDim.x), ntm, ntn, 8, tm, tn);
  }
  const int m0 = tm * BM, n0 = tn * BN;
  // a tile with no element in the updated triangle has nothing to do
  if ((p.tri == 1 && m0 + BM <= n0) || (p.tri == 2 && n0 + BN <= m0)) return;
  const int z = blockIdx.y;
  const int kbeg = z * p.k_per_split;
  const int kend = min(p.K, kbeg + p.k_per_split);
  gemm_tile<T, BM, BN, WGM, WGN, TA, TB, RS, kPlain, false>(
      p, m0, n0, kbeg, kend, smem,
      [&](const auto& acc, int lane, int wm, int wn) {
        tile_store<T, BM, BN, WGM, WGN>(p, p.alpha, m0, n0, z, gridDim.y > 1, acc, lane, wm, wn);
      });
}

// ---------------------------------------------------------------------------
// Balanced product: the tiles' k slices, one tile's after another's, are one
// line of units, cut into gridDim.x equal runs (all resident at once), so
// neither a tile count that is no multiple of what the chip holds nor tiles
// of unequal depth (a triangular operand) leave anything idle.  Tiles are
// 64x64 with four waves, three workgroups per CU: 128x128 tiles, two per CU,
// lose more to the larger cut tiles than they gain (FP64 1000x777x1203 86
// against 50 us, 2048x700x3000 190 against 159, FP32 1645x1384x2732 132 against
// 123); so do wave groups that share a tile's k slices (58, 178 us for four).
//
// A tile that lies inside one run is stored at once.  Of a tile cut between
// runs every workgroup writes its part to a slot (the first segment of run g
// to slot 2g, its last to 2g + 1) and takes a ticket; whoever takes the last
// one adds the parts, in run order, so the result does not depend on who that
// is, and clears the ticket.  Nobody waits for anybody.
// Without tickets every workgroup takes one whole tile.
// ---------------------------------------------------------------------------
// The parts travel between workgroups on different XCDs, whose L2s are not
// coherent: their stores and loads carry the device scope bit (sc1), which
// writes and reads past the L2, so no cache has to be written back or
// invalidated (a __threadfence per wave did that: FP64 1000x777x1203 took 126
// us instead of 59).
__device__ inline void slot_store(__amdgpu_buffer_rsrc_t r, uint32_t off, u32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)off, 0, 16);
}
__device__ inline u32x4 slot_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 16);
}

// The line of units of a product, on the host and in the kernel: lines of
// `cols` tiles, all tiles of line r over the k slices [begin(r), begin(r) +
// slices(r)*bk).  A dense product is one line of all tiles; a triangular
// operand gives one line per tile row of op(A) (tile column of op(B)), each of
// its tiles lengthened by kTileCost units that stand for the tile's first loads
// and its store (FP32 TRMM 1500 x 1100: 80, 49, 55 us with 0, 4, 10; FP64 3000 x
// 2900: 700, 575, 596).
constexpr int kTileCost = 4;
template <typename T>
struct BalancedLine {
  int lines, cols, K, bt, bk, mode;
  bool from0;  // triangular: k from 0 up to the tile's end, or from the tile's start up to K
  __host__ __device__ BalancedLine(const GemmParams<T>& p, int m) : mode(m) {
    constexpr int b = kBalancedTile;
    const int ntm = (p.M + b - 1) / b, ntn = (p.N + b - 1) / b;
    lines = m == kTriA ? ntm : m == kTriB ? ntn : 1;
    cols = m == kTriA ? ntn : m == kTriB ? ntm : ntm * ntn;
    K = p.K;
    bt = b;
    bk = 128 / (int)sizeof(T);
    from0 = (m == kTriA) == (p.lower != 0);
  }
  __host__ __device__ int begin(int r) const { return mode < kTriA || from0 ? 0 : r * bt; }
  __host__ __device__ int end(int r) const { return mode < kTriA || !from0 || (r + 1) * bt > K ? K : (r + 1) * bt; }
  __host__ __device__ int slices(int r) const { return (end(r) - begin(r) + bk - 1) / bk; }
  __host__ __device__ int span(int r) const { return slices(r) + (mode < kTriA ? 0 : kTileCost); }
  __host__ __device__ int64_t units() const {
    int64_t u = 0;
    for (int r = 0; r < lines; ++r) u += (int64_t)cols * span(r);
    return u;
  }
};

template <typename T, bool TA, bool TB, int MODE>
__global__ void __launch_bounds__(256, 3) gemm_balanced_kernel(GemmParams<T> p, int64_t units, unsigned* tickets) {
  using F = Mfma<T>;
  constexpr int BM = kBalancedTile, BN = kBalancedTile;
  constexpr int RM = BM / 2 / F::MI, RN = BN / 2 / F::NI;
  constexpr int BK = 128 / sizeof(T);
  constexpr int NT = 256;
  constexpr int VPB = F::ACC * sizeof(T) / 16;  // 16-byte vectors of one lane per MFMA block
  constexpr int NB = RM * RN;
  constexpr int CB = NB * VPB > 8 ? 8 / VPB : NB;  // blocks a thread adds up at a time (32 registers of parts)
  constexpr int SLOT = BM * BN * sizeof(T);     // bytes of a slot
  __shared__ __attribute__((aligned(16))) unsigned char smem[tile_smem_bytes<BM, BN>()];
  __shared__ int flag;
  const BalancedLine<T> line(p, MODE);
  const int64_t G = gridDim.x;
  const int64_t g = xcd_remap(blockIdx.x, gridDim.x);
  int r = 0;         // line of the current tile
  int64_t base = 0;  // first unit of that line
  int span = line.span(0);
  int64_t u0, u1;
  if (tickets) {
    u0 = units * g / G;
    u1 = units * (g + 1) / G;
    while (u0 >= base + (int64_t)line.cols * span) {
      base += (int64_t)line.cols * span;
      span = line.span(++r);
    }
  } else {
    r = (int)(g / line.cols);
    span = line.span(r);
    u0 = (g % line.cols) * span;
    u1 = u0 + span;
  }
  auto slot_rsrc = [&](int64_t i) {
    return make_rsrc(reinterpret_cast<unsigned char*>(p.W) + i * SLOT, (uint32_t)SLOT);
  };
  for (int64_t u = u0, end; u < u1; u = end) {
    if (u == base + (int64_t)line.cols * span) {
      base = u;
      span = line.span(++r);
    }
    const int c = (int)((u - base) / span), S = line.slices(r);
    const int64_t first = base + (int64_t)c * span;
    end = min(u1, first + span);
    const int s0 = (int)(u - first), s1 = min((int)(end - first), S);
    if (s0 >= S) continue;
    int tm, tn;
    if constexpr (MODE == kTriA) {
      tm = r;
      tn = c;
    } else if constexpr (MODE == kTriB) {
      tm = c;
      tn = r;
    } else {
      tile_coords(c, (p.M + BM - 1) / BM, (p.N + BN - 1) / BN, 8, tm, tn);
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const int kb = line.begin(r);
    auto finish = [&](auto& acc, int lane, int wm, int wn) {
      bool store = true;
      if (s0 != 0 || s1 != S) {
        unsigned* ticket = tickets + (int64_t)r * line.cols + c;
        // runs g0..g1 meet this tile: run h owns unit x for h = floor(((x + 1)G - 1) / units)
        const int64_t g0 = ((first + 1) * G - 1) / units, g1 = ((first + S) * G - 1) / units;
        const unsigned others = (unsigned)(g1 - g0);
        const __amdgpu_buffer_rsrc_t mine = slot_rsrc(2 * g + (u == u0 ? 0 : 1));
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const u32x4* a = reinterpret_cast<const u32x4*>(&acc[b / RN][b % RN]);
#pragma unroll
          for (int v = 0; v < VPB; ++v) slot_store(mine, (uint32_t)(((b * VPB + v) * NT + threadIdx.x) * 16), a[v]);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wave's part has reached memory
        __syncthreads();
        if (threadIdx.x == 0) {
          flag = atomicAdd(ticket, 1u) == others;
          if (flag) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        store = flag;
        if (store) {
          // CB blocks at a time, two parts in flight
#pragma unroll
          for (int b0 = 0; b0 < NB; b0 += CB) {
            typename F::acc_t sum[CB] = {};
            for (int64_t h = g0; h <= g1; h += 2) {
              u32x4 w[2][CB * VPB];
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                const int64_t hh = h + i <= g1 ? h + i : g1;
                const __amdgpu_buffer_rsrc_t part = slot_rsrc(2 * hh + (units * hh / G >= first ? 0 : 1));
#pragma unroll
                for (int v = 0; v < CB * VPB; ++v)
                  w[i][v] = slot_load(part, (uint32_t)(((b0 * VPB + v) * NT + threadIdx.x) * 16));
              }
#pragma unroll
              for (int i = 0; i < 2; ++i) {
                if (h + i > g1) break;
#pragma unroll
                for (int b = 0; b < CB; ++b) sum[b] += *reinterpret_cast<const typename F::acc_t*>(&w[i][b * VPB]);
              }
            }
#pragma unroll
            for (int b = 0; b < CB; ++b) acc[(b0 + b) / RN][(b0 + b) % RN] = sum[b];
          }
        }
      }
      if (store) tile_store<T, BM, BN, 2, 2>(p, MODE == kComplexA ? T(1) : p.alpha, m0, n0, 0, false, acc, lane, wm, wn);
    };
    gemm_tile<T, BM, BN, 2, 2, TA, TB, 2, MODE, true>(p, m0, n0, kb + s0 * BK, min(line.end(r), kb + s1 * BK), smem,
                                                      finish);
    __syncthreads();  // smem and flag are free again
  }
}

// Deterministic split-K reduction: C = alpha * sum_z W[z] + beta*C.
template <typename T>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(GemmParams<T> p, int splits) {
  const int64_t total = (int64_t)p.M * p.N;
  for (int64_t idx = blockIdx.x * 256ll + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int row = (int)(idx % p.M);
    const int64_t col = idx / p.M;
    if ((p.tri == 1 && row < col) || (p.tri == 2 && row > col)) continue;
    T s = T(0);
    for (int z = 0; z < splits; ++z) s += p.W[(int64_t)z * total + idx];
    T* dst = p.C + row + col * p.ldc;
    *dst = (p.beta == T(0)) ? p.alpha * s : fma_t(p.alpha, s, p.beta * *dst);
  }
}

// C = beta*C on the triangle `tri` (as GemmParams::tri) of C (beta==0 writes
// zeros without reading C).  Used when alpha==0 or k==0: the product term
// vanishes and A, B are not read.
template <typename T>
__global__ void __launch_bounds__(256) scale_c_kernel(T* C, int M, int N, int64_t ldc, T beta, int tri) {
  const int64_t total = (int64_t)M * N;
  for (int64_t idx = blockIdx.x * 256ll + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int row = (int)(idx % M);
    const int64_t col = idx / M;
    if ((tri == 1 && row < col) || (tri == 2 && row > col)) continue;
    T* dst = C + row + col * ldc;
    *dst = (beta == T(0)) ? T(0) : beta * *dst;
  }
}

// Result with an inner stride: C(i,j) = C[i*incc + j*ldc] gets
// alpha*W(i,j) + beta*C(i,j) (W = the unscaled product, m x n contiguous), in
// the epilogue's arithmetic; W == nullptr means the product term vanishes
// (C = beta*C).  beta == 0 never reads C.
template <typename T>
__global__ void __launch_bounds__(256) strided_combine_kernel(const T* W, int M, int N, T* C, int64_t incc,
                                                              int64_t ldc, T alpha, T beta) {
  const int64_t total = (int64_t)M * N;
  for (int64_t idx = blockIdx.x * 256ll + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int row = (int)(idx % M);
    const int64_t col = idx / M;
    T* dst = C + row * incc + col * ldc;
    if (W) {
      const T v = W[idx];
      *dst = (beta == T(0)) ? alpha * v : fma_t(alpha, v, beta * *dst);
    } else {
      *dst = (beta == T(0)) ? T(0) : beta * *dst;
    }
  }
}

}  // namespace eh
