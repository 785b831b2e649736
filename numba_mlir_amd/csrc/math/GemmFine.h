// Matrix products of few or short block tiles (included by Gemm.hip).
//
// A 128 x 128 tile costs its prologue, its epilogue and, where it is one of a
// few, most of the GPU, however little of K or of the tile there is; slices of K
// on top of that write and read whole tiles of partial sums, and operands off
// the word grid are copied first.  Here a block has a tile of 16 to 48 rows and
// columns to itself and its waves share out K, so that a small result still
// fills the GPU in one launch that reads the operands where they lie.
//
// What bounds it: for a result of a few tiles the chunks of K that a wave loads
// one after the other (0.2 to 0.4 us each); for more, the operands' way into the
// registers: tiles this small read them again and again from L2 (float64 1000 x 1100 x
// 1200 445 MB in 54 us, 8.3 TB/s), and a load of four neighbours of K from each of 16
// rows takes the vector cache four times as long as one of whole lines.  (Through LDS,
// coalesced: float32 2048^3 a fifth faster, which the bf16 parts do in 105 us, but float64
// 1000 x 1100 x 1200 5 % and 822 x 641 x 1048 14 % slower, one block a CU.)  48 x 48 is
// the largest tile of float64 that leaves two waves a SIMD.
//
// Kernels before (copies, tiles or the strided kernel, folds) / now, us, medians of 40
// calls on row-major operands: float32 126 x 1 x 100 11.4 / 3.4, 435 x 73 x 175 17.6 / 3.8,
// 111 x 290 x 1694 135 / 7.4, 496 x 691 x 74 13.4 / 5.4, 83 x 3325 x 852 28.0 / 21.9; float64
// 75 x 72 x 528 44.5 / 6.1, 583 x 175 x 280 25.9 / 6.4, 2391 x 420 x 140 25.5 / 13.6, 822 x
// 641 x 1048 57.3 / 28.8, 4023 x 93 x 2646 70.5 / 45.4, 1000 x 1100 x 1200 71.3 / 56.2 (47
// TFLOP/s; 53.6 where only this product runs).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

// v_mfma_<f32|f64>_16x16x4: A[l % 16][l / 16], B[l / 16][l % 16] of lane l.
template <typename T> struct FineMma;
template <> struct FineMma<float> {
  typedef float Acc __attribute__((ext_vector_type(4)));
  __device__ static __forceinline__ Acc mma(float a, float b, Acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int r, int lane) { return 4 * (lane / 16) + r; }
};
template <> struct FineMma<double> {
  typedef double Acc __attribute__((ext_vector_type(4)));
  __device__ static __forceinline__ Acc mma(double a, double b, Acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static __forceinline__ int row(int r, int lane) { return 4 * r + lane / 16; }
};

// n neighbouring elements, read and written at any element's address.
template <typename T, int n> struct FineElems {
  T v[n];
};

// A wave's 16 R rows (of C's row or column index) of one operand by 16 of K,
// loaded straight into the registers the matrix instructions read: lane l holds
// rows origin + R (l % 16) + t, k = 4 (l / 16) + j.  Which four k an instruction
// multiplies is free as long as both operands agree, and so is which rows a
// register holds: an operand contiguous in k comes as four neighbours of one
// row, any other as R neighbours of one k.
template <typename T, int R, bool K_CONTIG> struct FineFetch {
  typedef FineElems<T, K_CONTIG ? 4 : R> Elems;
  static constexpr int LOADS = K_CONTIG ? R : 4;
  const T *p;
  int64_t ld;
  // (R = 1: rows beyond the extent are read from the last; else the rows lie
  // inside it.)
  __device__ __forceinline__ void init(const T *base, int64_t ld_, int origin, int extent,
                                       int lane) {
    ld = ld_;
    int x = origin + R * (lane % 16);
    if (R == 1 && x >= extent)
      x = extent - 1;
    p = K_CONTIG ? base + int64_t(x) * ld + 4 * (lane / 16)
                 : base + int64_t(4 * (lane / 16)) * ld + x;
  }
  __device__ __forceinline__ void fetch(Elems (&e)[LOADS], int k0) const {
    const T *at = K_CONTIG ? p + k0 : p + int64_t(k0) * ld;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      e[i] = *reinterpret_cast<const Elems *>(at + i * ld);
  }
  // What lies before element `from` of the chunk counts as zero.
  __device__ static __forceinline__ void mask(Elems (&e)[LOADS], int from, int lane) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
#pragma unroll
      for (int q = 0; q < (K_CONTIG ? 4 : R); ++q)
        if (4 * (lane / 16) + (K_CONTIG ? q : i) < from)
          e[i].v[q] = T(0);
  }
  __device__ static __forceinline__ void scale(Elems (&e)[LOADS], T by) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
#pragma unroll
      for (int q = 0; q < (K_CONTIG ? 4 : R); ++q)
        e[i].v[q] *= by;
  }
  __device__ static __forceinline__ T value(const Elems (&e)[LOADS], int t, int j) {
    return K_CONTIG ? e[t].v[j] : e[j].v[t];
  }
};

// C[M,N] = alpha A B + beta C with the meaning of A_KC and B_NC of dgemm_mfma
// (Gemm.hip); operands and C at any element's address, K >= 16.  A block
// computes 16 RM x 16 RN of C; its W waves take the chunks of 16 of K in turn
// and their sums meet in LDS, always in the same order.  A tile that would end
// outside C is moved inside (RM, RN > 1: M >= 16 RM, N >= 16 RN) and stores
// only what no other tile has; the end of K is the last 16 of it, without what
// the whole chunks had.
//
// part: slices of sliceK of K leave their sums, unscaled, in part[slice][M][ldw] for
// gemm_splitk_fold, or gemm_thin_fold if there are more than kFineFewSlices.
//
// The tiles of all slices, slice by slice, go to the XCDs in eight equal stretches
// (grid: tiles * slices to a multiple of 8): neighbours, which run side by side, share
// operands in an XCD's L2, and no XCD has more than an eighth.  (An eighth of the tiles with all
// their slices each: one tile keeps to one XCD, 32 x 32 x 10^6 float32 218 us instead of
// 68; six of 42 tiles in six slices are 36 blocks for 32 CUs, 193 x 265 x 47979
// float64 288 instead of 148.)
constexpr int kFineFewSlices = 8;
template <typename T, int RM, int RN, int W, int WAVES, bool A_KC, bool B_NC>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(WAVES))) void
gemm_fine(const T *__restrict__ A, const T *__restrict__ B, T *__restrict__ C, int M, int N,
          int K, int64_t lda, int64_t ldb, int64_t ldc, T alpha, T beta, int tiles, int tilesN,
          int slices, int sliceK, T *__restrict__ part, int64_t ldw) {
  typedef typename FineMma<T>::Acc Acc;
  typedef FineFetch<T, RM, A_KC> FetchA;
  typedef FineFetch<T, RN, !B_NC> FetchB;
  constexpr int CK = 16, RUN = sizeof(T) == 4 ? 4 : 10, BM = 16 * RM, BN = 16 * RN, REGS = RM * RN * 4;
  __shared__ T sums[W][REGS][64];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  int tile = int(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8), slice = 0;
  if (part) {
    slice = int(uint32_t(tile) / uint32_t(tiles));
    tile -= slice * tiles;
  }
  if (slice >= slices || tile >= tiles)
    return;
  const int bm = tile / tilesN * BM, bn = tile % tilesN * BN;
  const int m0 = RM > 1 && bm > M - BM ? M - BM : bm, n0 = RN > 1 && bn > N - BN ? N - BN : bn;
  if (part) {
    const int k0 = slice * sliceK;
    A += A_KC ? int64_t(k0) : int64_t(k0) * lda;
    B += B_NC ? int64_t(k0) * ldb : int64_t(k0);
    K = K - k0 < sliceK ? K - k0 : sliceK;
    C = part + int64_t(slice) * M * ldw;
    ldc = ldw;
    alpha = T(1);
    beta = T(0);
  }
  FetchA fa;
  FetchB fb;
  fa.init(A, lda, m0, M, lane);
  fb.init(B, ldb, n0, N, lane);
  typename FetchA::Elems a[2][FetchA::LOADS];
  typename FetchB::Elems b[2][FetchB::LOADS];
  auto load = [&](int s, int k0) {
    fa.fetch(a[s], k0);
    fb.fetch(b[s], k0);
  };
  // float32's A is multiplied by 2^46 and its sums by 2^-46, so that products
  // among the subnormal numbers are rounded once, with their sum.  A tile in which
  // that overflows (an element or a sum from 2^82) or that holds an infinity or a
  // NaN is computed again as it is.
  constexpr bool SCALED = sizeof(T) == 4;
  T scale = SCALED ? T(1ll << 46) : T(1);
  Acc acc[RM][RN];
  auto multiply = [&](int s) {
    if (SCALED)
      fa.scale(a[s], scale);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
          acc[i][j] = FineMma<T>::mma(fa.value(a[s], i, k), fb.value(b[s], j, k), acc[i][j]);
  };
  // The wave's sums so far, to LDS, after every RUN chunks: no sum in registers is
  // longer than those of the slices of K that the larger tiles take (2-norm of the
  // error, float32 1000 x 1100 x 1200 in seven slices 2.0e-7, here 3.1e-7 without and
  // 1.9e-7 with; float64 4.5e-16 / 4.3e-16).
  bool added = false;
  auto flush = [&]() {
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          T &sum = sums[wave][(i * RN + j) * 4 + r][lane];
          sum = added ? sum + acc[i][j][r] : acc[i][j][r];
          acc[i][j][r] = T(0);
        }
    added = true;
  };
  // One chunk ahead in registers.  (No branch between a load and its use: where
  // ways meet, the compiler waits for all loads in flight.)
  const int whole = K / CK, rest = K % CK, last = CK * (whole - 1);
  constexpr int PAIRS = (4 * RM + W - 1) / W;
  FineElems<T, RN> v[PAIRS]; // of the wave's (row tile, register) pairs
  for (;;) {
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
      for (int j = 0; j < RN; ++j)
        acc[i][j] = Acc{T(0), T(0), T(0), T(0)};
    int n = (whole + W - 1 - wave) / W, k = CK * wave;
    if (n > 0)
      load(0, k);
    if (rest && whole % W == wave) {
      load(1, K - CK);
      fa.mask(a[1], CK - rest, lane);
      fb.mask(b[1], CK - rest, lane);
      multiply(1);
    }
    while (n > 1) {
      int run = n < RUN ? n & ~1 : RUN;
      n -= run;
#pragma nounroll
      for (; run > 0; run -= 2) {
        load(1, k + CK * W);
        multiply(0);
        k += 2 * CK * W;
        load(0, k < last ? k : last);
        multiply(1);
      }
      if (n > 1)
        flush();
    }
    if (n > 0)
      multiply(0);
    flush();
    __syncthreads();
    bool finite = true;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const int p = W * i + wave;
      if (p >= 4 * RM)
        break;
#pragma unroll
      for (int j = 0; j < RN; ++j) {
        const int at = (p / 4 * RN + j) * 4 + p % 4;
        T sum = sums[0][at][lane];
#pragma unroll
        for (int w = 1; w < W; ++w)
          sum += sums[w][at][lane];
        if (SCALED) {
          finite = finite && sum - sum == T(0);
          sum *= T(1) / scale;
        }
        v[i].v[j] = alpha * sum;
      }
    }
    if (!SCALED || scale == T(1) || !__syncthreads_or(!finite))
      break;
    scale = T(1);
    added = false;
  }
#pragma unroll
  for (int i = 0; i < PAIRS; ++i) {
    const int p = W * i + wave, t = p / 4, r = p % 4;
    if (p >= 4 * RM)
      break;
    const int m = m0 + RM * FineMma<T>::row(r, lane) + t, col = n0 + RN * (lane % 16);
    if (m < bm || m >= M)
      continue;
    T *dst = C + int64_t(m) * ldc + col;
    if (beta == T(0) && col >= bn && col + RN <= N) {
      *reinterpret_cast<FineElems<T, RN> *>(dst) = v[i];
      continue;
    }
#pragma unroll
    for (int j = 0; j < RN; ++j) {
      if (col + j < bn || col + j >= N)
        continue;
      if (beta != T(0))
        v[i].v[j] += beta * dst[j];
      dst[j] = v[i].v[j];
    }
  }
}

} // namespace
