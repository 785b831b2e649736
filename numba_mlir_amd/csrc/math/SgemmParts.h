// float32 matrix products on the bf16 matrix cores (included by Gemm.hip).
//
// gfx950 multiplies bf16 sixteen times as fast as float32 (2.5 PFLOP/s against
// 157 TFLOP/s), and a float32 is three bf16 without a bit lost: x = h + m + l,
// h = bf16(x), m = bf16(x - h), l = x - h - m, both differences exact (8 + 8 +
// 8 significant bits, the sign of m and l taking the place of the bit that
// rounding gave away; bf16 has float32's exponents).  A product of two floats
// is then the sum of nine exact bf16 products, of which
//   h l' + l h' + m m' + m h' + h m' + h h'
// are computed, smallest first, and the other three left out: together they
// are below 2^-24 |x y|, less than the rounding of one float32 product.  An
// instruction adds its sixteen products to a float32 accumulator in two groups
// of eight (measured, element by element): within a group what lies below 2^-24
// of the largest term is cut off, downwards, then the sum is rounded to nearest:
// 12 roundings for 16 terms of K, where the float32 instructions round each of
// the 16.  The cut leans every sum the same way: accumulators and A's parts
// change sign after 64 slabs and then every 128, and from one slice or piece of
// K to the next, so that what one leaned another takes back.
//
// 2-norm of the error against float64 over 2-norm of the result, float32
// instructions / this, centred data: K = 3 3.6e-8 / 3.3e-8, 16 7.4e-8 / 3.4e-8, 512
// 2.1e-7 / 1.7e-7, 4096 1.15e-6 / 0.98e-6, 16384 2.29e-6 / 1.88e-6, 262144 (in
// slices) 2.29e-6 / 1.89e-6 (without the changes of sign 2.08e-6 at 16384,
// 3.71e-6 at 262144); data in [0, 1): 4096 8.4e-7 / 5.2e-7, 16384 1.68e-6 /
// 1.03e-6, 262144 4.3e-7 / 2.6e-7 (4.5e-7).  A sum of which one or two products
// are not zero (a diagonal matrix times another) is not the nearest float32 as
// the float32 instructions' is, but within 1.7e-7 of itself.
//
// Which operands this holds for: every part must be a bf16 number and every
// sum a float32.  Operands are multiplied by 2^23 on their way to LDS, and sums
// by 2^-46 on their way out: the last bit of any float32, 2^-149 at least, then
// lies in bf16's normal range, so values of any smallness have parts.  An
// infinity, a NaN, an operand of 2^105 or a sum of 2^82 and more leaves a NaN
// or an infinity in the accumulators.  They are looked at after 4, 64 and every
// 128 slabs and at the end; the 32 x 32 tiles that hold one are computed again with
// the float32 instructions, whose results such inputs then have as before (at
// once, if they are most of a wave's).  us at 4096^3, float32 instructions
// alone / values of 2^-100 and less and all infinities computed again in whole
// 256 x 256 tiles / this: exp(-x) for x in [0, 100) 970 / 1284 / 613, an infinity
// in the last column of every 128th row 969 / 1715 / 1029, every sum too large
// 969 / 1281 / 1144 (ordinary data 972 / 617 / 613); at 1024^3 44.3 / 67.0 / 38.6,
// 44.4 / 63.0 / 47.9, 44.4 / 63.0 / 54.7.
//
// Time: six bf16 products take 6/16 of the float32 instructions' time.  At
// 4096^3 the 256 x 256 tile takes 577 to 640 us by box and temperature (238 to
// 215 TFLOP/s of float32 product) against 966 us; the matrix cores are busy 71
// to 76 % of the cycles at 1.77 GHz, the clock the power limit leaves (a loop of
// nothing but these instructions: 96 % at 1.86 GHz).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t uintx2 __attribute__((ext_vector_type(2)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

constexpr float kPartsScale = 8388608.0f; // 2^23

// The parts of two values, each pair packed into a register (nearest-even
// conversions; the differences are exact).
__device__ __forceinline__ void partsOf(float x, float y, uint32_t &h, uint32_t &m,
                                        uint32_t &l) {
  auto pack = [](float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{a, b}, bf16x2));
  };
  h = pack(x, y);
  x -= __builtin_bit_cast(float, h << 16);
  y -= __builtin_bit_cast(float, h & 0xffff0000u);
  m = pack(x, y);
  x -= __builtin_bit_cast(float, m << 16);
  y -= __builtin_bit_cast(float, m & 0xffff0000u);
  l = pack(x, y);
}

// One operand's slab of X rows (of C's row or column index) by 16 of K on its
// way to LDS.  A thread holds quads, four neighbours along k of one row:
// NQ = 2 of them (or 1, on twice the threads).
//   K_CONTIG: a 128-bit load a quad, rows X / NQ apart
//   else    : four loads of NQ neighbouring rows, one for each k
// Rows beyond the operand's extent are read from its last row (or pair): what
// they add to lies outside C.  K need not be whole slabs: what fetchTail does
// not find counts as zero.  A quad, and a pair of rows, must lie inside the
// operand's rows in memory: extents along the contiguous dimension are
// multiples of four, or the rows are padded to that.
template <int X, bool K_CONTIG, int THREADS> struct PartsFetch {
  static constexpr int NQ = X * 4 / THREADS;
  static_assert(NQ == 1 || NQ == 2, "one or two quads a thread");
  typedef float Rows __attribute__((ext_vector_type(NQ)));
  const float *p;
  int64_t ld, step;
  int row, quad; // K_CONTIG: the second quad's row is row + X / 2, else row + 1
  floatx4 q4[NQ];
  Rows rows[4];

  // Sixteen lanes cover four quads of four rows two apart (or of four pairs of
  // rows): the 64-bit words they write to LDS then fall on 32 different banks.
  __device__ __forceinline__ void init(const float *base, int64_t ld_, int origin, int extent,
                                       int k0, int tid) {
    ld = ld_;
    quad = K_CONTIG ? tid % 4 : tid / 4 % 4;
    const int last = extent - origin - 1; // the last row that there is
    if (K_CONTIG) {
      const int r = tid / 4 % 16;
      row = 16 * (tid / 64) + 2 * (r % 4) + (r / 4) % 2 + 8 * (r / 8);
      const int r0 = row < last ? row : last;
      p = base + int64_t(origin + r0) * ld + k0 + 4 * quad;
      const int r1 = row + X / 2 < last ? row + X / 2 : last;
      step = int64_t(r1 - r0) * ld;
    } else {
      row = NQ * (tid % 4 + 4 * (tid / 16));
      const int r0 = row < last ? row : last / NQ * NQ;
      p = base + int64_t(k0 + 4 * quad) * ld + origin + r0;
      step = 0;
    }
  }
  __device__ __forceinline__ int rowOf(int i) const {
    return K_CONTIG ? row + i * (X / 2) : row + i;
  }
  __device__ __forceinline__ float at(int i, int q) const {
    return K_CONTIG ? q4[i][q] : rows[q][i];
  }
  // The next slab, whole.
  __device__ __forceinline__ void fetch() {
    if (K_CONTIG) {
#pragma unroll
      for (int i = 0; i < NQ; ++i)
        q4[i] = *reinterpret_cast<const floatx4 *>(i ? p + step : p);
      p += 16;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        rows[q] = *reinterpret_cast<const Rows *>(p + q * ld);
      p += 16 * ld;
    }
  }
  // The next slab, of which `left` of K are left (1 to 15): the last one.
  __device__ __forceinline__ void fetchTail(int left) {
    if (K_CONTIG) {
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        q4[i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        if (4 * quad < left)
          q4[i] = *reinterpret_cast<const floatx4 *>(i ? p + step : p);
      }
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int i = 0; i < NQ; ++i)
          rows[q][i] = 0.0f;
        if (4 * quad + q < left)
          rows[q] = *reinterpret_cast<const Rows *>(p + q * ld);
      }
    }
  }
};

// Both operands' next slab, of which `left` of K are left: one branch for the
// two (where the ways of loading a whole and a cut slab meet, the second
// operand's loads waited for the first's).
template <typename FetchA, typename FetchB>
__device__ __forceinline__ void fetchBoth(FetchA &fa, FetchB &fb, int left) {
  if (left >= 16) {
    fa.fetch();
    fb.fetch();
  } else {
    fa.fetchTail(left);
    fb.fetchTail(left);
  }
}

// An operand's slab in LDS, in words of 16 bytes: three planes (h, m, l) of two
// halves of K of X rows of eight bf16.  One word of padding a half: the halves
// start 16 bytes apart among the banks.
template <int X> struct PartsSlab {
  static constexpr int HALF = X + 1, PLANE = 2 * HALF, WORDS = 3 * PLANE;
};

template <int X, bool KC, int THREADS>
__device__ __forceinline__ void stashParts(const PartsFetch<X, KC, THREADS> &f, uintx4 *lds,
                                           float scale) {
#pragma unroll
  for (int i = 0; i < f.NQ; ++i) {
    uint32_t h0, h1, m0, m1, l0, l1;
    partsOf(scale * f.at(i, 0), scale * f.at(i, 1), h0, m0, l0);
    partsOf(scale * f.at(i, 2), scale * f.at(i, 3), h1, m1, l1);
    uintx2 *at = reinterpret_cast<uintx2 *>(lds) +
                 2 * (f.quad / 2 * PartsSlab<X>::HALF + f.rowOf(i)) + f.quad % 2;
    at[0] = uintx2{h0, h1};
    at[2 * PartsSlab<X>::PLANE] = uintx2{m0, m1};
    at[4 * PartsSlab<X>::PLANE] = uintx2{l0, l1};
  }
}

// The operands as they are, for the float32 instructions: [half of K][row][two
// words] in the same memory.
template <int X, bool KC, int THREADS>
__device__ __forceinline__ void stashFloats(const PartsFetch<X, KC, THREADS> &f, uintx4 *lds) {
#pragma unroll
  for (int i = 0; i < f.NQ; ++i)
    reinterpret_cast<floatx4 *>(
        lds)[2 * (f.quad / 2 * PartsSlab<X>::HALF + f.rowOf(i)) + f.quad % 2] =
        floatx4{f.at(i, 0), f.at(i, 1), f.at(i, 2), f.at(i, 3)};
}

// C[M,N] = alpha A B + beta C with the meaning of A_KC, B_NC, sliceK, W, ldw
// and even of dgemm_mfma (Gemm.hip), K in slabs of 16.  WM x WN waves share a
// tile of BM x BN.  M, N and K may end anywhere (see PartsFetch).
//
// Two LDS stages: while slab s is multiplied, slab s + 1 goes from registers,
// split into its parts, to the other stage, and slab s + 2 is loaded into those
// registers; one barrier a slab.  256 x 256: eight waves of 128 x 64, two a
// SIMD (three 128-bit LDS reads for eight matrix instructions, and seven
// vector instructions of splitting for three; four waves of 128 x 128 would
// leave each SIMD one wave, whose waits nothing fills).  128 x 128: four
// waves of 64 x 64.
template <int BM, int BN, int WM, int WN, bool A_KC, bool B_NC>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(2, 2))) void
sgemm_parts(const float *__restrict__ A, const float *__restrict__ B, float *__restrict__ C,
            int M, int N, int K, int64_t lda, int64_t ldb, int64_t ldc, float alpha, float beta,
            int sliceK, float *__restrict__ W, int64_t ldw, EvenShares even) {
  constexpr int THREADS = 64 * WM * WN, BK = 16;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  __shared__ uintx4 As[2][PartsSlab<BM>::WORDS];
  __shared__ uintx4 Bs[2][PartsSlab<BN>::WORDS];
  if (sliceK > 0) {
    const int k0 = blockIdx.z * sliceK;
    A += A_KC ? int64_t(k0) : int64_t(k0) * lda;
    B += B_NC ? int64_t(k0) * ldb : int64_t(k0);
    K = K - k0 < sliceK ? K - k0 : sliceK;
    C = W + int64_t(blockIdx.z) * int64_t(M) * ldw;
    ldc = ldw;
    alpha = 1.0f;
    beta = 0.0f;
  }
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / WN, wn = wave % WN;
  // The word of its tile's first row that a lane reads as matrix operand: row
  // lane % 32, half lane / 32 of K.
  const int aWord = wm * (TM * 32) + lane % 32 + lane / 32 * PartsSlab<BM>::HALF;
  const int bWord = wn * (TN * 32) + lane % 32 + lane / 32 * PartsSlab<BN>::HALF;

  int64_t unit = 0, unitEnd = 0, wholeTile = blockIdx.x;
  const int slabsPerTile = even.slabs > 0 ? even.slabs : (K + BK - 1) / BK;
  if (even.slabs > 0) {
    const int64_t units =
        (int64_t((M + BM - 1) / BM) * even.tilesN - even.whole) * even.slabs;
    unit = evenSharesStart(blockIdx.x, units, gridDim.x);
    unitEnd = evenSharesStart(int64_t(blockIdx.x) + 1, units, gridDim.x);
  } else {
    unitEnd = slabsPerTile;
  }
#pragma nounroll
  for (int segment = 0; unit < unitEnd; ) {
    int bm = blockIdx.y * BM, bn = blockIdx.x * BN;
    int slab0 = 0, slab1 = slabsPerTile; // the K slabs of this segment
    const bool shared = wholeTile >= even.whole; // (else a tile before the shares)
    if (even.slabs > 0) {
      int64_t tile = wholeTile;
      if (shared) {
        tile = unit / even.slabs;
        slab0 = int(unit - tile * even.slabs);
        slab1 = unitEnd - unit < even.slabs - slab0 ? slab0 + int(unitEnd - unit) : even.slabs;
        tile += even.whole;
      }
      bm = int(tile / even.tilesN) * BM;
      bn = int(tile % even.tilesN) * BN;
      __syncthreads(); // every wave is done with the last segment's LDS slabs
    }
    const bool piece = even.slabs > 0 && !(slab0 == 0 && slab1 == even.slabs);
    const int slot = segment > 0 ? 1 : 0;
    if (shared) {
      unit += slab1 - slab0;
      ++segment;
    }
    wholeTile += gridDim.x;

    PartsFetch<BM, A_KC, THREADS> fa;
    PartsFetch<BN, !B_NC, THREADS> fb;
    fa.init(A, lda, bm, M, slab0 * BK, tid);
    fb.init(B, ldb, bn, N, slab0 * BK, tid);
    floatx16 acc[TM][TN];
    auto clear = [&] {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[i][j][r] = 0.0f;
    };
    clear();

    // One or two products lose more to the missing parts than their sum's few
    // roundings give back (2-norm of the error, K = 1: 2.5e-8 in float32, every
    // product rounded to nearest, 3.5e-8 in parts; K = 2: 3.1e-8, 3.4e-8; K = 3:
    // 3.6e-8, 3.3e-8): they stay with the float32 instructions (and with the
    // small tile: the large one's shapes begin at K = 16).
    bool early = BM == 128 && K <= 2; // the parts are given up before the end of K
    // A's scale, and its sign the accumulators': it changes from slice to slice
    // and from piece to piece of a tile, and along a longer K.
    // (The bits of it, so that it stays in a scalar register.)
    uint32_t turned = ((sliceK > 0 ? blockIdx.z : piece ? blockIdx.x : 0) & 1) << 31;
    auto left = [&] {
      return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, kPartsScale) ^ turned);
    };
    if (!early) {
      fetchBoth(fa, fb, K - slab0 * BK);
      stashParts(fa, As[0], left());
      stashParts(fb, Bs[0], kPartsScale);
      if (slab0 + 1 < slab1)
        fetchBoth(fa, fb, K - (slab0 + 1) * BK);
      __syncthreads();
    }

    // FETCH: 0 nothing is left to load, 1 a whole slab, 2 the last slab.
    auto slab = [&](int s, auto stash, auto fetch) {
      constexpr bool STASH = decltype(stash)::value != 0;
      constexpr int FETCH = decltype(fetch)::value;
      const int cur = (s - slab0) & 1;
      bf16x8 a[TM][3], b[TN][3];
      auto rowsOf = [&](int i) {
#pragma unroll
        for (int p = 0; p < 3; ++p)
          a[i][p] = __builtin_bit_cast(bf16x8, As[cur][p * PartsSlab<BM>::PLANE + aWord + i * 32]);
      };
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int p = 0; p < 3; ++p)
          b[j][p] = __builtin_bit_cast(bf16x8, Bs[cur][p * PartsSlab<BN>::PLANE + bWord + j * 32]);
      rowsOf(0);
      rowsOf(1);
      if (STASH) {
        stashParts(fa, As[cur ^ 1], left());
        stashParts(fb, Bs[cur ^ 1], kPartsScale);
      }
      if (FETCH == 1) {
        fa.fetch();
        fb.fetch();
      } else if (FETCH == 2) {
        fetchBoth(fa, fb, K - (s + 2) * BK);
      }
      constexpr int LEFT[6] = {2, 0, 1, 1, 0, 0}, RIGHT[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int t = 0; t < 6; ++t)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][LEFT[t]], b[j][RIGHT[t]],
                                                                acc[i][j], 0, 0, 0);
        if (i + 2 < TM)
          rowsOf(i + 2);
      }
      if (STASH)
        __syncthreads();
    };
    typedef std::integral_constant<int, 0> No;
    typedef std::integral_constant<int, 1> Yes;
    typedef std::integral_constant<int, 2> Last;
    // The wave's 32 x 32 tiles, one bit each, that hold an infinity or a NaN.
    auto tilesLost = [&] {
      uint32_t lost = 0;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float finite = 0.0f;
#pragma unroll
          for (int r = 0; r < 16; ++r)
            finite = __builtin_fmaf(acc[i][j][r], 0.0f, finite);
          if (__builtin_amdgcn_ballot_w64(finite != finite))
            lost |= 1u << (i * TN + j);
        }
      return lost;
    };
    uint32_t lost = 0;
    int s = slab0;
    // (A look costs 0.7 us on the large tile, as a third of a slab.  Where the end
    // is 24 slabs away or nearer there is none: 1000 x 1100 x 1200, of 11 slabs a
    // slice, 48.1 us with one, 47.4 without; of all sums too large 55 / 57.)
    for (int look = slab1 - slab0 > 24 ? 4 : 24; s + 3 < slab1 && !early;
         look = look == 4 ? 60 : 128) {
      const int stop = s + look < slab1 - 3 ? s + look : slab1 - 3;
      const bool more = stop < slab1 - 3, turn = more && look > 4;
      for (; s < (turn ? stop - 1 : stop); ++s)
        slab(s, Yes(), Yes());
      if (turn) {
        turned ^= 1u << 31; // of slab `stop`, which is split now
        slab(s++, Yes(), Yes());
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              acc[i][j][r] = -acc[i][j][r];
      }
      if (more)
        early = __syncthreads_or(2 * __builtin_popcount(tilesLost()) > TM * TN);
    }
    if (early) {
      lost = (1u << (TM * TN)) - 1;
    } else {
      if (s + 2 < slab1)
        slab(s++, Yes(), Last());
      if (s + 1 < slab1)
        slab(s++, Yes(), No());
      slab(s, No(), No());
      lost = tilesLost();
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const float unscale = 1.0f / (left() * kPartsScale);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[i][j][r] = lost >> (i * TN + j) & 1
                             ? 0.0f
                             : __builtin_fmaf(acc[i][j][r], unscale, 0.0f); // (no -0)
      }
    if (__syncthreads_or(lost != 0)) {
      // The lost tiles with v_mfma_f32_32x32x2_f32: lane half h of the wave
      // takes k = 8 h + t of the slab in step t.  Two LDS stages, the next
      // slab loaded while one is multiplied, one barrier a slab.
      fa.init(A, lda, bm, M, slab0 * BK, tid);
      fb.init(B, ldb, bn, N, slab0 * BK, tid);
      fetchBoth(fa, fb, K - slab0 * BK);
#pragma nounroll
      for (s = slab0; s < slab1; ++s) {
        const int cur = (s - slab0) & 1;
        stashFloats(fa, As[cur]);
        stashFloats(fb, Bs[cur]);
        __syncthreads(); // (also: every wave has read the slab before the last)
        if (s + 1 < slab1)
          fetchBoth(fa, fb, K - (s + 1) * BK);
        floatx4 a[TM][2], b[TN][2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            b[j][w] = reinterpret_cast<const floatx4 *>(Bs[cur])[2 * (bWord + j * 32) + w];
#pragma unroll
          for (int i = 0; i < TM; ++i)
            a[i][w] = reinterpret_cast<const floatx4 *>(As[cur])[2 * (aWord + i * 32) + w];
        }
        auto multiply = [&](int i, int j, int t) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][t / 4][t % 4], b[j][t / 4][t % 4],
                                                           acc[i][j], 0, 0, 0);
        };
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if (!(lost >> (i * TN + j) & 1))
              continue;
            multiply(i, j, 0);
            multiply(i, j, 1);
            if (BM == 128 && K <= 2)
              continue; // (the other steps multiply zeros: 1 us)
#pragma unroll
            for (int t = 2; t < 8; ++t)
              multiply(i, j, t);
          }
      }
    }

    // A whole tile goes to C, scaled; a piece of one goes to its workspace
    // slot as a dense BM x BN block, unscaled.
    // (The lane's number as if it were new, so that the places in C are worked
    // out here: the compiler would keep them in scratch over the whole of K.)
    int home = lane;
    asm volatile("" : "+v"(home));
    float *out = C + int64_t(bm) * ldc + bn;
    int64_t ldo = ldc;
    float scale = alpha, keep = beta;
    int rowsLeft = M - bm, colsLeft = N - bn;
    if (piece) {
      out = W + (int64_t(blockIdx.x) * 2 + slot) * (BM * BN);
      ldo = BN;
      scale = 1.0f;
      keep = 0.0f;
      rowsLeft = BM;
      colsLeft = BN;
    }
    // (bare stores where nothing is cut off or added: the guarded ones are five
    // times the instructions, which a product of a slab or two waits for: 1024 x
    // 1024 x 16 21.9 -> 20.0 us, 640 x 640 x 64 23.8 -> 22.0.  The large tile's
    // products hide them, and it has no registers for both.)
    const bool bare = BM == 128 && keep == 0.0f && rowsLeft >= BM && colsLeft >= BN;
    if (bare) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            out[int64_t(wm * (TM * 32) + i * 32 + Mfma<float>::accRow(r, home)) * ldo +
                wn * (TN * 32) + j * 32 + home % 32] = scale * acc[i][j][r];
    }
#pragma unroll
    for (int i = 0; i < TM && !bare; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int col = wn * (TN * 32) + j * 32 + home % 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = wm * (TM * 32) + i * 32 + Mfma<float>::accRow(r, home);
          if (!(row < rowsLeft && col < colsLeft))
            continue;
          float *dst = out + int64_t(row) * ldo + col;
          float v = scale * acc[i][j][r];
          if (keep != 0.0f)
            v += keep * *dst;
          *dst = v;
        }
      }
    }
  } // segments
}

} // namespace
