// float32 products whose operands are split into their bf16 parts once, ahead of
// the product (included by Gemm.hip after SgemmParts.h, whose arithmetic this is:
// six products of parts, scales, tiles computed again on the float32
// instructions).
//
// sgemm_parts splits an operand again beside every tile that reads it, and its
// 128 x 128 tile then has matrix cores and vector units busy half the time each
// (2047 x 2049 x 2051: 48 and 41 % of the cycles); operands off the word grid are
// copied first as well.  Here that copy is the split: 10 bytes of memory an
// element instead of 8, laid out as the matrix instructions read it, so that the
// product kernel moves it to LDS without passing a register and multiplies, 894
// cycles a slab of 16 of a tile where its matrix instructions take 768.  What
// bounds it then is the power limit: a slab takes 0.53 us with all CUs at it, 0.37 with
// four, 1.7 and 2.4 GHz.
//
// Kernels of a call, us, copies + tiles + fold before / split + tiles + fold now:
// 2047 x 2049 x 2051 13.9 + 105.4 + 14.3 / 19.6 + 95.4 + 9.2; calls 877 x 4531 x 1863 130 /
// 114, 4026 x 1410 x 3158 270 / 237, 5657 x 2051 x 481 130 / 98.  On the way: one
// wave a SIMD with its loads and LDS reads ahead of the matrix instructions instead
// of between them 1217 cycles a slab; two blocks a CU 567 us at 4096^3 and twice the
// pieces to add up; tiles of 256 x 128 545 us at 4096^3 against 576, but twice as
// long in a round that they do not fill, and no registers for a second sum.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

// One operand's parts: for every 32 rows (of C's row or column index) and slab of
// 16 of K, the three planes h, m, l as the 64 lanes of v_mfma_f32_32x32x16_bf16
// hold them (row lane % 32, k 8 (lane / 32) + j).  PLANE_WORDS words of 16 bytes
// a plane.
constexpr int kPlaneWords = 64, kPlanesWords = 3 * kPlaneWords;

// Element (r, k) of the operand is src[r * rowStride + k * kStride]; one of the
// strides is one.  rowTiles x slabs tiles are written, zero beyond R and K; run:
// slabs of every second run of so many have their sign changed (0: none).
//
// A tile of 32 rows and a slab that holds an infinity, a NaN or an element too large
// for parts is left out (its parts are zero) and flagged, a byte each in
// flags[rowTile / 4][slab][rowTile % 4]: the product kernel adds what it is part of
// from the operands themselves.
struct PlanesJob {
  const float *src;
  int64_t rowStride, kStride;
  int R, K, rowTiles, slabs, run;
  uintx4 *dst;
  unsigned char *flags;
  __host__ __device__ int64_t blocks() const { return int64_t(rowTiles) * ((slabs + 3) / 4); }
};

__global__ __launch_bounds__(256) void sgemm_split_planes(PlanesJob first, PlanesJob second) {
  const int64_t ahead = first.blocks();
  const bool two = blockIdx.x >= ahead;
  const PlanesJob job = two ? second : first;
  const uint32_t block = uint32_t(two ? blockIdx.x - ahead : blockIdx.x);
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const uint32_t groups = uint32_t(job.slabs + 3) / 4;
  const bool kContig = job.kStride == 1;
  // (neighbouring blocks read what lies side by side)
  const int tile = int(kContig ? block / groups : block % uint32_t(job.rowTiles));
  const int slab = 4 * int(kContig ? block % groups : block / uint32_t(job.rowTiles)) + wave;
  if (slab >= job.slabs)
    return;
  const int r = 32 * tile + lane % 32, k = 16 * slab + 8 * (lane / 32);
  const float scale = job.run && slab / job.run % 2 ? -kPartsScale : kPartsScale;
  float v[8];
  const float *at = job.src + int64_t(r) * job.rowStride + int64_t(k) * job.kStride;
  if (32 * tile + 32 <= job.R && 16 * slab + 16 <= job.K) {
    if (kContig) {
      const FineElems<float, 4> lo = *reinterpret_cast<const FineElems<float, 4> *>(at);
      const FineElems<float, 4> hi = *reinterpret_cast<const FineElems<float, 4> *>(at + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = lo.v[j];
        v[4 + j] = hi.v[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = at[j * job.kStride];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = r < job.R && k + j < job.K ? at[j * job.kStride] : 0.0f;
  }
  uint32_t largest = 0; // of the values' bits without their sign
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] *= scale;
    const uint32_t bits = __builtin_bit_cast(uint32_t, v[j]) & 0x7fffffffu;
    largest = bits > largest ? bits : largest;
  }
  // (what rounds to infinity as a bf16, and all beyond)
  const bool flag = __builtin_amdgcn_ballot_w64(largest >= 0x7f7f8000u) != 0;
  uintx4 h, m, l;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t ph, pm, pl;
    partsOf(flag ? 0.0f : v[2 * j], flag ? 0.0f : v[2 * j + 1], ph, pm, pl);
    h[j] = ph;
    m[j] = pm;
    l[j] = pl;
  }
  if (lane == 0)
    job.flags[(int64_t(tile / 4) * job.slabs + slab) * 4 + tile % 4] = flag;
  uintx4 *to = job.dst + (int64_t(tile) * job.slabs + slab) * kPlanesWords + lane;
  to[0] = h;
  to[kPlaneWords] = m;
  to[2 * kPlaneWords] = l;
}

// Where the tile-th block tile lies: panels of `panel` tiles along N, row by row.
__host__ __device__ inline void panelTile(int64_t tile, int tilesM, int tilesN, int panel, int &tm,
                                          int &tn) {
  const uint32_t t = uint32_t(tile), area = uint32_t(panel) * uint32_t(tilesM);
  const uint32_t p = t / area, in = t - p * area;
  const uint32_t rest = uint32_t(tilesN) - p * uint32_t(panel);
  const uint32_t width = rest < uint32_t(panel) ? rest : uint32_t(panel);
  tm = int(in / width);
  tn = int(p * uint32_t(panel) + in % width);
}

// The operands as they are, for what the parts cannot compute, and what that is: a
// word for each 128 rows and slab, a byte of it for each 32 rows.
struct PlanesSource {
  const float *X, *Y;
  int64_t xm, xk, yk, yn;
  int K;
  const uint32_t *xFlags, *yFlags;
};
constexpr int kPlanesMostSlabs = 256; // of a tile: a thread looks at the flags of one

__device__ __forceinline__ uint32_t ldsAddress(const uintx4 *p) {
  return uint32_t(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uintx4 *)p));
}

// Which tiles and slabs the blocks of a launch take: block g the whole tiles g,
// g + G, ... below `whole`, then its even share of the slabs of the others.
struct PlanesPlan {
  int tilesM, tilesN, panel; // see panelTile
  int slabs;                 // of a tile
  int run;                   // slabs whose products meet in the accumulators
  int64_t whole;             // a multiple of G, or all tiles
};
// Sums of a run of slabs leave the accumulators for float32 sums beside them; the
// left operand's parts change sign from run to run, so that what one run's sums
// lean downwards the next one's take back.  2-norm of the error, runs of 8 / 16 / 32
// slabs / none: K = 448 1.6e-7 / 2.3e-7 / 2.9e-7 / 2.9e-7, 2051 1.8e-7 / 2.4e-7 / 3.3e-7 /
// 6.8e-7, 4096 - / 2.4e-7 / 3.3e-7 / 9.9e-7.  On sgemm_parts in its slices or shares /
// this: K = 129 1.49e-7 / 1.15e-7, 433 1.81e-7 / 1.63e-7, 2051 4.54e-7 / 2.38e-7.  The ends of runs of 16 take 3 % of the time,
// of 8 7 %: the shorter ones where sgemm_parts cuts a short K.
constexpr int planesRun(int64_t K) { return K < 192 ? 4 : K < 768 ? 8 : 16; }

// One tile's slabs [slab0, slab1) for a block; tile < 0: there is nothing more.
// slot: which of its two slots a block's piece of a tile goes to.
struct PlanesSegment {
  int64_t tile;
  int slab0, slab1, slot;
};
struct PlanesWalk {
  int64_t tile, unit, unitEnd;
  int shares;
  __host__ __device__ void start(const PlanesPlan &plan, int64_t g, int64_t G) {
    const int64_t units = (int64_t(plan.tilesM) * plan.tilesN - plan.whole) * plan.slabs;
    tile = g;
    unit = evenSharesStart(g, units, G);
    unitEnd = evenSharesStart(g + 1, units, G);
    shares = 0;
  }
  __host__ __device__ PlanesSegment next(const PlanesPlan &plan, int64_t G) {
    PlanesSegment s = {-1, 0, plan.slabs, 0};
    if (tile < plan.whole) {
      s.tile = tile;
      tile += G;
    } else if (unit < unitEnd) {
      s.tile = unit / plan.slabs;
      s.slab0 = int(unit - s.tile * plan.slabs);
      if (unitEnd - unit < plan.slabs - s.slab0)
        s.slab1 = s.slab0 + int(unitEnd - unit);
      s.slot = shares++ ? 1 : 0;
      s.tile += plan.whole;
      unit += s.slab1 - s.slab0;
    }
    return s;
  }
};

// C[M,N] = alpha A B + beta C from the parts of both operands; C at any element's
// address.  Pieces of tiles go to their block's slots in W, in the order of the
// registers: [wave][tile row][tile column][four rows][lane][row], unscaled.
template <int BM, int BN, int STAGES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
sgemm_planes(const uintx4 *__restrict__ A, const uintx4 *__restrict__ B, float *__restrict__ C,
             int M, int N, int64_t ldc, float alpha, float beta, float *__restrict__ W,
             PlanesPlan plan, PlanesSource src) {
  constexpr int THREADS = 256, TM = BM / 64, TN = BN / 64;
  constexpr int AW = BM / 32 * kPlanesWords, BW = BN / 32 * kPlanesWords;
  constexpr int NA = AW / THREADS, NB = BW / THREADS;
  static_assert(AW % THREADS == 0 && BW % THREADS == 0, "whole words a thread");
  __shared__ uintx4 As[STAGES][AW];
  __shared__ uintx4 Bs[STAGES][BW];
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2, wn = wave % 2, slabs = plan.slabs;
  // (Blocks that run side by side on one XCD, every eighth, take neighbouring tiles.)
  const int G = gridDim.x, xcd = blockIdx.x % 8;
  const int me = xcd * (G / 8) + (xcd < G % 8 ? xcd : G % 8) + blockIdx.x / 8;
  uint32_t fromA[NA], fromB[NB]; // bytes, from an operand's slab on
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const uint32_t w = tid + THREADS * i;
    fromA[i] = 16 * (w / kPlanesWords * uint32_t(slabs) * kPlanesWords + w % kPlanesWords);
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const uint32_t w = tid + THREADS * i;
    fromB[i] = 16 * (w / kPlanesWords * uint32_t(slabs) * kPlanesWords + w % kPlanesWords);
  }
  PlanesWalk walk;
  walk.start(plan, me, G);
  PlanesSegment seg = walk.next(plan, G);
  int bm = 0, bn = 0, slab0 = 0, slab1 = 0;
  const uintx4 *a0 = A, *b0 = B;
  uint32_t flagA = 0, flagB = 0; // of slab tid of the segment
  // The n-th KiB of a wave's part of a slab of both operands on its way to LDS.
  // (Inline assembly, so that the waits are those written here: the compiler
  // lets every LDS read wait for all such loads.  They write LDS alone, from the
  // address in m0 on, which the compiler puts there.)
  auto fetch = [&](int n, int s, int stage) {
    const bool left = n < NA;
    const uint32_t to = ldsAddress(left ? As[stage] : Bs[stage]) +
                        16 * (wave * 64 + THREADS * (left ? n : n - NA));
    const uintx4 *from = (left ? a0 : b0) + int64_t(s) * kPlanesWords;
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "{m0}"(to), "v"(left ? fromA[left ? n : 0] : fromB[left ? 0 : n - NA]), "s"(from)
                 : "memory");
  };
  // A segment's first slabs on their way; no wave reads LDS any more.
  auto begin = [&] {
    int tm, tn;
    panelTile(seg.tile, plan.tilesM, plan.tilesN, plan.panel, tm, tn);
    bm = tm * BM;
    bn = tn * BN;
    slab0 = seg.slab0;
    slab1 = seg.slab1;
    a0 = A + int64_t(bm / 32) * slabs * kPlanesWords;
    b0 = B + int64_t(bn / 32) * slabs * kPlanesWords;
    flagA = flagB = 0; // (loaded ahead of the slabs: behind them a tile would wait for it)
    if (tid >= slab0 && tid < slab1) {
      flagA = src.xFlags[int64_t(tm) * slabs + tid];
      flagB = src.yFlags[int64_t(tn) * slabs + tid];
    }
#pragma unroll
    for (int i = 0; i < STAGES; ++i)
      if (slab0 + i < slab1) {
#pragma unroll
        for (int n = 0; n < NA + NB; ++n)
          fetch(n, slab0 + i, i);
      }
  };
  if (seg.tile >= 0)
    begin();
#pragma nounroll
  for (bool first = true; seg.tile >= 0; first = false) {
    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          acc[i][j][r] = 0.0f;
    // Sums of runs, with the sign that their parts have.
    floatx16 sum[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sum[i][j][r] = 0.0f;
    auto flush = [&](int s) {
      const float sign = s / plan.run % 2 ? -1.0f : 1.0f;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            sum[i][j][r] = __builtin_fmaf(acc[i][j][r], sign, sum[i][j][r]);
            acc[i][j][r] = 0.0f;
          }
    };
    int cur = 0; // the stage of the slab that is multiplied
    const bool inside = tid >= slab0 && tid < slab1;
    auto flagsHere = [&] { // (waited for here, not before the tile)
      asm volatile("" : "+v"(flagA), "+v"(flagB));
      return (flagA | flagB) != 0;
    };

    struct Operands {
      bf16x8 a[TM][3], b[TN][3];
    };
    // The n-th of the matrix instructions' 128-bit words of a slab.
    auto read = [&](Operands &o, int n, int stage) {
      if (n < 3 * TN)
        o.b[n / 3][n % 3] = __builtin_bit_cast(
            bf16x8, Bs[stage][(wn * TN + n / 3) * kPlanesWords + n % 3 * kPlaneWords + lane]);
      else
        o.a[n / 3 - TN][n % 3] = __builtin_bit_cast(
            bf16x8,
            As[stage][(wm * TM + n / 3 - TN) * kPlanesWords + n % 3 * kPlaneWords + lane]);
    };
    // Waits for the slab of which `behind` more may be on their way; and for all waves.
    auto arrive = [&](int behind) {
      if (behind >= 2)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(2 * (NA + NB)) : "memory");
      else if (behind == 1)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(NA + NB) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory");
    };
    Operands now, next;
    arrive(first ? slab1 - slab0 - 1 : 0); // (else: the last segment's stores are behind them)
#pragma unroll
    for (int n = 0; n < 3 * (TM + TN); ++n)
      read(now, n, 0);
    // Multiplies slab s while the words of the next go to registers and, FETCH,
    // slab s + STAGES starts on its way to the stage of s (which all waves have in
    // registers): a memory instruction behind a matrix instruction each.
    auto slab = [&](int s, Operands &o, Operands &to, auto fetches) {
      constexpr bool FETCH = decltype(fetches)::value != 0;
      arrive(FETCH ? STAGES - 2 : slab1 - s - 2 < STAGES - 2 ? slab1 - s - 2 : STAGES - 2);
      const int mine = cur;
      cur = cur + 1 < STAGES ? cur + 1 : 0;
      constexpr int LEFT[6] = {2, 0, 1, 1, 0, 0}, RIGHT[6] = {0, 2, 1, 0, 1, 0};
      constexpr int READS = 3 * (TM + TN), LOADS = FETCH ? NA + NB : 0;
      constexpr int PRODUCTS = 6 * TM * TN, OVER = PRODUCTS - 4;
#pragma unroll
      for (int q = 0; q < PRODUCTS; ++q) {
        const int i = q / (6 * TN), t = q / TN % 6, j = q % TN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(o.a[i][LEFT[t]], o.b[j][RIGHT[t]],
                                                            acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (q < OVER) {
#pragma unroll
          for (int n = q * READS / OVER; n < (q + 1) * READS / OVER; ++n)
            read(to, n, cur);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int n = q * LOADS / OVER; n < (q + 1) * LOADS / OVER; ++n)
            fetch(n, s + STAGES, mine);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    typedef std::integral_constant<int, 0> No;
    typedef std::integral_constant<int, 1> Yes;
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
            finite = __builtin_fmaf(sum[i][j][r], 0.0f, finite);
          if (__builtin_amdgcn_ballot_w64(finite != finite))
            lost |= 1u << (i * TN + j);
        }
      return lost;
    };
    bool early = false; // the parts are given up before the end of K
    uint32_t lost = 0;
    int s = slab0;
    // (A look for infinities costs a third of a slab: after 4 slabs, if more than 24
    // follow, and every 128.)
    int look = slab1 - slab0 > 28 ? slab0 + 4 : slab1;
    while (s < slab1 && !early) {
      int stop = (s / plan.run + 1) * plan.run;
      stop = stop < slab1 ? stop : slab1;
      stop = look > s && look < stop ? look : stop;
#pragma nounroll
      for (; s + 1 < stop && s + 1 + STAGES < slab1; s += 2) {
        slab(s, now, next, Yes());
        slab(s + 1, next, now, Yes());
      }
#pragma nounroll
      for (; s < stop; ++s) {
        if (s + STAGES < slab1)
          slab(s, now, next, Yes());
        else
          slab(s, now, next, No());
        now = next;
      }
      flush(s - 1);
      if (s >= look && s < slab1) {
        // (or most of the slabs are flagged)
        const bool many = 2 * __builtin_popcount(tilesLost()) > TM * TN;
        const uint64_t flagged = __builtin_amdgcn_ballot_w64(flagsHere());
        const uint64_t all = __builtin_amdgcn_ballot_w64(inside);
        if (__syncthreads_or(many || flagged))
          early = __syncthreads_or(many) ||
                  __syncthreads_and(2 * __builtin_popcountll(flagged) >= __builtin_popcountll(all));
        look = s + 128;
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); // (early: slabs on their way)
    lost = early ? (1u << (TM * TN)) - 1 : tilesLost();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          sum[i][j][r] = lost >> (i * TN + j) & 1
                             ? 0.0f
                             : __builtin_fmaf(sum[i][j][r], 1.0f / (kPartsScale * kPartsScale),
                                              0.0f); // (no -0)
    const bool flag = flagsHere();
    if (__syncthreads_or(lost != 0 || flag)) {
      // The lost tiles, and the flagged slabs of the others, with
      // v_mfma_f32_32x32x2_f32 on the operands themselves: lane half h of the wave takes
      // k = 8 h + t of the slab in step t.  In LDS a slab is [four of K][row], rows so
      // that neither four apart nor side by side share a bank.  Waves 0 and 1 load A's
      // rows, 2 and 3 B's, a thread four rows by four of K in four words, four slabs
      // ahead in registers (one wave a SIMD has no other to run beside its waits).
      //
      // us a call, on sgemm_parts / whole tiles again, a slab ahead / this: 2047 x 2049 x
      // 2051 (ordinary data 147 / 133 / 134) one NaN 178 / 297 / 136, an infinity in the
      // last column of every 128th row 220 / 319 / 141 and of every row 288 / 398 / 141,
      // all sums too large 248 / 315 / 244; 1801 x 1300 x 433 (46 / 43 / 43) 48 / 77 / 46,
      // 50 / 74 / 45, 53 / 86 / 46, 68 / 86 / 77.
      static_assert(BM == 128 && BN == 128 && STAGES == 4, "four by four a thread, four ahead");
      int here = tid; // (places are worked out here, not ahead of the tiles)
      asm volatile("" : "+v"(here));
      const int home = here % 64;
      constexpr int QUAD = 148; // words of four of K
      auto placeOf = [](int row) { return row % 4 * 34 + row / 4; };
      uint32_t *flags = reinterpret_cast<uint32_t *>(As[0] + 4 * QUAD); // A's, then B's
      uint64_t *need = reinterpret_cast<uint64_t *>(flags + 2 * kPlanesMostSlabs);
      static_assert((AW - 4 * QUAD) * 16 >= 8 * kPlanesMostSlabs + 8 * THREADS / 64 &&
                        THREADS == kPlanesMostSlabs,
                    "room behind the slab; a flag a thread");
      const bool whole = __syncthreads_or(lost != 0); // all slabs, not the flagged ones alone
      const uint64_t bits = __builtin_amdgcn_ballot_w64(inside && (whole || flag));
      flags[here] = flagA;
      flags[kPlanesMostSlabs + here] = flagB;
      if (lane == 0)
        need[wave] = bits;
      __syncthreads();
      auto uniform = [](uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); };
      const int full = src.K / 16, end = slab1 < full ? slab1 : full; // whole slabs
      auto following = [&](int k) { // the next slab after k, or end
        for (++k; k < end; k = (k | 63) + 1) {
          const uint64_t word = need[k >> 6] >> (k & 63);
          const uint64_t rest = uint64_t(uniform(uint32_t(word >> 32))) << 32 |
                                uniform(uint32_t(word));
          if (rest) {
            k += __builtin_ctzll(rest);
            break;
          }
        }
        return k < end ? k : end;
      };
      const bool forA = wave < 2;
      const int64_t rowStride = forA ? src.xm : src.yn, kStride = forA ? src.xk : src.yk;
      const int origin = forA ? bm : bn, extent = forA ? M : N;
      const bool kContig = kStride == 1, ragged = !kContig && origin + BM > extent;
      // (its rows: kContig row, row + 32, ..., else row, row + 1, ...)
      const int quad = kContig ? here % 4 : here % 128 / 32;
      const int row = kContig ? here % 128 / 4 : 4 * (here % 32);
      const int r0 = origin + row, r4 = r0 < extent - 4 ? r0 : extent - 4;
      const int shift = r0 - r4 < 3 ? r0 - r4 : 3; // (rows beyond the last are the last again)
      const float *at[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = r0 + 32 * i < extent ? r0 + 32 * i : extent - 1;
        at[i] = (forA ? src.X : src.Y) + (kContig ? int64_t(r) * rowStride + 4 * quad
                                                  : r4 + int64_t(4 * quad + i) * kStride);
      }
      typedef FineElems<float, 4> Word;
      auto load = [&](floatx4 (&v)[4], int k) {
        k = k < end ? k : full - 1; // (nothing more: loaded in vain, so that no load is in a branch)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const Word w = *reinterpret_cast<const Word *>(at[i] + int64_t(k) * (16 * kStride));
          v[i] = floatx4{w.v[0], w.v[1], w.v[2], w.v[3]};
        }
      };
      auto stash = [&](floatx4 (&v)[4], int stage) {
        if (ragged) {
#pragma unroll
          for (int by = 1; by <= 2; ++by)
            if (shift & by) {
#pragma unroll
              for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  v[i][e] = v[i][e + by < 3 ? e + by : 3];
            }
        }
        floatx4 *to = reinterpret_cast<floatx4 *>(forA ? As[stage] : Bs[stage]) +
                      quad * QUAD + placeOf(row);
        const int apart = kContig ? placeOf(32) : placeOf(1);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          to[i * apart] = kContig ? v[i] : floatx4{v[0][i], v[1][i], v[2][i], v[3][i]};
      };
      auto add = [&](int k, int stage) {
        floatx4 left[TM][2], right[TN][2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
            left[i][w] = reinterpret_cast<const floatx4 *>(
                As[stage])[(home / 32 * 2 + w) * QUAD + placeOf((wm * TM + i) * 32 + home % 32)];
#pragma unroll
          for (int j = 0; j < TN; ++j)
            right[j][w] = reinterpret_cast<const floatx4 *>(
                Bs[stage])[(home / 32 * 2 + w) * QUAD + placeOf((wn * TN + j) * 32 + home % 32)];
        }
        const uint32_t fa = uniform(flags[k]) >> (8 * TM * wm);
        const uint32_t fb = uniform(flags[kPlanesMostSlabs + k]) >> (8 * TN * wn);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) {
            if (!(lost >> (i * TN + j) & 1 || (fa >> (8 * i) & 1) || (fb >> (8 * j) & 1)))
              continue;
#pragma unroll
            for (int t = 0; t < 8; ++t)
              sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(left[i][t / 4][t % 4],
                                                               right[j][t / 4][t % 4], sum[i][j],
                                                               0, 0, 0);
          }
      };
      // (waits for LDS alone: loads stay on their way)
      auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory"); };
      floatx4 v0[4], v1[4], v2[4], v3[4];
      int next = following(slab0 - 1), k0, k1, k2, k3; // the slab after those in v0 to v3
      auto start = [&](floatx4 (&v)[4], int &k) {
        load(v, k = next);
        next = following(next);
      };
      auto step = [&](floatx4 (&v)[4], int &k, int stage) {
        stash(v, stage);
        meet(); // (also: every wave has read the stage of three slabs before)
        const int of = k;
        start(v, k);
        if (of < end)
          add(of, stage);
      };
      start(v0, k0);
      start(v1, k1);
      start(v2, k2);
      start(v3, k3);
#pragma nounroll
      while (k0 < end) { // (four steps without a way out between: see load)
        step(v0, k0, 0);
        step(v1, k1, 1);
        step(v2, k2, 2);
        step(v3, k3, 3);
      }
      if (slab1 > full && need[full >> 6] >> (full & 63) & 1) { // the end of K
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v0[i][e] = 16 * full + 4 * quad + (kContig ? e : i) < src.K
                               ? at[i][int64_t(full) * (16 * kStride) + e]
                               : 0.0f;
        __syncthreads();
        stash(v0, 0);
        __syncthreads();
        add(full, 0);
      }
    }

    // A whole tile goes to C, scaled; a piece of one to its slot.
    int home = lane;
    asm volatile("" : "+v"(home)); // (places in C are worked out here, not kept over K)
    const bool piece = slab0 > 0 || slab1 < slabs;
    const int rowsLeft = M - bm, colsLeft = N - bn;
    float *out = piece ? W + (int64_t(me) * 2 + seg.slot) * (BM * BN) + wave * (TM * TN * 1024)
                       : C + int64_t(bm) * ldc + bn;
    __syncthreads(); // every wave is done with this segment's slabs in LDS
    seg = walk.next(plan, G);
    if (seg.tile >= 0)
      begin();
    if (piece) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; r += 4)
            reinterpret_cast<floatx4 *>(out)[((i * TN + j) * 4 + r / 4) * 64 + home] =
                floatx4{sum[i][j][r], sum[i][j][r + 1], sum[i][j][r + 2], sum[i][j][r + 3]};
    } else if (beta == 0.0f && rowsLeft >= BM && colsLeft >= BN) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            out[int64_t(wm * (TM * 32) + i * 32 + Mfma<float>::accRow(r, home)) * ldc +
                wn * (TN * 32) + j * 32 + home % 32] = alpha * sum[i][j][r];
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int col = wn * (TN * 32) + j * 32 + home % 32;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = wm * (TM * 32) + i * 32 + Mfma<float>::accRow(r, home);
            if (!(row < rowsLeft && col < colsLeft))
              continue;
            float *dst = out + int64_t(row) * ldc + col;
            float v = alpha * sum[i][j][r];
            if (beta != 0.0f)
              v += beta * *dst;
            *dst = v;
          }
        }
      }
    }
  } // segments
}

// C[tile] = alpha * (piece + piece + ...) + beta * C[tile] for the tiles behind
// `whole`, pieces in the order of K; grid (tiles, BM * BN / 1024).  A thread adds
// one 128-bit word of every piece: four rows of a column.
template <int BM, int BN>
__global__ __launch_bounds__(256) void
sgemm_planes_fold(const float *__restrict__ W, int64_t G, PlanesPlan plan, float *__restrict__ C,
                  int M, int N, int64_t ldc, float alpha, float beta) {
  constexpr int TM = BM / 64, TN = BN / 64;
  const int64_t units = (int64_t(plan.tilesM) * plan.tilesN - plan.whole) * plan.slabs;
  const int64_t u0 = int64_t(blockIdx.x) * plan.slabs, u1 = u0 + plan.slabs;
  // the block whose share holds the tile's first unit
  int64_t g = evenSharesStart(u0, G, units);
  while (g > 0 && evenSharesStart(g, units, G) > u0)
    --g;
  while (g + 1 < G && evenSharesStart(g + 1, units, G) <= u0)
    ++g;
  if (evenSharesStart(g, units, G) <= u0 && evenSharesStart(g + 1, units, G) >= u1)
    return; // one block computed the whole tile and stored it itself
  const int word = blockIdx.y * 256 + threadIdx.x;
  floatx4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  for (; g < G; ++g) {
    const int64_t begin = evenSharesStart(g, units, G);
    if (begin >= u1)
      break;
    sum += reinterpret_cast<const floatx4 *>(
        W + (g * 2 + (begin >= u0 ? 0 : 1)) * int64_t(BM * BN))[word];
  }
  const int lane = word % 64, r = word / 64 % 4 * 4, j = word / 256 % TN, i = word / (256 * TN) % TM;
  const int wave = word / (256 * TN * TM);
  int tm, tn;
  panelTile(plan.whole + blockIdx.x, plan.tilesM, plan.tilesN, plan.panel, tm, tn);
  const int col = tn * BN + wave % 2 * (TN * 32) + j * 32 + lane % 32;
  const int row = tm * BM + wave / 2 * (TM * 32) + i * 32;
  if (col >= N)
    return;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int at = row + Mfma<float>::accRow(r + q, lane);
    if (at >= M)
      break;
    float *dst = C + int64_t(at) * ldc + col;
    float v = alpha * sum[q];
    if (beta != 0.0f)
      v += beta * *dst;
    *dst = v;
  }
}

} // namespace
