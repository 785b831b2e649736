// Copies of gemm operands into word-aligned, zero-padded rows (gemm_pack_rows
// in Gemm.hip), and how they are dealt to launches.  Host code but for the
// counts, which the kernel takes as well; also compiled without HIP.
#pragma once

#include <cstdint>

#ifndef __HIP__
#define __host__
#define __device__
#endif

namespace {

// dst[r][c] (rows of Cp elements, Rp of them) = src[r * ld + c] where r < R and
// c < C, zero elsewhere; Cp a multiple of VEC.
template <typename T, int VEC> struct PackJob {
  const T *src = nullptr;
  int64_t ld = 0, R = 0, C = 0;
  T *dst = nullptr;
  int64_t Cp = 0, Rp = 0;
  __host__ __device__ int64_t words() const { return Rp * (Cp / VEC); }
  __host__ __device__ int64_t blocks() const { return (words() + 255) / 256; }
};

// launch(a, b) for both jobs at once where `most` blocks hold them; longer ones
// in runs of rows, and none for nothing: a launch counts its work-items in 32
// bits, and one of no blocks is an error.
template <typename Job, typename Launch>
void launchPacks(Job first, Job second, int64_t most, Launch launch) {
  if (first.blocks() + second.blocks() <= most) {
    if (first.blocks() + second.blocks() > 0)
      launch(first, second);
    return;
  }
  for (Job job : {first, second})
    while (job.words() > 0) {
      const int64_t wordsOfRow = job.words() / job.Rp;
      int64_t rows = most * 256 / wordsOfRow;
      rows = rows < 1 ? 1 : rows < job.Rp ? rows : job.Rp;
      Job run = job;
      run.Rp = rows;
      run.R = run.R < rows ? run.R : rows;
      launch(run, Job());
      job.src += rows * job.ld;
      job.dst += rows * job.Cp;
      job.R -= run.R;
      job.Rp -= rows;
    }
}

} // namespace
