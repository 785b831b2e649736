"""Host-only check of how copies of gemm operands are dealt to launches: one
launch for both where it counts the blocks, runs of rows beyond that, and never a
launch of no blocks, which HIP refuses."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
MATH = os.path.join(os.path.dirname(HERE), "numba_mlir_amd", "csrc", "math")

PROGRAM = r"""
#include "PackJobs.h"
#include <cstdio>
#include <vector>
typedef PackJob<float, 4> Job;

int main() {
  // rows, columns, padded columns, padded rows; none of one operand
  const int64_t shapes[][4] = {{0, 0, 0, 0},        {1, 1, 4, 1},      {5, 7, 8, 5},
                               {37, 1021, 1024, 64}, {300, 33, 48, 512}, {64, 4093, 4096, 64}};
  for (int64_t most : {1, 2, 5, 16, 1000})
    for (auto &s : shapes)
      for (auto &t : shapes) {
        std::vector<float> from[2], to[2];
        Job jobs[2];
        int i = 0;
        for (auto *u : {s, t}) {
          const int64_t ld = u[1] + 3;
          from[i].resize(u[0] * ld + 1);
          for (size_t k = 0; k < from[i].size(); ++k)
            from[i][k] = float(k + 1);
          to[i].assign(u[2] * u[3], -1.0f);
          if (u[0])
            jobs[i] = Job{from[i].data(), ld, u[0], u[1], to[i].data(), u[2], u[3]};
          ++i;
        }
        int launches = 0;
        launchPacks(jobs[0], jobs[1], most, [&](const Job &a, const Job &b) {
          const int64_t blocks = a.blocks() + b.blocks();
          ++launches;
          // (a row is the least that a launch takes)
          if (blocks <= 0 || (blocks > most && a.Rp > 1)) {
            std::printf("a launch of %lld blocks, %lld at most\n", (long long)blocks,
                        (long long)most);
            std::exit(1);
          }
          for (const Job &j : {a, b})
            for (int64_t r = 0; r < j.Rp; ++r)
              for (int64_t c = 0; c < j.Cp; ++c)
                j.dst[r * j.Cp + c] = r < j.R && c < j.C ? j.src[r * j.ld + c] : 0.0f;
        });
        if (jobs[0].blocks() + jobs[1].blocks() <= most && launches > 1)
          return std::printf("%d launches where one holds both\n", launches), 1;
        i = 0;
        for (auto *u : {s, t}) {
          for (int64_t r = 0; r < u[3]; ++r)
            for (int64_t c = 0; c < u[2]; ++c) {
              const float want =
                  r < u[0] && c < u[1] ? from[i][r * (u[1] + 3) + c] : 0.0f;
              if (to[i][r * u[2] + c] != want)
                return std::printf("operand %d, row %lld, column %lld\n", i, (long long)r,
                                   (long long)c), 1;
            }
          ++i;
        }
      }
  return 0;
}
"""


def test_copies_dealt_to_launches(tmp_path):
    cxx = os.environ.get("CXX", "g++")
    if shutil.which(cxx) is None:
        pytest.skip("no host compiler")
    source, program = tmp_path / "pack.cpp", tmp_path / "pack"
    source.write_text("#include <cstdlib>\n" + PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-I", MATH, str(source), "-o",
                    str(program)], check=True)
    run = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0, run.stdout
