"""The trainer's step schedule and the check of it (mlp_schedule.hpp): every sample is taken once, every
row of a step by one workgroup, and arrays one element short are refused."""
import os
import shutil
import subprocess

import pytest

from test_host_sanitizers import CSRC

DRIVER = r"""
#include "mlp_schedule.hpp"

#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace ebgpu;

#define CHECK(c)                                                                                  \
  do {                                                                                            \
    if (!(c)) {                                                                                   \
      std::printf("check failed at line %d: %s\n", __LINE__, #c);                                 \
      std::exit(1);                                                                               \
    }                                                                                             \
  } while (0)

int main()
{
  const std::pair<uint64_t, int> cases[] = {{64, 32},    {65, 64},     {100, 4096}, {4096, 4096}, {4097, 4096},
                                            {8191, 8192}, {8193, 8192}, {8257, 8256}, {65537, 65536}};
  for (const auto& [n, batch] : cases) {
    const int   rows = int(std::min<uint64_t>(n, batch)), blocks = mlp_train_blocks(batch);
    std::string why;
    CHECK(check_train_schedule(n, batch, n, blocks, &why));
    CHECK(!check_train_schedule(n, batch, n - 1, blocks, &why) && why == "training batch reaches past the samples");
    CHECK(!check_train_schedule(n, batch, n, mlp_train_blocks(rows) - 1, &why));
    CHECK(why == "training batch larger than its buffers");
    std::vector<int> taken(n, 0);
    for (uint64_t k = 0; k < train_steps(n, batch); k++) {
      const TrainStep t = train_step(n, batch, k);
      CHECK(check_train_step(t.rows, n - t.first, blocks, nullptr));
      CHECK(!check_train_step(t.rows, t.rows - 1, blocks, nullptr));
      const int nb = mlp_train_blocks(t.rows);
      for (int b = 0; b < nb; b++) // the kernel's loop
        for (int row0 = b * kTrainRows; row0 < t.rows; row0 += nb * kTrainRows)
          for (int r = row0; r < std::min(row0 + kTrainRows, t.rows); r++) taken[t.first + r]++;
    }
    for (int x : taken) CHECK(x == 1);
  }
  CHECK(!check_train_schedule(0, 64, 0, 1, nullptr) && !check_train_schedule(64, 0, 64, 1, nullptr));
  CHECK(!check_train_step(0, 64, 1, nullptr));
  std::printf("schedules checked\n");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ absent")
def test_training_schedule(tmp_path):
    src = tmp_path / "schedule.cpp"
    src.write_text(DRIVER)
    exe = tmp_path / "schedule"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I" + CSRC, str(src), "-o", str(exe)], capture_output=True,
                       text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and "schedules checked" in run.stdout, (run.stdout, run.stderr)
