"""Set-up that belongs to a device (a kernel's dynamic-LDS limit) runs once on
each one a process uses, again after a failure, and from several threads."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "attention_nn_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "per_device.h"

int main() {
  ann::PerDevice p;
  int runs[3] = {0, 0, 0};
  auto at = [&](int dev, int rc) { return p.once(dev, [&] { ++runs[dev]; return rc; }); };
  if (at(0, 0) || at(0, 7) || runs[0] != 1) return 1;      // done: not run again
  if (at(1, 7) != 7 || at(1, 0) || at(1, 7) || runs[1] != 2) return 2;   // a failure is not kept
  if (at(2, 0) || runs[2] != 1) return 3;                  // each device its own
  int high = 0;
  for (int i = 0; i < 2; ++i) p.once(64, [&] { ++high; return 0; });
  if (high != 2) return 4;
  ann::PerDevice q;
  std::atomic<int> bad{0};
  std::vector<std::thread> ts;
  for (int t = 0; t < 8; ++t)
    ts.emplace_back([&] {
      for (int d = 0; d < 64; ++d)
        if (q.once(d, [] { return 0; })) ++bad;
    });
  for (auto& t : ts) t.join();
  for (int d = 0; d < 64; ++d)
    if (q.once(d, [] { return 1; })) ++bad;
  return bad ? 5 : 0;
}
"""


def test_once_per_device(tmp_path):
    src, exe = tmp_path / "per_device.cpp", tmp_path / "per_device"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


def test_limits_are_not_kept_per_process():
    """Every launcher asks through PerDevice: none keeps the answer in a static
    of its own."""
    for name in os.listdir(CSRC):
        with open(os.path.join(CSRC, name)) as f:
            lines = [ln for ln in f if "hipFuncSetAttribute" in ln]
        assert not any("static" in ln for ln in lines), name
        assert not lines or name in ("launch.h", "gemm_ring.hip"), name
