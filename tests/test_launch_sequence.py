"""A call of several launches that takes a scratch slot first: a refused launch ends it, and gives the slot back
if it was taken. Compiled for the host, with launches that fail where they are told to."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cstdio>
#include "launch_sequence.hpp"
int main() {
  for (int fail = 0; fail <= 4; ++fail) {
    int taken = 0, enqueued = 0;
    const int rc = ds41g::launch_sequence(
        4,
        [&](int i) {
          if (i == fail) return 700 + i;
          ++enqueued;
          if (i == 0) ++taken;
          if (i == 3) --taken;
          return 0;
        },
        [&] { --taken; });
    std::printf("%d %d %d\n", rc, enqueued, taken);
  }
}
"""


def test_refused_launch_gives_the_slot_back(tmp_path):
    src, exe = tmp_path / "sequence.cpp", tmp_path / "sequence"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "deepseek-v4.1-flash-pro6000_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True, timeout=120)
    got = [tuple(map(int, line.split())) for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=60).stdout.splitlines()]
    assert got == [(700 + f, f, 0) for f in range(4)] + [(0, 4, 0)]


def test_wide_sampler_reports_a_refused_launch():
    """Without a device the first launch is refused: the call returns its error."""
    import sys
    sys.path.insert(0, os.path.join(ROOT, "deepseek-v4.1-flash-pro6000_amd"))
    import ds41_gfx950 as G
    import torch
    if torch.cuda.is_available():
        return  # the addresses below are never read
    assert G.lib().ds41_spark_verify_gpu_v2(None, None, 256, 0, 20000, 0, 1, 2, 512, None) != 0
    assert G.lib().ds41_spark_sample_gpu_v2(256, 20000, 1, 2, 0, 0, 512, None) != 0
